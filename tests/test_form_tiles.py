"""The forms kernels at the edges of their tiles: a grid large enough for the
form-pair launch against the same columns in a grid that takes the small tile,
for component counts around the 128-row tiles, rows that end early and an odd
number of forms of a type.  Both run the same bf16 operands, so they differ by
the order of FP32 sums only: 1e-5 of the field scale, the library's FP32 bound."""
import numpy as np
import pytest

from cfdwavemaker_amd.seastate import make_sea
from tests.conftest import scaled_err


@pytest.fixture(scope="module")
def eng():
    from cfdwavemaker_amd import engine
    engine.load()
    return engine


@pytest.mark.gpu
@pytest.mark.parametrize("nfreq,ndir,depth,kw", [
    (5, 2, 30.0, {}),                            # far below one tile
    (64, 1, 20.0, {}),                           # half a tile: the second 64 rows have no pairs
    (65, 1, 60.0, {}),                           # one row into the second half
    (32, 4, 100.0, {}),                          # one whole tile
    (43, 3, 45.0, {}),                           # 129: one row into a second tile
    (60, 4, 150.0, dict(bandwidth=0.6)),         # 240, rows that end inside a tile
    (100, 4, 10.0, dict(cutoff=2.0)),            # 400, rows past the cutoff empty
])
@pytest.mark.parametrize("mode", ["bf16", "fp32"])
def test_large_launch_equals_small(eng, mode, nfreq, ndir, depth, kw):
    s = make_sea(nfreq, 2.0, 8.0, depth, seed=nfreq, ndir=ndir).as_dict()
    s.update(kw)
    prec = eng.BF16 if mode == "bf16" else eng.FP32
    dx = 6.0
    n, m = 96, 5                                 # 36,864 and 100 column-slots
    big = eng.Sea(s, precision=prec, with_direct=False).grid((0.0, (n - 1) * dx, 0.0, (n - 1) * dx), n, n, 4, 0.0,
                                                             0.5, 0.7, 1.5, depth)
    small = eng.Sea(s, precision=prec, with_direct=False).grid((0.0, (m - 1) * dx, 0.0, (m - 1) * dx), m, m, 4, 0.0,
                                                               0.5, 0.7, 1.5, depth)
    assert big.qform_info() and small.qform_info()
    for f, tail in (("ETA", ()), ("UX", (4,)), ("UY", (4,)), ("UZ", (4,))):
        a = big.export(f).reshape((4, n, n) + tail)[:, :m, :m].ravel()
        b = small.export(f)
        if not np.any(b):
            assert not np.any(a)
            continue
        assert scaled_err(a, b) <= 1e-5, (f, scaled_err(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("n,depth,nl", [(2, 30.0, 4), (130, 30.0, 16), (200, 120.0, 9)])
def test_seas_along_x_leave_the_v_forms_out(prec, n, depth, nl):
    """Along x every v coefficient is zero and the v forms are left out: the other
    fields are the bits of the same sea with directions of 1e-20, whose v forms run."""
    from cfdwavemaker_amd import engine as eng
    from cfdwavemaker_amd.seastate import make_sea
    p = eng.FP32 if prec == "fp32" else eng.BF16
    s = make_sea(n, 2.0, 8.0, depth, seed=n, ndir=1).as_dict()
    g = []
    for th in (0.0, 1e-20):
        s["theta"] = np.full(len(s["omega"]), th)
        g.append(eng.Sea(s, precision=p, with_direct=False).grid((0.0, 60.0, 0.0, 45.0), 21, 16, nl, 0.0, 0.5, 0.7, 1.5,
                                                                 depth))
    assert g[0].qform_info()["nform"] < g[1].qform_info()["nform"]
    for f in ("ETA", "UX", "UZ"):
        assert np.array_equal(g[0].export(f), g[1].export(f)), f
    assert not np.any(g[0].export("UY"))


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["fp32", "bf16"])
@pytest.mark.parametrize("nx,ny", [(8, 4), (32, 31), (33, 32), (41, 40), (56, 72), (64, 65), (64, 80), (90, 88)])
def test_every_tile_of_a_launch(eng, mode, nx, ny):
    """Every column of launches whose last group of point tiles is whole, short by
    one, one tile or an odd one, of small and of wide tiles and of form pairs,
    against the same columns in grids of 8 rows; bound as above."""
    s = make_sea(40, 2.0, 8.0, 30.0, seed=nx, ndir=4).as_dict()
    prec = eng.BF16 if mode == "bf16" else eng.FP32
    sea = eng.Sea(s, precision=prec, with_direct=False)

    def part(j0, j1):
        return sea.grid((0.0, 6.0 * (nx - 1), 6.0 * j0, 6.0 * (j1 - 1)), nx, j1 - j0, 4, 0.0, 0.5, 0.7, 1.5, 30.0)
    at = list(range(0, max(ny - 1, 1), 8))
    rows = [part(j, k) for j, k in zip(at, at[1:] + [ny])]
    big = part(0, ny)
    assert big.qform_info()
    for f, tail in (("ETA", ()), ("UX", (4,)), ("UY", (4,)), ("UZ", (4,))):
        a = big.export(f).reshape((4, nx, ny) + tail)
        b = np.concatenate([g.export(f).reshape((4, nx, -1) + tail) for g in rows], axis=2)
        assert a.shape == b.shape
        assert scaled_err(a.ravel(), b.ravel()) <= 1e-5, f
