"""FP64 s-grid fills through the depth nodes and quadratic forms: grids around the
tile edges against the oracle's column body, and the forms against the pair loop."""
import numpy as np
import pytest

from cfdwavemaker_amd.seastate import make_sea
from tests.conftest import scaled_err

# rounding of the interpolation (4e-15 of a profile of size <= 2) and of FP64
# sums over up to 2e4 pairs, far inside the library's FP64 contract of 1e-9
TOL = 1e-11


@pytest.fixture(scope="module")
def eng():
    from cfdwavemaker_amd import engine
    engine.load()
    return engine


def _ignore(dom, frac):
    return (dom[0], dom[0] + frac * (dom[1] - dom[0]), dom[2], dom[3])


@pytest.mark.gpu
@pytest.mark.parametrize("nfreq,ndir,nx,ny,nl,kw", [
    (2, 1, 40, 26, 4, {}),                       # one pair
    (63, 1, 16, 16, 5, {}),                      # one short 64-row tile
    (64, 1, 17, 16, 4, {}),                      # one whole tile
    (13, 5, 33, 8, 7, {}),                       # 65 components: a second tile of one row
    (24, 8, 8, 9, 16, dict(depth=150.0)),        # deep: more nodes
    (40, 4, 11, 9, 11, dict(depth=6.0)),         # shallow: fewest nodes
    (48, 3, 64, 4, 4, dict(bandwidth=0.7, cutoff=1.9)),   # filtered rows end early
    (30, 4, 20, 11, 6, dict(swl=1.5, ignore=0.4)),
])
def test_fill_and_update_vs_oracle(eng, oracle, nfreq, ndir, nx, ny, nl, kw):
    s = make_sea(nfreq, 3.0, 9.0, kw.get("depth", 40.0), seed=nfreq, ndir=ndir).as_dict()
    for k in ("bandwidth", "cutoff", "swl"):
        if k in kw:
            s[k] = kw[k]
    dom = (10.0, 10.0 + 7.0 * max(nx - 1, 1), -5.0, -5.0 + 6.0 * max(ny - 1, 1))
    ig = _ignore(dom, kw["ignore"]) if "ignore" in kw else (1e12, -1e12, 1e12, -1e12)
    args = (dom, nx, ny, nl, 3.0, 0.5, 0.7, 1.5, s["depth"], s.get("swl", 0.0), ig, 0)
    g = eng.Sea(s, precision=eng.FP64, with_direct=False).grid(*args)
    o = oracle.sea(s).grid(*args)
    for step in range(2):
        if step:
            g.force_update(3.75)
            o.force_update(3.75)
        for f in ("ETA", "UX", "UY", "UZ"):
            a, b = g.export(f), o.export(f)
            if not np.any(b):
                assert not np.any(a), f
                continue
            assert scaled_err(a, b) <= TOL, (step, f, scaled_err(a, b))


@pytest.mark.gpu
def test_forms_and_pair_loop_agree(eng, monkeypatch):
    """The same fill through both routes (a grid of fewer points than twice
    the padded component count takes the pair loop)."""
    s = make_sea(20, 3.0, 9.0, 40.0, seed=4, ndir=4).as_dict()
    dx = 8.0
    big = eng.Sea(s, with_direct=False).grid((0.0, 31 * dx, 0.0, 31 * dx), 32, 32, 4, 0.0, 0.5, 0.7, 1.5, 40.0)
    small = eng.Sea(s, with_direct=False).grid((0.0, 2 * dx, 0.0, 2 * dx), 3, 3, 4, 0.0, 0.5, 0.7, 1.5, 40.0)
    for f, tail in (("ETA", ()), ("UX", (4,)), ("UY", (4,)), ("UZ", (4,))):
        a = big.export(f).reshape((4, 32, 32) + tail)[:, :3, :3].ravel()
        assert scaled_err(a, small.export(f)) <= TOL, f


@pytest.mark.gpu
def test_components_ramped_apart_take_the_pair_loop(eng, oracle):
    s = make_sea(12, 3.0, 9.0, 40.0, seed=5).as_dict()
    s["ramptime"], s["starttime"], s["duration"] = np.linspace(1, 4, 12), np.zeros(12), np.full(12, 1e6)
    args = ((0.0, 100.0, 0.0, 60.0), 32, 16, 4, 0.5, 0.5, 0.7, 1.5, 40.0)
    g, o = eng.Sea(s, with_direct=False).grid(*args), oracle.sea(s).grid(*args)
    for f in ("ETA", "UX", "UZ"):
        assert scaled_err(g.export(f), o.export(f)) <= TOL, f


@pytest.mark.gpu
@pytest.mark.parametrize("nseg", ["", "1", "5"])
def test_troughs_below_the_bed(eng, oracle, nseg, monkeypatch):
    """Waves far too high for the depth: columns whose elevation lies below the
    bed have levels there, past the depth nodes; their neighbours do not."""
    if nseg:
        monkeypatch.setenv("CFDWM_NSEG", nseg)
    s = make_sea(30, 9.0, 8.0, 6.0, seed=3, ndir=2).as_dict()
    args = ((0.0, 600.0, 0.0, 60.0), 41, 12, 9, 1.0, 0.5, 0.7, 1.5, s["depth"])
    o = oracle.sea(s).grid(*args)
    eta = o.export("ETA")
    assert 20 < np.sum(eta < -1.05 * s["depth"]) < 0.3 * eta.size
    g = eng.Sea(s, with_direct=False).grid(*args)
    for step in range(2):
        if step:
            g.force_update(1.6)
            o.force_update(1.6)
        for f in ("ETA", "UX", "UY", "UZ"):
            assert scaled_err(g.export(f), o.export(f)) <= TOL, (step, f)


@pytest.mark.gpu
def test_report_of_the_route(eng, monkeypatch):
    """Forms used, with what they took, or why not."""
    def grid(s, nx=32, depth=None):
        return eng.Sea(s, with_direct=False).grid((0.0, 100.0, 0.0, 60.0), nx, 16, 4, 0.5, 0.5, 0.7, 1.5,
                                                  depth or s["depth"])
    s = make_sea(12, 3.0, 9.0, 40.0, seed=5, ndir=2).as_dict()
    g = grid(s)
    info = g.qform_info()
    assert g.qform_reason() == "used" and info["products"] == 0
    assert info["nform"] == 1 + 3 * info["rank"] and info["basis_err"] <= 4e-15
    # 24 components in one 64-row tile up to 32, 2048 points, a cosine and a sine product
    assert info["mfma_flop"] == 64 * 32 * 4 * 2048 * info["nform"]
    few = grid(s, nx=1)                      # 256 points and levels: the pair loop up to 128
    assert few.qform_reason() == "used"
    small = eng.Sea(s, with_direct=False).grid((0.0, 9.0, 0.0, 9.0), 2, 2, 4, 0.5, 0.5, 0.7, 1.5, 40.0)
    assert small.qform_info() is None and small.qform_reason() == "fp64"
    assert grid(s, depth=41.0).qform_reason() == "grid deeper than the depth basis"
    r = dict(s, ramptime=np.linspace(1, 4, 24), starttime=np.zeros(24), duration=np.full(24, 1e6))
    assert grid(r).qform_reason() == "frequency ramps differ"
    one = make_sea(1, 3.0, 9.0, 40.0, seed=5).as_dict()
    assert grid(one).qform_reason() == "no second-order pairs"
    monkeypatch.setenv("CFDWM_QFORM", "0")
    off = grid(s)
    assert off.qform_info() is None and off.qform_reason() == "switched off"


@pytest.mark.gpu
def test_one_workspace_for_all_grids(eng, monkeypatch):
    """A grid's fields take the same memory with the forms as without, whatever
    the number of grids; the workspace goes when all have released it."""
    import torch
    s = make_sea(12, 3.0, 9.0, 40.0, seed=5, ndir=2).as_dict()

    def grids(n):
        return [eng.Sea(s, with_direct=False).grid((0.0, 999.0, 0.0, 999.0), 160, 160, 2, 0.0, 0.5, 0.7, 1.5, 40.0)
                for _ in range(n)]

    def used(n):
        torch.cuda.synchronize()
        a = torch.cuda.mem_get_info()[0]
        g = grids(n)
        return g, a - torch.cuda.mem_get_info()[0]
    monkeypatch.setenv("CFDWM_QFORM", "0")
    loop, plain = used(4)
    monkeypatch.delenv("CFDWM_QFORM")
    first = grids(1)
    values = first[0].qform_info()["nform"] * 4 * 160 * 160 * 8
    assert values > 40 << 20
    more, forms = used(4)
    assert forms < plain + values // 2
    free = torch.cuda.mem_get_info()[0]
    for g in first + more:
        g.release_workspace()
    assert torch.cuda.mem_get_info()[0] - free >= values
    more[0].refill()
    assert all(np.array_equal(more[0].export(f), first[0].export(f)) for f in ("ETA", "UX", "UY", "UZ"))
    assert scaled_err(more[0].export("UX"), loop[0].export("UX")) <= TOL


@pytest.mark.gpu
def test_fills_from_several_threads(eng):
    """Grids of different sizes (the shared workspace grows in between) filled and
    updated side by side give what each gives alone, bit for bit."""
    import threading

    def run(k, rounds):
        s = make_sea(10 + 9 * k, 3.0, 9.0, 40.0, seed=k, ndir=1 + k % 3).as_dict()
        nx = 24 + 20 * k
        g = eng.Sea(s, with_direct=False).grid((0.0, 300.0, 0.0, 90.0), nx, 20, 3, 0.0, 0.5, 0.7, 1.5, 40.0)
        assert g.qform_reason() == "used"
        out = []
        for r in range(rounds):
            g.refill() if r % 2 else g.force_update(0.75 + 0.5 * r)
            out.append([g.export(f) for f in ("ETA", "UX", "UZ")])
        return out
    ref = [run(k, 6) for k in range(4)]
    got, errors = [None] * 4, []

    def worker(k):
        try:
            got[k] = run(k, 6)
        except Exception as e:            # reported below, in the test's own thread
            errors.append((k, e))
    th = [threading.Thread(target=worker, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors
    for a, b in zip(ref, got):
        for p, q in zip(a, b):
            assert all(np.array_equal(x, y) for x, y in zip(p, q))
