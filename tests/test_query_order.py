"""Cell-ordered spline queries: a batch large enough to be sorted by cell
(65,536 queries or more) returns bit for bit what the same queries return in
the caller's order (batches below that size, whose results the golden query
vectors pin), for the host FP64 entry and the device FP32 entry, in both
grid precisions."""
import numpy as np
import pytest

from tests.conftest import golden, sea_from_golden
from tests.golden.cases import GRID_CASE

pytestmark = pytest.mark.gpu

N_BIG, N_CHUNK = 200_000, 50_000
# the golden grid (35 columns) and a 64 x 48 column grid (12-bit sort keys)
SHAPES = {"golden": GRID_CASE,
          "64x48": dict(GRID_CASE, domain=(0.0, 630.0, -235.0, 235.0), nx=64, ny=48, nl=8)}


def _grid(prec, shape):
    from cfdwavemaker_amd import engine as eng
    c = SHAPES[shape]
    sea = eng.Sea(sea_from_golden(golden("points.npz"), "B"), precision=prec, with_direct=False)
    g = sea.grid(c["domain"], c["nx"], c["ny"], c["nl"], c["t0"], c["dt"], c["tan_a"], c["tan_b"], c["depth"])
    return sea, g


def _points(seed, shape):
    c = SHAPES[shape]
    rng = np.random.default_rng(seed)
    x0, x1, y0, y1 = c["domain"]
    # a margin outside the domain exercises the edge clamps
    x = rng.uniform(x0 - 5.0, x1 + 5.0, N_BIG)
    y = rng.uniform(y0 - 5.0, y1 + 5.0, N_BIG)
    z = rng.uniform(-c["depth"], 1.0, N_BIG)
    t = rng.uniform(c["t0"], c["t0"] + c["dt"], N_BIG)
    return t, x, y, z


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_host_queries_cell_order_matches_caller_order(precision, shape):
    from cfdwavemaker_amd import engine as eng
    prec = eng.FP64 if precision == "fp64" else eng.FP32
    sea, g = _grid(prec, shape)
    t, x, y, z = _points(11, shape)
    big = g.query(t, x, y, z)
    parts = [g.query(t[a:a + N_CHUNK], x[a:a + N_CHUNK], y[a:a + N_CHUNK], z[a:a + N_CHUNK])
             for a in range(0, N_BIG, N_CHUNK)]
    small = np.concatenate(parts)
    assert np.all(np.isfinite(big))
    assert np.array_equal(big, small)


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_device_f32_queries_cell_order_matches_caller_order(precision, shape):
    import torch
    from cfdwavemaker_amd import engine as eng
    prec = eng.FP64 if precision == "fp64" else eng.FP32
    sea, g = _grid(prec, shape)
    t, x, y, z = _points(12, shape)
    tq = float(t[0])
    dev = torch.device("cuda:0")
    X, Y, Z = (torch.tensor(a, dtype=torch.float32, device=dev) for a in (x, y, z))
    big = [torch.empty(N_BIG, dtype=torch.float32, device=dev) for _ in range(4)]
    small = [torch.empty(N_BIG, dtype=torch.float32, device=dev) for _ in range(4)]
    g.query_device_f32(N_BIG, tq, X.data_ptr(), Y.data_ptr(), Z.data_ptr(), *[o.data_ptr() for o in big])
    eng.sync()
    for a in range(0, N_BIG, N_CHUNK):
        g.query_device_f32(N_CHUNK, tq, X[a:].data_ptr(), Y[a:].data_ptr(), Z[a:].data_ptr(),
                           *[o[a:].data_ptr() for o in small])
    eng.sync()
    for b, s in zip(big, small):
        b, s = b.cpu().numpy(), s.cpu().numpy()
        assert np.all(np.isfinite(b))
        assert np.array_equal(b, s)


@pytest.mark.parametrize("nx,ny,nl,n", [(1, 1, 1, 65536), (1, 37, 3, 65537), (130, 1, 5, 70_001), (67, 131, 4, 300_003),
                                        (300, 260, 2, 1_100_000)])
def test_tiles_of_odd_grids(nx, ny, nl, n):
    """Grids one column or level wide, tiles that overhang the grid, batch sizes
    around the ordering threshold, the blocks' shares and the largest tile
    counts; a cluster of queries in one cell and a run of NaN coordinates (which
    clamp to an edge cell): bit for bit what batches below the threshold give."""
    from cfdwavemaker_amd import engine as eng
    import torch
    from cfdwavemaker_amd.seastate import make_sea
    sea = eng.Sea(make_sea(6, 1.0, 8.0, 20.0, seed=1, ndir=2).as_dict(), precision=eng.FP32, with_direct=False)
    dom = (3.0, 3.0 + 2.0 * (nx - 1), -4.0, -4.0 + 3.0 * (ny - 1))
    g = sea.grid(dom, nx, ny, nl, 0.0, 0.5, 0.7, 1.5, 20.0)
    rng = np.random.default_rng(n)
    x = rng.uniform(dom[0] - 5, dom[1] + 5, n).astype(np.float32)
    y = rng.uniform(dom[2] - 5, dom[3] + 5, n).astype(np.float32)
    z = rng.uniform(-21.0, 2.0, n).astype(np.float32)
    x[: n // 3], y[: n // 3] = dom[0], dom[2]
    x[n // 2: n // 2 + 70] = np.nan
    X, Y, Z = (torch.tensor(a, device="cuda") for a in (x, y, z))
    big = torch.full((n, 4), 7.0, dtype=torch.float32, device="cuda")
    small = torch.full((n, 4), 8.0, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    g.kinematics_device_f32(n, 0.2, X.data_ptr(), Y.data_ptr(), Z.data_ptr(), big.data_ptr())
    for a in range(0, n, 50_000):
        m = min(50_000, n - a)
        g.kinematics_device_f32(m, 0.2, X[a:].data_ptr(), Y[a:].data_ptr(), Z[a:].data_ptr(), small[a:].data_ptr())
    eng.sync()
    assert torch.equal(torch.nan_to_num(big, nan=1e30), torch.nan_to_num(small, nan=1e30))
