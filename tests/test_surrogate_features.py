"""The surrogate's linear features at the edges of their component blocks (8 and 256
at a time) and level groups (4, 8 and 16 a pass), and the eta2 of points asked for alone."""
import ctypes as C

import numpy as np
import pytest

from cfdwavemaker_amd.seastate import make_sea

# against FP64 sums in numpy, of each field's largest value.  FP32: phases to
# 1e-7, exponents up to 60 at half an ulp; FP64: exponents up to 60 eps.
TOL = {"fp64": 1e-12, "fp32": 1e-5}


@pytest.fixture(scope="module")
def eng():
    from cfdwavemaker_amd import engine
    engine.load()
    return engine


def _reference(s, x, y, t, sigma, h):
    w, A, k, ph, th = (np.asarray(s[q], float)[:, None] for q in ("omega", "A", "k", "phase", "theta"))
    rt, ts, du = (np.asarray(s[q], float)[:, None] for q in ("ramptime", "starttime", "duration"))
    r = np.clip((t - ts) / (rt + 1e-12), 0, 1) * np.clip(1 - (t - ts - du + rt) / (rt + 1e-12), 0, 1)
    a = k * (np.cos(th) * x + np.sin(th) * y) - w * t + ph
    c, sn = np.cos(a) * r, np.sin(a) * r
    g, rho, d = 9.81, s["rho"], s["depth"]
    eta = (A * c).sum(0)
    z = eta + sigma[:, None] * (h + eta)
    zt, zp = np.maximum(z, 0), np.minimum(z, 0)
    out = [eta]
    den = 1 / (1 + np.exp(-2 * k * d))
    for l in range(len(sigma)):
        E, G = np.exp(k * zp[l]), np.exp(-k * (zp[l] + 2 * d))
        ch, sh = (E + G) * den, (E - G) * den
        out += [(A * g * k / w * np.cos(th) * c * ch).sum(0) + zt[l] * (A * w * k * np.cos(th) * c).sum(0),
                (A * g * k / w * np.sin(th) * c * ch).sum(0) + zt[l] * (A * w * k * np.sin(th) * c).sum(0),
                (A * g * k / w * sn * sh).sum(0) + zt[l] * (A * w * k / np.tanh(k * d) * sn).sum(0),
                (A * rho * g * c * ch).sum(0) + zt[l] * (A * rho * g * k * c).sum(0)]
    return np.stack(out, 1)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nfreq,ndir,nlev,n,depth", [(1, 1, 1, 1, 20.0), (7, 1, 4, 64, 30.0), (8, 1, 5, 257, 90.0),
                                                     (3, 3, 16, 255, 8.0), (32, 8, 17, 300, 60.0),
                                                     (257, 1, 32, 70, 150.0)])
def test_features_vs_numpy(eng, prec, nfreq, ndir, nlev, n, depth):
    import torch
    s = make_sea(nfreq, 2.0, 8.0, depth, seed=nfreq, ndir=ndir).as_dict()
    N = len(s["omega"])
    rng = np.random.default_rng(N)
    s.update(ramptime=rng.uniform(1.0, 40.0, N), starttime=np.zeros(N), duration=np.full(N, 300.0))
    s.setdefault("rho", 1025.0)
    sea = eng.Sea(s, precision=eng.FP64 if prec == "fp64" else eng.FP32, with_direct=False)
    x, y, t, h = rng.uniform(0, 400, n), rng.uniform(0, 400, n), 11.5, 0.9 * depth
    sigma = np.sort(rng.uniform(-1.0, 0.0, nlev))
    if nlev > 4:
        sigma[[0, 3]] = sigma[[3, 0]]                 # levels need not ascend
    nx = 3 + 3 * ((nlev + 1) // 2) + 2
    X = torch.full((n, nx + 3), np.nan, dtype=torch.float32, device="cuda")
    L = torch.full((n, 1 + 4 * nlev), np.nan, dtype=torch.float32, device="cuda")
    xd, yd = (torch.tensor(a, device="cuda") for a in (x, y))
    torch.cuda.synchronize()
    eng.check(sea.L.cfdwm_surrogate_features(sea.h, n, xd.data_ptr(), yd.data_ptr(), t, h, nlev,
                                             sigma.ctypes.data_as(C.POINTER(C.c_double)), 2, 0.05, nx + 3,
                                             X.data_ptr(), L.data_ptr()), "cfdwm_surrogate_features")
    eng.sync()
    L, X = L.cpu().numpy().astype(float), X.cpu().numpy()
    assert not np.isnan(X).any()
    ref = _reference(s, x, y, t, sigma, h)
    f = 6e-8 if prec == "fp64" else 0.0               # the outputs are FP32
    for j in range(1 + 4 * nlev):
        scale = np.max(np.abs(ref[:, 0])) if j == 0 else np.max(np.abs(ref[:, 1 + (j - 1) % 4::4]))
        assert np.max(np.abs(L[:, j] - ref[:, j])) <= (TOL[prec] + f) * scale, j
    assert np.array_equal(X[:, 3], L[:, 1].astype(np.float32)) and np.all(X[:, nx - 1] == np.float32(0.05))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2048, 3001])
@pytest.mark.parametrize("nfreq,ndir", [(1, 3), (5, 5), (40, 8)])
def test_eta2_alone_is_the_same(eng, nfreq, ndir, n):
    """A call for eta2 alone (the gradients and eta1 left out) gives the bits of the whole call."""
    import torch
    sea = eng.Sea(make_sea(nfreq, 2.0, 8.0, 40.0, seed=3, ndir=ndir).as_dict(), precision=eng.FP32)
    q = [torch.rand(n, dtype=torch.float64, device="cuda") * 50 for _ in range(3)]
    a = sea.eval_fields_device(*q, want=("eta2",))["eta2"]
    b = sea.eval_fields_device(*q, want=("eta1", "eta2"))["eta2"]
    assert torch.equal(a, b)
