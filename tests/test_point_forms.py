"""Direct-mode points of long-crested seas through the split pair profiles on the
matrix cores: against the oracle, and against the pair loop (the same sea with one
component's direction an ulp away) at the edges of tiles, row blocks and segments."""
import numpy as np
import pytest

from cfdwavemaker_amd.seastate import make_sea

# FP64: rounding of sums over up to 1e4 pairs, exponents up to 100 eps.
# FP32: terms good to a few FP32 ulps, at most 130 in a row in a chain.
TOL = {"fp64": 1e-11, "fp32": 1e-5}
FIELDS = ("eta1", "eta2", "u", "v", "w", "p")


@pytest.fixture(scope="module")
def eng():
    from cfdwavemaker_amd import engine
    engine.load()
    return engine


def _sea(n, depth, **kw):
    s = make_sea(n, 3.0, 9.0, depth, seed=n, ndir=1).as_dict()
    s["theta"] = np.full(len(s["omega"]), 0.4)
    s.update(kw)
    return s


def _pair_loop(s):
    r = dict(s, theta=np.array(s["theta"], float))
    r["theta"][0] = np.nextafter(r["theta"][0], 1.0)
    return r


def _points(m, depth, seed, lo=-1.0, hi=2.0):
    rng = np.random.default_rng(seed)
    return (rng.uniform(0.0, 40.0, m), rng.uniform(-60.0, 90.0, m), rng.uniform(-30.0, 30.0, m),
            np.concatenate([rng.uniform(lo * depth, hi, m)]))


def _fields(eng, sea, q):
    import torch
    f = sea.eval_fields_device(*(torch.tensor(a, device="cuda") for a in q))
    return {k: v.cpu().numpy() for k, v in f.items()}


def _check(got, ref, tol):
    for k in FIELDS:
        ok = np.isfinite(ref[k])          # coth(k h) itself is not a number past k h = 710
        assert np.array_equal(ok, np.isfinite(got[k])), k
        scale = np.max(np.abs(ref[k][ok]), initial=0.0)
        err = np.max(np.abs(got[k] - ref[k])[ok], initial=0.0)
        assert err <= tol * scale or (scale == 0 and err == 0), (k, err, scale)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,m,depth", [(1, 5, 20.0), (2, 64, 20.0), (15, 65, 30.0), (16, 1, 30.0), (17, 63, 8.0),
                                       (32, 1000, 150.0), (33, 129, 50.0), (130, 300, 60.0)])
def test_against_the_pair_loop(eng, prec, n, m, depth):
    p = eng.FP64 if prec == "fp64" else eng.FP32
    extra = dict(bandwidth=0.8, cutoff=1.7, swl=0.5) if n % 2 else {}
    s = _sea(n, depth, **extra)
    q = _points(m, depth, n)
    _check(_fields(eng, eng.Sea(s, precision=p), q), _fields(eng, eng.Sea(_pair_loop(s)), q), TOL[prec])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nseg", ["1", "2", "7", "1000"])
def test_segments(eng, prec, nseg, monkeypatch):
    """Runs of the table that end anywhere: inside a row block, between two, in its first steps."""
    p = eng.FP64 if prec == "fp64" else eng.FP32
    s, q = _sea(50, 30.0), _points(70, 30.0, 3)
    ref = _fields(eng, eng.Sea(_pair_loop(s)), q)
    monkeypatch.setenv("CFDWM_NSEG", nseg)
    _check(_fields(eng, eng.Sea(s, precision=p), q), ref, TOL[prec])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_components_far_apart(eng, prec):
    """Rows of a block so far apart in k that the split leaves the number range in
    FP32: those waves go pair by pair."""
    p = eng.FP64 if prec == "fp64" else eng.FP32
    s = _sea(20, 400.0, omega=np.linspace(0.2, 6.0, 20), k=np.linspace(0.2, 6.0, 20) ** 2 / 9.81)
    q = _points(200, 400.0, 4)
    _check(_fields(eng, eng.Sea(s, precision=p), q), _fields(eng, eng.Sea(_pair_loop(s)), q), TOL[prec])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_raw_depths(eng, prec):
    """The second-order terms alone take z as given: above the surface and below the bed."""
    p = eng.FP64 if prec == "fp64" else eng.FP32
    s = _sea(40, 25.0)
    t, x, y, z = _points(300, 25.0, 5, lo=-2.5, hi=6.0)
    a, b = eng.Sea(s, precision=p), eng.Sea(_pair_loop(s))
    for kind in ("u2", "v2", "w2", "dp2"):
        g, r = a.eval(kind, t, x, y, z), b.eval(kind, t, x, y, z)
        # every point on its own: the profiles span many orders of magnitude
        # over these depths, so the scale is the largest field of points as high
        assert np.all(np.isfinite(g) == np.isfinite(r))
        order = np.argsort(z)
        scale = np.maximum.accumulate(np.abs(r[order]))
        deep = z[order] < -25.0
        scale = np.where(deep, np.max(np.abs(r)), scale)
        assert np.all(np.abs(g - r)[order] <= 4 * TOL[prec] * np.max(scale)), kind


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_against_the_oracle(eng, oracle, prec):
    p = eng.FP64 if prec == "fp64" else eng.FP32
    s = _sea(45, 35.0, ramptime=np.full(45, 20.0), starttime=np.zeros(45), duration=np.full(45, 30.0))
    t, x, y, z = _points(50, 35.0, 6)
    a, o = eng.Sea(s, precision=p), oracle.sea(s)
    for kind in ("u", "v", "w", "dp"):
        g, r = a.eval(kind, t, x, y, z), o.eval(kind, t, x, y, z)
        assert np.max(np.abs(g - r)) <= TOL[prec] * np.max(np.abs(r)), kind


@pytest.mark.gpu
def test_outputs_that_share_memory_with_inputs(eng):
    import torch
    s, q = _sea(30, 30.0), _points(100, 30.0, 7)
    sea = eng.Sea(s)
    ref = _fields(eng, sea, q)
    t, x, y, z = (torch.tensor(a, device="cuda") for a in q)
    u = torch.empty(100, dtype=torch.float64, device="cuda")
    eng.check(sea.L.cfdwm_eval_fields(sea.h, 99, t.data_ptr(), x.data_ptr(), y.data_ptr(), z.data_ptr(), None, None,
                                      u.data_ptr(), x[1:].data_ptr(), z.data_ptr(), None, 1), "cfdwm_eval_fields")
    assert np.array_equal(u[:99].cpu().numpy(), ref["u"][:99])
    assert np.array_equal(x[1:].cpu().numpy(), ref["v"][:99])
    assert np.array_equal(z[:99].cpu().numpy(), ref["w"][:99])


@pytest.mark.gpu
def test_unordered_components_take_the_pair_loop(eng):
    """k out of order: the split does not hold, the fields do not change."""
    s, q = _sea(40, 30.0), _points(80, 30.0, 8)
    o = np.random.default_rng(1).permutation(40)
    r = dict(s)
    for k in ("omega", "A", "k", "phase", "theta"):
        r[k] = np.asarray(s[k])[o]
    _check(_fields(eng, eng.Sea(r), q), _fields(eng, eng.Sea(_pair_loop(r)), q), TOL["fp64"])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,ndir,m", [(1, 3, 1), (7, 3, 65), (20, 5, 700)])
def test_eta2_beside_the_pair_loop(eng, prec, n, ndir, m):
    """Directional seas: eta2 asked for with the velocities goes along with their pair
    loop (every pair, filtered ones left out); alone it has its own pass."""
    import torch
    p = eng.FP64 if prec == "fp64" else eng.FP32
    s = make_sea(n, 3.0, 9.0, 30.0, seed=n, ndir=ndir).as_dict()
    s.update(bandwidth=0.7, cutoff=1.6)
    sea = eng.Sea(s, precision=p)
    q = [torch.tensor(a, device="cuda") for a in _points(m, 30.0, n)]
    a = sea.eval_fields_device(*q)
    b = sea.eval_fields_device(*q[:3], want=("eta1", "eta2"))
    for k in ("eta1", "eta2"):
        x, y = a[k].cpu().numpy(), b[k].cpu().numpy()
        assert np.max(np.abs(x - y)) <= TOL[prec] * np.max(np.abs(y)), k


def _kernels(eng, call):
    """The launches of a call, by the library's own timers."""
    eng.prof_enable(True)
    eng.prof_read()
    try:
        return call(), set(eng.prof_read())
    finally:
        eng.prof_enable(False)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 2, 40])
def test_switched_off(eng, prec, n, monkeypatch):
    """CFDWM_QFORM=0 at the call takes the pair loop of the same sea (whose tables
    then go up), without it the forms again."""
    s, q = _sea(n, 30.0), _points(70, 30.0, 9)
    sea = eng.Sea(s, precision=eng.FP64 if prec == "fp64" else eng.FP32)
    a, ka = _kernels(eng, lambda: _fields(eng, sea, q))
    monkeypatch.setenv("CFDWM_QFORM", "0")
    b, kb = _kernels(eng, lambda: _fields(eng, sea, q))
    monkeypatch.delenv("CFDWM_QFORM")
    c, kc = _kernels(eng, lambda: _fields(eng, sea, q))
    assert "k_point_forms" in ka and "k_point_forms" in kc
    assert "k_levels_points" in kb and "k_point_forms" not in kb
    _check(a, b, TOL[prec])
    assert all(np.array_equal(a[k], c[k]) for k in FIELDS)


@pytest.mark.gpu
@pytest.mark.parametrize("n,m", [(512, 400_000), (1024, 3_000_000)])
def test_memory_of_large_batches(eng, n, m):
    """The segments' totals stay within 256 MiB (2 MiB for the allocator's granules),
    and the result is that of small batches, which split the pairs otherwise."""
    import torch
    s = _sea(n, 30.0)
    sea = eng.Sea(s, precision=eng.FP32)
    t, x, y, z = (torch.tensor(a, device="cuda") for a in _points(m, 30.0, 10))
    u = torch.zeros(m, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]

    def call(a, b, out):
        eng.check(sea.L.cfdwm_eval_fields(sea.h, b - a, *(v[a:].data_ptr() for v in (t, x, y, z)), None, None,
                                          out.data_ptr(), None, None, None, 1), "cfdwm_eval_fields")
    call(0, m, u)
    assert free - torch.cuda.mem_get_info()[0] <= (256 + 2) << 20
    part = torch.zeros(2000, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for a in (0, m - 2000):
        call(a, a + 2000, part)
        assert float((part - u[a:a + 2000]).abs().max()) <= TOL["fp32"] * float(u.abs().max())


@pytest.mark.gpu
def test_more_points_than_a_launch_holds(eng):
    """2^30 points and some: four threads a point are more than a launch's 2^32.
    One array serves as t, x, y and z."""
    import torch
    n = (1 << 30) + 100
    q = torch.linspace(0.0, 30.0, n, dtype=torch.float64, device="cuda")
    u = torch.full((n,), 1e30, dtype=torch.float64, device="cuda")
    sea = eng.Sea(_sea(2, 30.0), precision=eng.FP32)
    p = q.data_ptr()
    torch.cuda.synchronize()
    eng.check(sea.L.cfdwm_eval_fields(sea.h, n, p, p, p, p, None, None, u.data_ptr(), None, None, None, 1),
              "cfdwm_eval_fields")
    for a in (0, (1 << 28) - 50, (1 << 29) - 50, n - 100):
        v = sea.eval_fields_device(*[q[a:a + 100].contiguous()] * 4)["u"]
        assert float(v.abs().max()) > 0 and torch.equal(v, u[a:a + 100]), a
    assert float(u.max()) < 1e29


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_one_component_against_the_oracle(eng, oracle, prec):
    """No pairs: the linear, diagonal and pressure terms alone (test_against_the_pair_loop's
    other sea of one component takes the point forms as well)."""
    s, (t, x, y, z) = _sea(1, 20.0), _points(40, 20.0, 11)
    sea, o = eng.Sea(s, precision=eng.FP64 if prec == "fp64" else eng.FP32), oracle.sea(s)
    for kind in ("eta1", "eta2", "u", "v", "w", "dp"):
        g, r = sea.eval(kind, t, x, y, z), o.eval(kind, t, x, y, z)
        assert np.max(np.abs(g - r)) <= TOL[prec] * np.max(np.abs(r)), kind


@pytest.mark.gpu
def test_long_chains(eng, monkeypatch):
    """512 components in FP32: up to 512 terms in a row in an accumulator, four times
    those of TOL, whose roundings add up as their square root."""
    s, q = _sea(512, 30.0), _points(300, 30.0, 12)
    got = _fields(eng, eng.Sea(s, precision=eng.FP32), q)
    monkeypatch.setenv("CFDWM_QFORM", "0")
    _check(got, _fields(eng, eng.Sea(s), q), 2 * TOL["fp32"])
