"""Seas with components of k h > 710: coth(k h) there is not a number in FP64,
and with it the vertical Taylor gradient and the s-grid's w.  Everything that
does not contain it stays as good as in shallower water."""
import numpy as np
import pytest

from cfdwavemaker_amd.seastate import make_sea, wavenumber

pytestmark = pytest.mark.gpu
DEPTH = 1000.0


def _sea(n=24, theta=None):
    s = make_sea(n, 3.0, 9.0, DEPTH, seed=n, ndir=1).as_dict()
    s["omega"] = np.linspace(0.4, 3.0, n)
    s["k"] = wavenumber(s["omega"], DEPTH)
    assert np.max(s["k"]) * DEPTH > 710.0
    s["theta"] = np.full(n, 0.4) if theta is None else theta
    return s


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_query_of_u_and_v_beside_a_w_that_is_no_number(prec):
    """At a node of the bed level and the time of the grid's first slot the
    interpolation is the node value itself (FP32: but for the rounding of the
    depth map, the library's 2e-5 of the field); elsewhere it is finite."""
    from cfdwavemaker_amd import engine as eng
    sea = eng.Sea(_sea(), precision=eng.FP64 if prec == "fp64" else eng.FP32, with_direct=False)
    nx, ny, nl = 6, 5, 7
    g = sea.grid((0.0, 50.0, 0.0, 40.0), nx, ny, nl, 0.0, 0.5, 0.7, 1.5, DEPTH)
    node = {f: g.export(f).reshape(4, nx, ny, nl)[1, :, :, 0].ravel() for f in ("UX", "UY", "UZ")}
    assert np.all(np.isnan(node["UZ"])) and np.all(np.isfinite(node["UX"])) and np.any(node["UX"])
    x, y = (a.ravel() for a in np.meshgrid(10.0 * np.arange(nx), 10.0 * np.arange(ny), indexing="ij"))
    q = g.query(0.0, x, y, -DEPTH)
    for k, f in ((1, "UX"), (2, "UY")):
        tol = 0.0 if prec == "fp64" else 2e-5 * np.max(np.abs(g.export(f)))
        assert np.max(np.abs(q[:, k] - node[f])) <= tol, f
    rng = np.random.default_rng(1)
    q = g.query(rng.uniform(0, 0.5, 300), rng.uniform(-5, 55, 300), rng.uniform(-5, 45, 300), rng.uniform(-DEPTH, 1, 300))
    assert np.all(np.isfinite(q[:, :3])) and np.all(np.isnan(q[:, 3]))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_points_without_taylor_terms(prec):
    """The second-order members (no Taylor terms asked for) of a long-crested sea
    against the pair loop, which the same sea takes with its components in
    descending order.  Tolerance: FP64 rounding of sums over 276 pairs; FP32
    terms good to a few ulps, at most 24 in a chain."""
    from cfdwavemaker_amd import engine as eng
    s = _sea()
    r = dict(s, **{k: np.asarray(s[k])[::-1].copy() for k in ("omega", "A", "k", "phase", "theta")})
    a = eng.Sea(s, precision=eng.FP64 if prec == "fp64" else eng.FP32)
    b = eng.Sea(r)
    rng = np.random.default_rng(2)
    q = rng.uniform(0, 40, 90), rng.uniform(-60, 90, 90), rng.uniform(-30, 30, 90), rng.uniform(-30.0, 0.0, 90)
    for kind in ("u2", "w2"):
        g, ref = a.eval(kind, *q), b.eval(kind, *q)
        assert np.all(np.isfinite(ref)) and np.any(ref)
        assert np.max(np.abs(g - ref)) <= (1e-11 if prec == "fp64" else 1e-5) * np.max(np.abs(ref)), kind


@pytest.mark.parametrize("depth", [900.0, 2200.0])
def test_fp64_forms_in_deep_water(depth, monkeypatch):
    """kmax h of 570 and 1400, towards the largest the depth nodes serve, against the
    pair loop; tolerance as in shallower water (rounding of sums over 700 pairs).
    (One direction: across directions the combined wavenumbers reach beyond kmax.)"""
    from cfdwavemaker_amd import engine as eng
    s = make_sea(38, 3.0, 9.0, depth, seed=4, ndir=1).as_dict()
    s["theta"] = np.full(38, 0.4)
    args = ((0.0, 310.0, 0.0, 150.0), 32, 16, 9, 0.5, 0.5, 0.7, 1.5, depth)
    forms = eng.Sea(s, with_direct=False).grid(*args)
    monkeypatch.setenv("CFDWM_QFORM", "0")
    loop = eng.Sea(s, with_direct=False).grid(*args)
    assert forms.qform_reason() == "used" and loop.qform_reason() == "switched off"
    for f in ("ETA", "UX", "UY") + (("UZ",) if depth < 1000 else ()):
        a, b = forms.export(f), loop.export(f)
        assert np.any(b) and np.max(np.abs(a - b)) <= 1e-11 * np.max(np.abs(b)), f
