"""The ordered march (eik_march.hip), as one workgroup per source and as whole-device rounds, against
the tile solver and the oracle's heap: the same traveltimes bit for bit, in FP64 and in the mixed
precision (both solvers end at the local replay's fixed point, which does not depend on the order
of the replays).  Grids around the brick edges (4 in 3D, 8 in 2D), down to two nodes along an axis,
every grid kind, with and without refinement; a list longer than what a workgroup keeps in LDS; a
constant-velocity model, whose equal values make cascade keys and ties (to rounding there).
"""
import numpy as np
import pytest

import cases
from eikonalsolvers.grids import ExtraParams, Grid2DCart, Grid2DSphere, Grid3DCart, Grid3DSphere

pytestmark = pytest.mark.gpu

SHAPES = {
    "cart2d": [(2, 2), (3, 9), (8, 8), (9, 17), (65, 7), (40, 33)],
    "sphere2d": [(2, 8), (7, 9), (31, 24)],
    "cart3d": [(2, 2, 2), (4, 4, 4), (5, 3, 9), (13, 12, 11), (33, 8, 21)],
    "sphere3d": [(2, 4, 5), (6, 9, 7), (13, 8, 12)],
}


def _grid(kind, n):
    if kind == "cart2d":
        return Grid2DCart(hgrid=0.5, cooinit=(1.0, -2.0), grsize=n)
    if kind == "cart3d":
        return Grid3DCart(hgrid=2.0, cooinit=(0.0, 3.0, 1.0), grsize=n)
    if kind == "sphere2d":
        return Grid2DSphere(Δr=2.0, Δθ=0.2, grsize=n, cooinit=(6251.0, 40.0))
    return Grid3DSphere(Δr=2.0, Δθ=0.2, Δφ=0.2, grsize=n, cooinit=(6300.0, 30.0, 10.0))


def _axes(grd):
    if hasattr(grd, "hgrid"):
        return [c + grd.hgrid * np.arange(m) for c, m in zip(grd.cooinit, grd.grsize)]
    return list(grd.axes())


def _setup(kind, n, nsrc, seed):
    grd = _grid(kind, n)
    vel = cases.smooth_field(n, seed, passes=2, lo=1.5, hi=6.0, base=3.5, amp=0.8)
    ax = _axes(grd)
    lo, hi = np.array([a[0] for a in ax]), np.array([a[-1] for a in ax])
    rng = np.random.default_rng(seed)
    src = lo + rng.uniform(0.03, 0.97, size=(nsrc, len(n))) * (hi - lo)
    recs = [lo + rng.uniform(0, 1, size=(3, len(n))) * (hi - lo) for _ in range(nsrc)]
    return grd, vel, src, recs


def _solve(eik, monkeypatch, mode, setup, ep):
    monkeypatch.setenv("EIK_MARCH", str(mode))
    grd, vel, src, recs = setup
    return eik.eiktraveltime(vel, grd, src, recs, returntt=True, extraparams=ep)


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("kind", sorted(SHAPES))
def test_march_equals_tiles_and_heap(eik, oracle, monkeypatch, kind, refine):
    if kind == "sphere3d" and refine:
        pytest.skip("3D spheres have no refinement")
    for k, n in enumerate(SHAPES[kind]):
        for nsrc in (1, 5):
            setup = _setup(kind, n, nsrc, 100 * k + nsrc)
            for prec in ("fp64", "mixed"):
                ep = ExtraParams(refinearoundsrc=refine, precision=prec)
                print(f"march {kind} {n} x {nsrc} {prec} refine={refine}", flush=True)
                p0, t0 = _solve(eik, monkeypatch, 0, setup, ep)
                for mode in (1, 2):
                    p, t = _solve(eik, monkeypatch, mode, setup, ep)
                    for s in range(nsrc):
                        assert np.array_equal(t[s], t0[s]), (mode, n, s)
                        assert np.array_equal(p[s], p0[s]), (mode, n, s)
            _, to = oracle.traveltime(setup[1], setup[0], setup[2], setup[3], returntt=True,
                                      extraparams=ExtraParams(refinearoundsrc=refine))
            _, t = _solve(eik, monkeypatch, 2, setup, ExtraParams(refinearoundsrc=refine))
            for s in range(nsrc):
                assert np.allclose(t[s], to[s], rtol=1e-12, atol=0), (n, s)


@pytest.mark.parametrize("n,nsrc", [((72, 64, 56), 1), ((70, 75, 33), 17)])
def test_march_long_lists(eik, monkeypatch, n, nsrc):
    setup = _setup("cart3d", n, nsrc, 7)
    print(f"march long lists {n} x {nsrc}", flush=True)
    _, t0 = _solve(eik, monkeypatch, 0, setup, ExtraParams())
    for mode in (1, 2):
        _, t = _solve(eik, monkeypatch, mode, setup, ExtraParams())
        for s in range(nsrc):
            assert np.array_equal(t[s], t0[s]), (mode, s)


@pytest.mark.parametrize("n", [(33, 26), (17, 14, 12)])
def test_march_ties(eik, monkeypatch, n):
    """Constant velocity, sources on a node and half-way between nodes: whole fronts of equal values.
    Both solvers then agree to rounding (1e-12 relative: a tied node may take either side)."""
    grd = _grid("cart2d" if len(n) == 2 else "cart3d", n)
    o, h = np.array(grd.cooinit), grd.hgrid
    src = np.array([o + h * (np.array(n) // 2), o + h * (np.array(n) // 3 + 0.5)])
    setup = (grd, np.full(n, 2.0), src, [src[:1] + 0.1 * h, src[1:] + 0.1 * h])
    for refine in (False, True):
        ep = ExtraParams(refinearoundsrc=refine)
        print(f"march ties {n} refine={refine}", flush=True)
        _, t0 = _solve(eik, monkeypatch, 0, setup, ep)
        for mode in (1, 2):
            _, t = _solve(eik, monkeypatch, mode, setup, ep)
            for s in range(2):
                assert np.allclose(t[s], t0[s], rtol=1e-12, atol=0), (mode, s)
