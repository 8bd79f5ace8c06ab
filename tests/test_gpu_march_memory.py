"""The march's buffers are the first to go.  A call that fits the device on the tile solver fits it with
the march enabled too, whatever the march took first, kept from an earlier call, or took from the other
half of a split call.  EIK_POOL_LIMIT makes the device small; the limit is the least the tile solver runs
with, found by bisection on fresh contexts."""
import numpy as np
import pytest

from eikonalsolvers.grids import ExtraParams, Grid3DCart
from eikonalsolvers.synthetic import smooth_velocity

pytestmark = pytest.mark.gpu

SIZES = {"one stream": ((40, 36, 33), 6), "split": ((96, 96, 96), 15)}  # (split: 3 x 2^22 source-nodes and more)


def _call(n, nsrc, seed=9):
    grd = Grid3DCart(hgrid=1.0, cooinit=(0.0, 0.0, 0.0), grsize=n)
    rng = np.random.default_rng(seed)
    top = np.array(n) - 1.0
    src = (0.1 + 0.8 * rng.random((nsrc, 3))) * top
    recs = [rng.random((5, 3)) * top for _ in range(nsrc)]
    obs = [np.full(5, 4.0) for _ in range(nsrc)]
    std = [np.full(5, 0.1) for _ in range(nsrc)]
    return grd, smooth_velocity(n, 77), src, recs, obs, std


def _run(eik, ctx, kind, args, nsrc=None):
    grd, vel, src, recs, obs, std = args
    model = eik.EikModel(vel, grd, ctx=ctx)
    k = len(src) if nsrc is None else nsrc
    try:
        if kind == "traveltime":
            return [np.array(p) for p in model.traveltime(src[:k], recs[:k], extraparams=ExtraParams())]
        gv, m = model.gradient(src[:k], recs[:k], obs[:k], std[:k], "gradvel", extraparams=ExtraParams())
        return [np.array(gv), np.array([m])]
    finally:
        model.close()


def _least(eik, monkeypatch, kind, args):
    """The least EIK_POOL_LIMIT (bytes, within 1/200) that a fresh context runs the call with on tiles."""
    monkeypatch.setenv("EIK_MARCH", "0")
    n, s = np.prod(args[0].grsize), len(args[2])
    lo, hi = 8 * n * s, 400 * n * s
    while hi - lo > hi // 200:
        mid = (lo + hi) // 2
        monkeypatch.setenv("EIK_POOL_LIMIT", str(mid))
        try:
            _run(eik, eik.Context(0), kind, args)
            hi = mid
        except MemoryError:
            lo = mid
    return hi


@pytest.mark.parametrize("kind", ["traveltime", "gradient"])
@pytest.mark.parametrize("how", sorted(SIZES))
def test_what_fits_on_tiles_fits_with_the_march(eik, monkeypatch, how, kind):
    args = _call(*SIZES[how])
    limit = _least(eik, monkeypatch, kind, args)
    per = limit / (np.prod(args[0].grsize) * len(args[2]))
    print(f"march memory {how} {kind}: least limit {limit} B, {per:.1f} a source-node", flush=True)
    monkeypatch.delenv("EIK_MARCH")
    monkeypatch.delenv("EIK_POOL_LIMIT")
    want = _run(eik, eik.Context(0), kind, args)
    # (two streams take their buffers in either order: a little room for what is freed late)
    for room in (1.02, 1.2, 1.6, 2.5):
        monkeypatch.setenv("EIK_POOL_LIMIT", str(int(room * limit)))
        ctx = eik.Context(0)
        for k in (2, None, 2, None):  # a small call's march buffers are kept, and in the way of the whole
            got = _run(eik, ctx, kind, args, k)
        for a, b in zip(want, got):
            assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(a), (room, kind)
    monkeypatch.delenv("EIK_POOL_LIMIT")
    got = _run(eik, ctx, kind, args)  # and the context is sound afterwards
    for a, b in zip(want, got):
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(a)
