"""Lists of the ordered march at their limits.  A march whose lists are too short stops and the call is
solved by the tile solver (EIK_LIST_LIMIT shortens them here); a device round that lists more nodes
than its LDS buffer holds (3072 a block) loses none of them.  In FP64 both ways end at the tile
solver's bits."""
import time

import numpy as np
import pytest

import cases
from eikonalsolvers.grids import ExtraParams
from eikonalsolvers.synthetic import c5_request
from test_zz_no_alloc import _call

pytestmark = pytest.mark.gpu

MODELS = {
    "cart2d": lambda: cases.random2d(seed=31, n=(70, 61), nsrc=3),
    "cart3d": lambda: cases.random3d(seed=32, n=(25, 22, 19), nsrc=3),
    "sphere2d": cases.sphere2d,
    "sphere3d": cases.sphere3d,
}


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("kind", sorted(MODELS))
def test_short_lists_end_on_the_tile_solver(eik, monkeypatch, kind, refine):
    if kind == "sphere3d" and refine:
        pytest.skip("3D spheres have no refinement")
    grd, vel, src, recs = MODELS[kind]()
    ep = ExtraParams(refinearoundsrc=refine)
    monkeypatch.setenv("EIK_MARCH", "0")
    _, t0 = eik.eiktraveltime(vel, grd, src, recs, returntt=True, extraparams=ep)
    model = eik.EikModel(vel, grd)
    for mode in (1, 2):
        monkeypatch.setenv("EIK_MARCH", str(mode))
        for limit in (1, 30):  # the seeds alone, and a front some rounds on
            monkeypatch.setenv("EIK_LIST_LIMIT", str(limit))
            print(f"short lists {kind} refine={refine} mode={mode} limit={limit}", flush=True)
            at = time.perf_counter()
            _, t = eik.eiktraveltime(vel, grd, src, recs, returntt=True, extraparams=ep)
            took = time.perf_counter() - at
            st = eik.default_context().last_stats()
            for s in range(len(src)):
                assert np.array_equal(t[s], t0[s]), (mode, limit, s)
            if limit == 1 or mode == 1:  # (segments of 30 entries are enough for the smallest grids)
                assert st["verify_rounds"] >= 1, "the tile solver did not run"
            assert took < 1.0, "the march went on after its lists had overflowed"
            rc0, p0, g0 = _call("eik_traveltime", model, src, recs, ep, True)
            rc1, p1, g1 = _call("eik_traveltime_noalloc", model, src, recs, ep, True)
            assert rc0 == 0 and rc1 == 0
            assert np.array_equal(p1, p0) and np.array_equal(g1, g0), (mode, limit)
    model.close()


def test_more_newly_listed_nodes_than_a_round_collects(eik, monkeypatch):
    """222 sources on six 3D grids in one call: two blocks a source, on two XCDs, each running up to 1024
    nodes of a wide front a round, which wake about three new ones each.  (Nodes that both blocks list in
    one round once kept an entry each, and five calls in six did not end.)"""
    ep = ExtraParams()
    reqs = [c5_request(i) for i in (3, 10, 11, 23, 24, 28)]
    models = [eik.EikModel(r["vel"], r["grd"]) for r in reqs]
    print("wide rounds " + ", ".join(f"{r['grd'].grsize}x{len(r['src'])}" for r in reqs), flush=True)
    calls = [(m, r["src"], r["recs"]) for r, m in zip(reqs, models)]
    monkeypatch.setenv("EIK_MARCH", "0")
    p0 = eik.traveltime_batch(calls, extraparams=ep)
    monkeypatch.setenv("EIK_MARCH", "2")
    p = eik.traveltime_batch(calls, extraparams=ep)
    st = eik.default_context().last_stats()
    for a, b in zip(p0, p):
        for pa, pb in zip(a, b):
            assert np.array_equal(pa, pb)
    nodes = sum(len(r["src"]) * np.prod(r["grd"].grsize) for r in reqs)
    assert st["verify_rounds"] == 0 and st["node_updates"] < 2 * nodes, "the march did not solve the call itself"
    for m in models:
        m.close()


def test_unlike_grids_in_one_call_take_the_faster_solver(eik):
    """The same six grids go to the tile solver (the device rounds would leave most blocks idle beside the
    largest grid's: 841 ms against 308); three grids of like size march."""
    for ids, tiles in (((3, 10, 11, 23, 24, 28), True), ((10, 11, 24), False)):
        reqs = [c5_request(i) for i in ids]
        models = [eik.EikModel(r["vel"], r["grd"]) for r in reqs]
        print("unlike grids " + ", ".join(f"{r['grd'].grsize}x{len(r['src'])}" for r in reqs), flush=True)
        p = eik.traveltime_batch([(m, r["src"], r["recs"]) for r, m in zip(reqs, models)])
        assert (eik.default_context().last_stats()["verify_rounds"] > 0) == tiles
        for r, m, got in zip(reqs, models, p):
            for a, b in zip(m.traveltime(r["src"], r["recs"]), got):
                assert np.array_equal(a, b)
            m.close()


def test_noalloc_marches_many_small_sources(eik):
    """200 sources on a small grid fit the no-allocation block with the march's buffers."""
    grd, vel, src, _ = cases.random2d(seed=51, n=(61, 44), nsrc=200)
    recs = [src[:3] for _ in src]
    ep = ExtraParams(refinearoundsrc=False)
    model = eik.EikModel(vel, grd)
    print("noalloc 61x44 x 200", flush=True)
    rc0, p0, _ = _call("eik_traveltime", model, src, recs, ep, False)
    rc1, p1, _ = _call("eik_traveltime_noalloc", model, src, recs, ep, False)
    st = eik.default_context().last_stats()
    assert rc0 == 0 and rc1 == 0 and np.array_equal(p0, p1)
    assert st["verify_rounds"] == 0, "the tile solver solved it"
    model.close()
