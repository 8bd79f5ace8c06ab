"""A device round of the ordered march that lists more nodes than its LDS buffer holds (3072 a block)
loses none of them: the tile solver's bits in FP64."""
import numpy as np
import pytest

from eikonalsolvers.grids import ExtraParams
from eikonalsolvers.synthetic import c5_request

pytestmark = pytest.mark.gpu


def test_more_newly_listed_nodes_than_a_round_collects(eik, monkeypatch):
    """222 sources on six 3D grids in one call: two blocks a source, each running up to 1024 nodes of
    a wide front a round, which wake about three new ones each."""
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
