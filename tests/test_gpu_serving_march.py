"""The march's buffers on a server whose memory budget binds: they hold no request back that fits without
them, a waiting request gets their room when the march ends, and kept ones count against the budget."""
import time

import numpy as np
import pytest

from eikonalsolvers.grids import ExtraParams, Grid3DCart
from eikonalsolvers.serving import request_bytes
from eikonalsolvers.synthetic import smooth_velocity

pytestmark = pytest.mark.gpu

EP = ExtraParams()


def _request(n, nsrc, seed):
    grd = Grid3DCart(hgrid=1.0, cooinit=(0.0, 0.0, 0.0), grsize=(n, n, n))
    rng = np.random.default_rng(seed)
    src = (0.1 + 0.8 * rng.random((nsrc, 3))) * (n - 1.0)
    recs = [rng.random((6, 3)) * (n - 1.0) for _ in range(nsrc)]
    return {"grd": grd, "vel": smooth_velocity(grd.grsize, seed), "src": src, "recs": recs,
            "obs": [np.full(6, 10.0) for _ in range(nsrc)], "std": [np.full(6, 0.1) for _ in range(nsrc)]}


def _submit(srv, m, r):
    return srv.submit_gradient(m, r["src"], r["recs"], r["obs"], r["std"], "gradvel", extraparams=EP)


def _same(m, r, got):
    gv, misf = m.gradient(r["src"], r["recs"], r["obs"], r["std"], "gradvel", extraparams=EP)
    assert np.linalg.norm(got[0] - gv) <= 1e-12 * np.linalg.norm(gv)
    assert got[-1] == pytest.approx(misf, rel=1e-12)


@pytest.mark.parametrize("sizes", [(8, 8), (5, 14)])
def test_requests_that_fit_without_the_march_run_together(eik, sizes):
    """Two gradient requests whose working sets just fit the budget side by side: equal ones (the first is
    granted no march), and a small one with a larger behind it (the small one's march gives its room back)."""
    reqs = [_request(100, k, 70 + k) for k in sizes]
    models = [eik.EikModel(r["vel"], r["grd"]) for r in reqs]
    b = [request_bytes(m, len(r["src"]), "gradient", extraparams=EP) for m, r in zip(models, reqs)]
    budget = int(1.02 * sum(b))
    print(f"together {sizes}: working sets {b}, budget {budget}", flush=True)
    with eik.Server(nslots=2, mem_budget=budget) as srv:
        # on empty slots, and for equal requests on slots that keep the pools of such a one
        for turn in range(2 if sizes[0] == sizes[1] else 1):
            t, hs = [], []
            for m, r in zip(models, reqs):
                t.append(time.perf_counter())
                hs.append(_submit(srv, m, r))
            out = [h.result() for h in hs]
            st = srv.stats()
            start = [x + h.queue_ms / 1e3 for x, h in zip(t, hs)]
            end = [x + (h.queue_ms + h.run_ms) / 1e3 for x, h in zip(t, hs)]
            print(f"  turn {turn}: start {start[1] - start[0]:.4f} s apart, first ran {end[0] - start[0]:.4f} s, {st}")
            assert start[1] < end[0], "the second request waited for the first"
            assert st["pool_bytes"] <= budget
            for m, r, o in zip(models, reqs, out):
                _same(m, r, o)
    for m in models:
        m.close()


def test_kept_march_buffers_count_against_the_budget(eik):
    """A request that marches, then one that takes nearly the whole budget: the slot gives up the buffers
    it kept."""
    small, large = _request(100, 5, 81), _request(100, 15, 82)
    models = [eik.EikModel(r["vel"], r["grd"]) for r in (small, large)]
    b = [request_bytes(m, len(r["src"]), "gradient", extraparams=EP) for m, r in zip(models, (small, large))]
    budget = int(1.02 * b[1])
    print(f"kept march buffers: working sets {b}, budget {budget}", flush=True)
    with eik.Server(nslots=1, mem_budget=budget) as srv:
        for m, r in zip(models, (small, large)):
            h = _submit(srv, m, r)
            _same(m, r, h.result())
            st = srv.stats()
            print(f"  rounds {h.stats['rounds']}, {st}")
            assert st["pool_bytes"] <= budget
            if r is small:
                assert h.stats["verify_rounds"] == 0, "the small request should march"
    for m in models:
        m.close()
