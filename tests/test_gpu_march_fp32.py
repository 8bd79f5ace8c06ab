"""The FP32 march, as one workgroup per source and as device rounds, on Cartesian grids: within the FP32
mode's tolerances of the heap (relative L2 and 99.5 % of the nodes, receivers of the random models), on
models whose equal values make near-ties too, and ended by itself (a march that circulates among
near-ties would go on to its round limit and then to the tile solver)."""
import numpy as np
import pytest

import cases
from eikonalsolvers.grids import ExtraParams, Grid2DCart, Grid3DCart

pytestmark = pytest.mark.gpu


def _ties(n, layered):
    grd = (Grid2DCart if len(n) == 2 else Grid3DCart)(hgrid=1.0, cooinit=(0.0,) * len(n), grsize=n)
    vel = np.full(n, 2.0)
    if layered:
        vel += 0.5 * (np.arange(n[-1]) // 6)
    top = np.array(n) - 1.0
    src = np.array([np.floor(0.5 * top), 0.3 * top + 0.5])  # on a node, and off every node
    recs = [np.linspace(0.1, 0.9, 4)[:, None] * top for _ in range(2)]
    return grd, vel, src, recs


MODELS = {
    "rand2d": cases.random2d,
    "rand3d": cases.random3d,
    "const2d": lambda: _ties((71, 58), False),
    "const3d": lambda: _ties((27, 24, 21), False),
    "layers2d": lambda: _ties((71, 58), True),
    "layers3d": lambda: _ties((27, 24, 21), True),
}


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("name", sorted(MODELS))
def test_fp32_march_within_tolerance(eik, oracle, monkeypatch, name, mode):
    grd, vel, src, recs = MODELS[name]()
    monkeypatch.setenv("EIK_MARCH", str(mode))
    for refine in (False, True):
        print(f"march fp32 {name} mode={mode} refine={refine}", flush=True)
        pg, tg = eik.eiktraveltime(vel, grd, src, recs, returntt=True,
                                   extraparams=ExtraParams(precision="fp32", refinearoundsrc=refine))
        st = eik.default_context().last_stats()
        po, to = oracle.traveltime(vel, grd, src, recs, returntt=True, extraparams=ExtraParams(refinearoundsrc=refine))
        assert st["verify_rounds"] == 0, "the march did not end by itself"
        for s in range(len(tg)):
            rel = np.abs(tg[s] - to[s]) / np.maximum(np.abs(to[s]), 1e-300)
            q = float(np.quantile(rel, 0.995))
            l2 = np.linalg.norm(tg[s] - to[s]) / np.linalg.norm(to[s])
            print(f"  src {s}: 99.5% {q:.3e}, rel L2 {l2:.3e}, rounds {st['rounds']}")
            assert l2 <= 1e-4 and q <= 1e-4
            if name.startswith("rand"):
                assert np.all(np.abs(pg[s] - po[s]) <= 1e-5 * np.abs(po[s]))
