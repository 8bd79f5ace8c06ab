"""The march orders nodes by an expected value held as a float; the values themselves are doubles.
Models whose times leave the float range, in part (an inclusion of next to no velocity) or as a whole,
are solved all the same: the oracle's heap to rounding.  Where all
expected values are one number ("slow": the largest float, "faster": underflow) the order means nothing,
the march circulates, and the tile solver takes the call over at the march's limit of rounds."""
import numpy as np
import pytest

import cases
from eikonalsolvers.grids import ExtraParams

pytestmark = pytest.mark.gpu

SCALE = {"wall": None, "slow": 1e-40, "fast": 1e42, "faster": 1e46}


@pytest.mark.parametrize("refine", [False, True])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("how", sorted(SCALE))
def test_times_beyond_the_float_range(eik, oracle, monkeypatch, how, dim, refine):
    grd, vel, src, recs = (cases.random2d(seed=41, n=(34, 29), nsrc=2) if dim == 2 else
                           cases.random3d(seed=42, n=(14, 13, 11), nsrc=2))
    vel = vel.copy()
    if how == "wall":
        vel[vel.shape[0] // 2 - 1:vel.shape[0] // 2 + 2, 4:7] = 1e-42
    else:
        vel *= SCALE[how]
    ep = ExtraParams(refinearoundsrc=refine)
    _, to = oracle.traveltime(vel, grd, src, recs, returntt=True, extraparams=ep)
    for mode in (1, 2):
        monkeypatch.setenv("EIK_MARCH", str(mode))
        print(f"range {how} {dim}D refine={refine} mode={mode}", flush=True)
        _, t = eik.eiktraveltime(vel, grd, src, recs, returntt=True, extraparams=ep)
        if how == "fast":
            assert eik.default_context().last_stats()["verify_rounds"] == 0, "the march did not solve it itself"
        for s in range(len(src)):
            assert np.allclose(t[s], to[s], rtol=1e-12, atol=0), (mode, s)
