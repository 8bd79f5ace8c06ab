"""The adjoint's tiles at their edges, against the CPU oracle.

One node beyond, at and short of a multiple of the tile (16 in 2D, 8 in 3D), a grid of a single tile, one
thinner than the halo, and more tiles than one block of the selection takes (1024).  The same linear system as the
oracle's in another summation order: the 1e-7 relative L2 of the other gradient tests.
"""
import numpy as np
import pytest

from cases import random2d, random3d, sphere2d, sphere3d
from eikonalsolvers.grids import ExtraParams
from test_gpu_gradient import _obs, _rel_l2

pytestmark = pytest.mark.gpu

GRIDS = {
    "one_tile": lambda: random2d(seed=21, n=(12, 11), nsrc=2, nrec=5),
    "edge2d": lambda: random2d(seed=22, n=(33, 16), nsrc=3, nrec=7),
    "short2d": lambda: random2d(seed=23, n=(31, 47), nsrc=2, nrec=7),
    "thin2d": lambda: random2d(seed=24, n=(130, 9), nsrc=2, nrec=7),
    "many2d": lambda: random2d(seed=25, n=(530, 513), nsrc=2, nrec=9),
    "edge3d": lambda: random3d(seed=26, n=(17, 16, 15), nsrc=2, nrec=7),
    "sph2d": sphere2d,
    "sph3d": sphere3d,
}


@pytest.mark.parametrize("name", list(GRIDS))
def test_gradient_at_tile_edges_matches_oracle(eik, oracle, name):
    grd, vel, src, recs = GRIDS[name]()
    ep = ExtraParams(refinearoundsrc=False)
    print(f"case={name} grid={grd.grsize} nsrc={len(src)}", flush=True)
    obs, std = _obs(oracle, vel, grd, src, recs, ep, 91)
    gg, mg = eik.eikgradient(vel, grd, src, recs, obs, std, "gradvel", extraparams=ep)
    go, mo = oracle.gradient(vel, grd, src, recs, obs, std, "gradvel", extraparams=ep)
    e = _rel_l2(gg, go)
    print(f"  misfit gpu {mg:.12e} oracle {mo:.12e}; gradvel rel L2 {e:.3e}")
    assert np.isfinite(gg).all()
    assert mg == pytest.approx(mo, rel=1e-10)
    assert e <= 1e-7
