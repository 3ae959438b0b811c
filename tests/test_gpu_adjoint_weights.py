"""P2G adjoint beside faces whose weight is not a number.

A particle whose mass is NaN makes the weight sums of the faces around it NaN;
such faces, like faces without weight, pass no cotangent on: the particle's own
gradients are exactly zero and every other particle's are finite.
"""
import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("phase", ["TYPEFLUID", "TYPEAIR"])
def test_p2g_adjoint_nan_mass(pkg, phase):
    say("p2g_adjoint, a mass that is not a number", phase)
    dims = (13, 17, 23)
    cfg = pkg.default_config(*dims, particle_capacity=16384, adjoint_enabled=1, heat_enabled=0, gas_enabled=0,
                             mc_enabled=0)
    rng = np.random.default_rng(5)
    n = 12000
    pos = (rng.uniform(0.0, 1.0, (n, 3)) * np.array(dims) * float(cfg.dx)).astype(np.float32)
    flag = np.full(n, pkg.TYPEFLUID, np.int8)
    flag[rng.uniform(size=n) < 0.3] = pkg.TYPEAIR
    mass = np.ones(n, np.float32)
    mass[np.flatnonzero(flag == getattr(pkg, phase))[100]] = np.nan
    sim = pkg.Simulator(cfg)
    sim.set_particles(n, pos=pos, vel=rng.standard_normal((n, 3)).astype(np.float32), flag=flag, mass=mass)
    sim.hash_sort()
    nan = np.isnan(sim.get_particles()["mass"])
    assert nan.sum() == 1
    nx, ny, nz = dims
    shapes = [(nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)] * 2
    gv, gx = sim.p2g_adjoint([rng.standard_normal(s) for s in shapes])
    assert not gv[nan].any() and not gx[nan].any()
    assert np.isfinite(gv).all() and np.isfinite(gx).all()
    assert (np.abs(gv[~nan]).sum(1) > 0).mean() > 0.9
