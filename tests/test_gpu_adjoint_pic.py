"""G2P adjoint of a pure PIC step (flip_alpha = 0): the old velocities do not
enter the step, so their cotangents are exactly zero, also where the cotangent
of a velocity is infinite or not a number.  With FLIP it reaches them."""
import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("given_lists", [False, True])
@pytest.mark.parametrize("alpha", [0.0, 0.95])
def test_old_velocity_cotangents(pkg, alpha, given_lists):
    say("g2p_adjoint, alpha", alpha, "given lists" if given_lists else "own sort")
    dims = (9, 13, 10)
    cfg = pkg.default_config(*dims, particle_capacity=8192, adjoint_enabled=1, flip_alpha=alpha, heat_enabled=0,
                             gas_enabled=0, mc_enabled=0)
    rng = np.random.default_rng(3)
    n = 6000
    pos = (rng.uniform(0.05, 0.95, (n, 3)) * np.array(dims) * float(cfg.dx)).astype(np.float32)
    flag = np.where(rng.uniform(size=n) < 0.3, pkg.TYPEAIR, pkg.TYPEFLUID).astype(np.int8)
    sim = pkg.Simulator(cfg)
    sim.set_particles(n, pos=pos, vel=rng.standard_normal((n, 3)).astype(np.float32), flag=flag,
                      mass=np.ones(n, np.float32))
    sim.hash_sort()
    if given_lists:
        for nm in ("CELL_START", "CELL_END"):
            sim.set_field(nm, sim.get_field(nm))
    g = rng.standard_normal((n, 3))
    g[100] = np.inf
    g[2000, 1] = np.nan
    r = sim.g2p_adjoint(g)
    assert any(not np.isfinite(u).all() for u in r["u"])
    for u, old in zip(r["u"], r["u_old"]):
        if alpha == 0.0:
            assert not old.any()
        else:
            assert np.array_equal(np.isfinite(u), np.isfinite(old))
