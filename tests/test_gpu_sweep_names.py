"""Eikonal passes over two fields and over one are timed under names of their
own: the benchmark's bytes per launch differ by a factor of two."""
import importlib

import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


def test_passes_over_one_field_have_their_own_name(pkg):
    say("names of the eikonal passes")
    cfg = pkg.default_config(16, 16, 16, particle_capacity=1024, heat_enabled=0, mc_enabled=0)
    n = 512
    rng = np.random.default_rng(1)
    sim = pkg.Simulator(cfg)
    sim.set_particles(n, pos=rng.uniform(0.1, 0.2, (n, 3)).astype(np.float32), vel=np.zeros((n, 3), np.float32),
                      flag=np.where(np.arange(n) % 3, pkg.TYPEFLUID, pkg.TYPESOLID).astype(np.int8),
                      mass=np.ones(n, np.float32))
    sim.hash_sort()
    sim.set_kernel_timing(True)
    sim.levelset_update()  # both level sets: five passes outward, five inward
    sim.p2g()
    sim.extrapolate_bc()   # both phase distances: three
    sim.g2p()
    sim.advect()           # the solid distance: three
    t = sim.kernel_times()
    assert t["sweep"][0] == 13 and t["sweep_one"][0] == 3
    b = importlib.import_module("bench").KERNEL_BYTES
    assert b["sweep"][0] == 2 * b["sweep_one"][0]
