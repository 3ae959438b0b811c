"""Neighbour searches at the edges of their splits: the level set's window
(row bits, rings) and the position correction (row ranges, words of 32
particles, lists), against the float oracle bit for bit, with the library's own
sort and with the same cell lists given by the caller.

Random particles, from less than one in three cells to 70 in some cells
(several words a row, full lists), a capacity of exactly the particles, rows
around the 64-cell words of the level set (62, 126 cells), and a correction
radius of half a cell, of nearly a cell and of a tenth.
"""
import numpy as np
import pytest

from helpers import say
from test_gpu_parity import bitexact, copy_fields, copy_particles

pytestmark = pytest.mark.gpu

DIMS = [(4, 4, 12), (5, 9, 7), (13, 17, 23), (6, 5, 62), (5, 4, 126)]


def _sims(pkg, dims, per_cell, **over):
    nx, ny, nz = dims
    rng = np.random.default_rng([nx, ny, nz, int(10 * per_cell)])
    n = max(1, int(nx * ny * nz * per_cell))
    cfg = pkg.default_config(nx, ny, nz, particle_capacity=n + (70 if per_cell > 1 else 0), heat_enabled=0,
                             gas_enabled=0, mc_enabled=0, **over)
    h = float(cfg.dx)
    u = rng.uniform(0.0, 1.0, (n, 3))
    pos = u * np.array(dims) * h
    if per_cell > 1:  # 70 particles in one cell, the last ones of the array in the last cell
        cell = np.array([nx // 2, ny // 2, nz // 2])
        pos = np.concatenate([pos, (cell + rng.uniform(0.0, 1.0, (70, 3))) * h])
        pos[-9:] = (np.array(dims) - rng.uniform(0.0, 1.0, (9, 3))) * h
    pos = pos.astype(np.float32)
    n = len(pos)
    flag = rng.choice([pkg.TYPEFLUID, pkg.TYPESOLID, pkg.TYPEAIR, pkg.TYPEAIRSOLO], n, p=[0.7, 0.1, 0.15, 0.05])
    if per_cell > 1:  # whole regions without air
        flag[(flag != pkg.TYPESOLID) & (pos[:, 2] < 0.6 * nz * h)] = pkg.TYPEFLUID
    own = pkg.Simulator(cfg)
    own.set_particles(n, pos=pos, flag=flag.astype(np.int8), mass=rng.uniform(0.5, 2.0, n).astype(np.float32),
                      vel=rng.standard_normal((n, 3)).astype(np.float32))
    own.hash_sort()
    given = pkg.Simulator(cfg)
    given.set_particles(n, **own.get_particles())
    for nm in ("CELL_START", "CELL_END"):
        given.set_field(nm, own.get_field(nm))
    return cfg, own, given


def _oracle(orc, cfg, sim):
    o = orc.Oracle(cfg)
    copy_particles(sim, o)
    copy_fields(sim, o, ["CELL_START", "CELL_END"])
    return o


@pytest.mark.parametrize("per_cell", [0.3, 8.0])
@pytest.mark.parametrize("dims", DIMS)
def test_levelset_window(pkg, orc, dims, per_cell):
    say("level set", dims, per_cell)
    cfg, own, given = _sims(pkg, dims, per_cell)
    o = _oracle(orc, cfg, own)
    o.levelset_update()
    for sim in (own, given):
        sim.levelset_update()
        for f in ("LSFLUID", "LSAIR", "LSMERGE"):
            bitexact(sim.get_field(f), o.get_field(f).astype(np.float32), f)
        bitexact(sim.get_field("MARK"), o.get_field("MARK"), "MARK")


@pytest.mark.parametrize("radius", [0.1, 0.5, 0.97])
@pytest.mark.parametrize("per_cell", [0.3, 8.0])
@pytest.mark.parametrize("dims", DIMS)
def test_correct_positions_edges(pkg, orc, dims, per_cell, radius):
    say("position correction", dims, per_cell, radius)
    cfg, own, given = _sims(pkg, dims, per_cell, correction_radius=radius, correction_spring=50.0)
    o = _oracle(orc, cfg, own)
    o.correct_positions()
    want = o.get_particles()["pos"].astype(np.float32)
    before = own.get_particles()["pos"]
    for sim in (own, given):
        sim.correct_positions()
        bitexact(sim.get_particles()["pos"], want, "pos")
    if per_cell > 1 and radius > 0.1:
        assert np.any(want != before)
