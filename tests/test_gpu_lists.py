"""Gathers and scatters over rows of cells against their forms for caller-given
cell lists.

With the library's own sort a row of cells along k is one range of particles,
which the air P2G, the P2G adjoint and the G2P adjoint read as such; cell lists
set by the caller take the same kernels cell by cell (the G2P adjoint: particle
by particle).  Both forms add the same terms: the air P2G in the same order
(equal bits), the adjoints in FP64 in another order.  A sum of at most
n = 4000 FP64 terms differs between two orders by at most n * 2^-53 times the
sum of the terms' magnitudes, so 1e-12 of the largest value bounds every
element; the cotangents of P2G divide by the weights' sum, whose relative
change is as small.
"""
import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu

FACE = ["WATER_UX", "WATER_UY", "WATER_UZ", "AIR_UX", "AIR_UY", "AIR_UZ"]


@pytest.mark.parametrize("dims", [(4, 4, 12), (5, 9, 7), (8, 16, 8), (13, 17, 23), (33, 31, 10)])
def test_row_ranges(pkg, dims):
    say("row ranges", dims)
    nx, ny, nz = dims
    cfg = pkg.default_config(nx, ny, nz, particle_capacity=nx * ny * nz * 6 + 64, adjoint_enabled=1, flip_alpha=0.95,
                             heat_enabled=0, gas_enabled=0, mc_enabled=0)
    rng = np.random.default_rng(nx * 1000 + ny * 10 + nz)
    n = nx * ny * nz * 6
    h = float(cfg.dx)
    # some particles on cell borders and some outside the domain (cell 0);
    # liquid, air and solids mixed, whole bricks without air
    pos = (rng.uniform(0.0, 1.0, (n, 3)) * np.array(dims) * h).astype(np.float32)
    pos[::17] = (np.round(pos[::17] / h) * h).astype(np.float32)
    pos[::101] -= np.float32(3 * h * nx)
    flag = np.where(rng.uniform(size=n) < 0.2, pkg.TYPESOLID, pkg.TYPEFLUID).astype(np.int8)
    air = (pos[:, 2] > 0.5 * nz * h) & (rng.uniform(size=n) < 0.5)
    flag[air] = pkg.TYPEAIR
    vel = rng.standard_normal((n, 3)).astype(np.float32)
    own = pkg.Simulator(cfg)
    own.set_particles(n, pos=pos, vel=vel, flag=flag, mass=rng.uniform(0.5, 2.0, n).astype(np.float32))
    own.hash_sort()
    p = own.get_particles()
    given = pkg.Simulator(cfg)
    given.set_particles(n, **p)
    for nm in ("CELL_START", "CELL_END"):
        given.set_field(nm, own.get_field(nm))
    gf = [rng.standard_normal(m) for m in own.face_sizes()]
    gv = rng.standard_normal((n, 3))
    out = []
    for sim in (own, given):
        sim.p2g()
        faces = [sim.get_field(f) for f in FACE]
        pv, px = sim.p2g_adjoint(gf)
        r = sim.g2p_adjoint(gv)
        out.append((faces, [pv, px, r["vel"], r["pos"]] + list(r["u"]) + list(r["u_old"])))
    for f, a, b in zip(FACE, out[0][0], out[1][0]):
        if f.startswith("AIR"):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), f
    assert np.any(out[0][0][3]) and np.any(out[0][0][0])
    for q, (a, b) in enumerate(zip(out[0][1], out[1][1])):
        err = np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)
        say("  adjoint output %d: %.2e" % (q, err))
        assert np.any(b) and err <= 1e-12


@pytest.mark.parametrize("odd", ["none", "nan velocity", "infinite mass", "off the grid"])
@pytest.mark.parametrize("dims", [(4, 4, 5), (12, 9, 30), (9, 21, 11)])
def test_air_window(pkg, dims, odd):
    """Air P2G leaves out the window's cells beyond the kernel's radius when
    every air particle is finite and on the grid (library's own sort), and
    visits them otherwise and for given lists: the same bits either way (a NaN
    or an infinity two cells off reaches the face as 0 times it), and the same
    adjoint for finite particles."""
    say("air window", dims, odd)
    nx, ny, nz = dims
    rng = np.random.default_rng(nx * 1000 + ny * 10 + nz)
    n = nx * ny * nz * 4
    cfg = pkg.default_config(nx, ny, nz, particle_capacity=n, adjoint_enabled=1, heat_enabled=0, gas_enabled=0,
                             mc_enabled=0)
    h = float(cfg.dx)
    pos = (rng.uniform(0.0, 1.0, (n, 3)) * np.array(dims) * h * 0.999999).astype(np.float32)
    flag = np.where(rng.uniform(size=n) < 0.4, pkg.TYPEAIR, pkg.TYPEFLUID).astype(np.int8)
    vel = rng.standard_normal((n, 3)).astype(np.float32)
    mass = rng.uniform(0.5, 2.0, n).astype(np.float32)
    a = np.flatnonzero(flag == pkg.TYPEAIR)[n // 5]
    if odd == "nan velocity":
        vel[a] = np.nan
    elif odd == "infinite mass":
        mass[a] = np.inf
    elif odd == "off the grid":
        pos[a, 0] = (nx + 0.3) * h
    own = pkg.Simulator(cfg)
    own.set_particles(n, pos=pos, vel=vel, flag=flag, mass=mass)
    own.hash_sort()
    given = pkg.Simulator(cfg)
    given.set_particles(n, **own.get_particles())
    for nm in ("CELL_START", "CELL_END"):
        given.set_field(nm, own.get_field(nm))
    gf = [rng.standard_normal(m) for m in own.face_sizes()]
    adj = []
    for sim in (own, given):
        sim.p2g()
        adj.append(sim.p2g_adjoint(gf))
    for f in FACE[3:]:
        u, v = own.get_field(f), given.get_field(f)
        assert np.array_equal(u, v, equal_nan=True), f
        assert np.isnan(u).any() == (odd in ("nan velocity", "infinite mass"))
    if odd in ("none", "off the grid"):
        for u, v in zip(*adj):
            assert np.max(np.abs(u - v)) <= 1e-12 * np.max(np.abs(v))


@pytest.mark.parametrize("per_cell", [0.4, 9.0])
@pytest.mark.parametrize("dims", [(4, 4, 5), (13, 17, 23), (8, 16, 8)])
def test_tile_gather(pkg, dims, per_cell):
    """G2P, the bubble-side correction and the heat transfer interpolate from
    tiles staged in LDS with the library's own sort, from memory with given
    lists: the same bits, for tiles with many and with few particles and for
    particles off the grid."""
    say("tile gather", dims, per_cell)
    nx, ny, nz = dims
    rng = np.random.default_rng([nx, ny, nz, int(10 * per_cell)])
    n = int(nx * ny * nz * per_cell)
    for alpha in (1.0, 0.95):
        cfg = pkg.default_config(nx, ny, nz, particle_capacity=n, flip_alpha=alpha, heat_enabled=1, gas_enabled=0,
                                 mc_enabled=0)
        h = float(cfg.dx)
        pos = (rng.uniform(0.0, 1.0, (n, 3)) * np.array(dims) * h).astype(np.float32)
        pos[::37] += np.float32(0.6 * nx * h)
        flag = rng.choice([pkg.TYPEFLUID, pkg.TYPESOLID, pkg.TYPEAIR, pkg.TYPEAIRSOLO], n, p=[0.6, 0.1, 0.25, 0.05])
        own = pkg.Simulator(cfg)
        own.set_particles(n, pos=pos, flag=flag.astype(np.int8), vel=rng.standard_normal((n, 3)).astype(np.float32),
                          mass=np.ones(n, np.float32), T=rng.uniform(250.0, 400.0, n).astype(np.float32))
        own.hash_sort()
        own.levelset_update()
        given = pkg.Simulator(cfg)
        given.set_particles(n, **own.get_particles())
        for nm in ("CELL_START", "CELL_END"):
            given.set_field(nm, own.get_field(nm))
        given.levelset_update()
        fields = [f + s for f in FACE for s in ("", "_OLD")]
        values = {f: rng.standard_normal(own.get_field(f).shape).astype(np.float32) for f in fields}
        before = own.get_particles()
        for sim in (own, given):
            for f, v in values.items():
                sim.set_field(f, v)
            sim.g2p()
            sim.heat()
            sim.correct_bubble_positions()
        a, b = own.get_particles(), given.get_particles()
        for f in ("vel", "T", "lheat", "pos"):
            assert np.array_equal(a[f].view(np.uint32), b[f].view(np.uint32)), f
        assert np.any(a["vel"] != before["vel"]) and np.any(a["T"] != before["T"])
