"""The projection's resident solve (the vectors in registers, one launch per
solve) over the shapes it accepts, and the launch-per-iteration kernels on the
shapes it does not (a row along k longer than a block has threads), against
the FP64 oracle.

The grids cover one to eight cells per thread, tiles clipped along i and j,
blocks with spare threads, rows of more than a wave and of almost a whole
block, and k sizes that are no multiple of anything; with an air ball (slow
rows, also in the ring between blocks) or with a solid block.

Tolerances: the FP64 and mixed forms are solved to 1e-10 on the FP64
residual; with condition numbers below 1e5 on these grids that leaves less
than 1e-5 in the pressure.  The FP32 form is solved to 1e-6 and held to 1e-3
(pressure) and 1e-4 (faces), as elsewhere in these tests.
"""
import threading

import numpy as np
import pytest

from helpers import rel_l2, say

pytestmark = pytest.mark.gpu

FACE = ["WATER_UX", "WATER_UY", "WATER_UZ", "AIR_UX", "AIR_UY", "AIR_UZ"]


def _system(pkg, dims, precision, with_air, seed=5):
    nx, ny, nz = dims
    rng = np.random.default_rng([seed, nx, ny, nz])
    I, J, K = np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij")
    inner = (I >= 1) & (I <= nx - 2) & (J >= 1) & (J <= ny - 2) & (K >= 1) & (K <= nz - 2)
    liquid = inner & (K < 0.75 * nz + 0.8 * np.sin(0.7 * I) * np.cos(0.5 * J))
    cfg = pkg.default_config(nx, ny, nz, precision=precision, rho_liquid=1000.0, rho_air=1.0,
                             tol=1e-6 if precision == pkg.FP32 else 1e-10, max_iters=20000,
                             solid_constraint=0 if with_air else 1, heat_enabled=0, gas_enabled=0, mc_enabled=0,
                             particle_capacity=64)
    h = cfg.dx
    mark = np.full(dims, pkg.TYPEVACUUM, np.int8)
    mark[liquid] = pkg.TYPEFLUID
    ls = np.where(liquid, -1.0, 0.5) * h
    if with_air:
        r = max(1.2, min(nx, ny, nz) / 4.5)
        c = (0.5 * nx, 0.45 * ny, max(r + 1.5, 0.35 * nz))
        phi = r - np.sqrt((I + 0.5 - c[0]) ** 2 + (J + 0.5 - c[1]) ** 2 + (K + 0.5 - c[2]) ** 2)
        mark[liquid & (phi > 0)] = pkg.TYPEAIR
        ls = np.where(liquid, np.clip(phi, -2.5, 2.5) * h, ls)
    else:
        mark[liquid & (I < nx // 2) & (I > nx // 4) & (J < ny // 2) & (K > nz // 4) & (K < nz // 2)] = pkg.TYPESOLID
    edge = ~((I > 0) & (I < nx - 1) & (J > 0) & (J < ny - 1) & (K > 0) & (K < nz - 1))
    mark[edge] = pkg.TYPEBOUNDARY
    ls[edge] = -0.5 * h
    shapes = [(nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1)] * 2
    fields = {"MARK": mark, "LSMERGE": ls.astype(np.float32)}
    for name, s in zip(FACE, shapes):
        fields[name] = (0.3 * rng.standard_normal(s)).astype(np.float32)
    return cfg, fields


def _project(sim, fields):
    for f, v in fields.items():
        sim.set_field(f, v)
    return sim.project()


SMALL = [(4, 4, 12), (5, 70, 33), (20, 20, 20), (37, 21, 64), (16, 16, 300), (33, 40, 66), (9, 11, 1024), (8, 9, 1030)]
LARGE = [(64, 80, 96), (96, 90, 100), (121, 99, 110), (128, 128, 128)]


@pytest.mark.parametrize("with_air", [False, True])
@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("dims", SMALL + LARGE)
def test_projection_shapes(pkg, orc, dims, precision, with_air):
    say("projection", dims, "precision", precision, "air" if with_air else "solid")
    if dims in LARGE and with_air != (precision == 1):
        pytest.skip("one scene per precision on the large grids")
    cfg, fields = _system(pkg, dims, precision, with_air)
    sim = pkg.Simulator(cfg)
    gi = _project(sim, fields)
    say("  gpu", gi)
    assert gi["converged"] == 1
    tight = pkg.Config.from_buffer_copy(cfg)
    tight.tol = 1e-12
    o64 = orc.Oracle(tight, use_double=True)
    for f, v in fields.items():
        o64.set_field(f, v)
    say("  fp64 oracle", o64.project())
    if precision != pkg.FP32:
        assert gi["rel_residual"] <= 1e-9
    for f in ["PRESSURE"] + FACE:
        e = rel_l2(sim.get_field(f), o64.get_field(f))
        say("  %s rel L2 vs FP64 = %.2e" % (f, e))
        if precision != pkg.FP32:
            assert e <= 1e-5, f
        else:
            assert e <= (1e-3 if f == "PRESSURE" else 1e-4), f


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_same_bits_again_and_side_by_side(pkg, precision):
    """A solve gives the same bits every time (also right after a solve of
    another system in the same context), and when two contexts on two threads
    solve at once."""
    say("repeated and concurrent solves, precision", precision)
    dims = (40, 44, 52)
    cfg, a = _system(pkg, dims, precision, True)
    _, b = _system(pkg, dims, precision, True, seed=6)
    sims = [pkg.Simulator(cfg), pkg.Simulator(cfg)]
    want = []
    for fields in (a, b):
        _project(sims[0], fields)
        want.append([sims[0].get_field(f) for f in ["PRESSURE"] + FACE])
    got = [[], []]

    def work(q, fields):
        for _ in range(6):
            _project(sims[q], fields)
            got[q].append([sims[q].get_field(f) for f in ["PRESSURE"] + FACE])

    threads = [threading.Thread(target=work, args=(q, f)) for q, f in enumerate((a, b))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for q in range(2):
        assert len(got[q]) == 6
        for rep in got[q]:
            for u, v in zip(rep, want[q]):
                assert np.array_equal(u, v)


def test_zero_right_hand_side_and_nonfinite(pkg):
    """No divergence: converged at once with zero pressure; a NaN velocity: reported as non-finite."""
    for precision in (0, 1, 2):
        say("zero and non-finite systems, precision", precision)
        cfg, fields = _system(pkg, (20, 22, 24), precision, False)
        for f in FACE:
            fields[f][...] = 0.0
        sim = pkg.Simulator(cfg)
        info = _project(sim, fields)
        assert info["converged"] == 1 and info["iterations"] == 0
        assert not sim.get_field("PRESSURE").any()
        fields["WATER_UX"][10, 5, 5] = np.nan
        with pytest.raises(pkg.MpfError) as e:
            _project(sim, fields)
        assert e.value.status == pkg.NONFINITE
