"""The pressure solve by launches on grids whose k extent leaves a 128-cell
tile mostly empty: the kernels then take 64-cell tiles.

Grids with nz > 1024 (never solved in one launch).  (30, 9, 1060) takes narrow
tiles in every form with 512 blocks (mixed, FP64, slow rows), (44, 9, 1060) in
the FP32 form without slow rows (768 blocks).  The scene with air has slow
rows.  Same system, oracle and tolerances as the other grids of the solve
(tol 1e-10 in MIXED and FP64: 1e-5; 1e-6 in FP32: 1e-3 pressure, 1e-4 faces).
"""
import pytest

from helpers import rel_l2, say
from test_gpu_resident import FACE, _project, _system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("with_air", [False, True])
@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("dims", [(30, 9, 1060), (44, 9, 1060)])
def test_projection_narrow_tiles(pkg, orc, dims, precision, with_air):
    say("projection", dims, "precision", precision, "air" if with_air else "solid")
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
