"""The cell sort at the sizes where its launches change: 2.5M particles (one or
four waves' worth per wave; the last wave partly filled) and 4096 x 4096 cells
(above them a launch scans the block sums), with and without a context, against
a stable sort of the keys on the host: every integer equal.
"""
import numpy as np
import pytest

from helpers import say
from test_zz_no_alloc import _noalloc, _reference

pytestmark = pytest.mark.gpu

MANY = 2500000


@pytest.mark.parametrize("context", [True, False])
@pytest.mark.parametrize("dims,n", [((40, 41, 42), MANY - 1), ((40, 41, 42), MANY), ((90, 91, 50), MANY + 1027),
                                    ((260, 256, 257), 70001)])
def test_sort_sizes(pkg, dims, n, context):
    say("sort sizes", dims, n, "context" if context else "no context")
    nx, ny, nz = dims
    rng = np.random.default_rng([n, nx])
    cfg = pkg.default_config(nx, ny, nz, particle_capacity=n, mc_enabled=0, heat_enabled=0, gas_enabled=0)
    h = np.float32(cfg.dx)
    cell = rng.integers(0, dims, (n, 3))
    pos = ((cell + 0.5) * h).astype(np.float32)  # centres: the key does not depend on rounding
    key = ((cell[:, 0] * ny + cell[:, 1]) * nz + cell[:, 2]).astype(np.uint32)
    got = _reference(pkg, cfg, pos) if context else _noalloc(pkg, cfg, pos)
    order = np.argsort(key, kind="stable").astype(np.uint32)
    assert np.array_equal(got["GRID_INDEX"], order)
    assert np.array_equal(got["GRID_HASH"], key[order])
    count = np.bincount(key, minlength=nx * ny * nz)
    end = np.cumsum(count)
    undef = np.uint32(pkg.CELL_UNDEF)
    assert np.array_equal(got["CELL_START"].ravel(), np.where(count > 0, end - count, undef).astype(np.uint32))
    assert np.array_equal(got["CELL_END"].ravel(), np.where(count > 0, end, undef).astype(np.uint32))
