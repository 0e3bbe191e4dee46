"""Tangents in several batches of directions, each with its own directions on the
device: a direction gives the same column, bit for bit, at the same place of
every batch (same records, slices and order of the sums)."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.refine import scattering_table

pytestmark = pytest.mark.gpu


def test_directions_in_batches():
    n, per = 400_000, 60           # 60 directions a batch: 5 weights x 46 slices x 33^3 points x 8 bytes in 4 GB
    assert int(4.0e9 / (5 * 46 * 8 * 33 ** 3)) == per
    rng = np.random.default_rng(1)
    pos, types = rng.random((n, 3)), np.ones(n, np.int32)
    occ, bdw = rng.uniform(0.7, 1.0, n), rng.uniform(0.3, 1.5, n)
    eck, vi, inc = FR.grid_block((-2.0,) * 3, (2.0,) * 3, (33, 33, 33))
    cf = scattering_table(X.random_form_factors(rng, 1))
    few = rng.normal(0.0, 1.0, (5, n, 5))
    dirs = np.empty((3 * per, n, 5))
    for k in range(3 * per):
        dirs[k] = few[k % 5]       # per is a multiple of 5
    F = rng.standard_normal(33 ** 3) + 1j * rng.standard_normal(33 ** 3)
    with _lib.Context(precision="fp16x3") as ctx:
        ctx.set_slice_atoms(8704)
        d, keep = ctx.model_desc(pos, types, occ, bdw, cf, eck, vi, inc, np.eye(3) / 25.0)
        di = ctx.model_jvp(d, F, dirs)
    assert np.array_equal(di[:, :per], di[:, per:2 * per]) and np.array_equal(di[:, :per], di[:, 2 * per:])
    assert len({di[:, k].tobytes() for k in range(5)}) == 5
