"""Slice planes of a run without lots: they are all held at once, so where slices of
the usual length would take more than the plane budget (6 GB) the plan takes
longer ones.  4,000,000 atoms of three types on 161^3 points: 17 MB a plane."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR

pytestmark = pytest.mark.gpu


def test_planes_of_a_large_run():
    rng = np.random.default_rng(1)
    pos, _ = X.supercell(X.FCC_SITES, np.zeros(4, np.int32), (100,) * 3)
    types = rng.integers(1, 4, pos.shape[0]).astype(np.int32)
    c = X.Crystal(pos, types, (100,) * 3, 4, (4.0, 4.0, 4.0, 90.0, 90.0, 90.0), X.random_form_factors(rng, 3), np.ones(3), np.zeros(3))
    eck, vi, inc = FR.grid_block((-4.0,) * 3, (4.0,) * 3, (161,) * 3)
    with _lib.Context(precision="fp16x3") as ctx:
        ctx.crystal_set(c)
        desc, keep = ctx.run_desc(eck, vi, inc, c.rten(), FR.formtab(c))
        out = ctx.four_run(desc, want_var=False)
        slices = ctx.stats()["slices"]
    plane = 8 * 81 * 161 * 161
    assert slices * plane <= 6.0e9 + 3 * plane
    # the undisturbed crystal's Bragg peak at the origin: every atom in phase
    f = FR.formtab(c)
    F0 = sum((types == t + 1).sum() * f[0, t] for t in range(3))
    assert abs(out["dsi"][80, 80, 80] - abs(F0) ** 2) <= 1e-5 * abs(F0) ** 2
