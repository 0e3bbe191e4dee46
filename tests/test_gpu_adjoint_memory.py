"""Reverse pass of many atoms on a long line: the partial sets of its row chunks stay
within their bound, and the gradients are those of the atoms one by one.  The
gradient of an atom for a given F and dL/dI does not depend on the others, so a few
atoms alone, whose row chunks all have sets of their own, are the reference."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.refine import scattering_table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
def test_row_chunks_in_several_launches(prec):
    import torch
    n, few = 2_500_000, np.arange(0, 2_500_000, 2_311)
    rng = np.random.default_rng(1)
    pos, types = rng.random((n, 3)), np.ones(n, np.int32)
    occ, bdw = rng.uniform(0.7, 1.0, n), rng.uniform(0.3, 1.5, n)
    eck, vi, inc = FR.grid_block((-4.0, 0.25, 0.5), (4.0, 0.25, 0.5), (4001, 1, 1))
    cf = scattering_table(X.random_form_factors(rng, 1))
    rten = np.eye(3) / 25.0
    F = rng.standard_normal(4001) + 1j * rng.standard_normal(4001)
    gi = rng.standard_normal(4001)
    with _lib.Context(precision=prec) as ctx:
        d, keep = ctx.model_desc(pos[few], types[few], occ[few], bdw[few], cf, eck, vi, inc, rten)
        ref = ctx.model_vjp(d, F, gi)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        d, keep = ctx.model_desc(pos, types, occ, bdw, cf, eck, vi, inc, rten)
        g = ctx.model_vjp(d, F, gi)[few]
        used = free - torch.cuda.mem_get_info()[0]
    for k in range(5):
        assert np.abs(g[:, k] - ref[:, k]).max() <= 2e-6 * np.abs(ref[:, k]).max()
    # partial sets 2 GiB, atoms (records 48, positions and parameters 40, index 4, gradient 40 bytes) 0.33 GB
    assert used <= 2.8e9
