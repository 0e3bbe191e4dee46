"""Reverse pass (dc_adjoint.hip) over many column tiles a work-group: the values
of the next tile's columns are stored while other waves still contract the one
before, the column phases are carried from tile to tile between exact ones,
and runs of the ordinate as short as a tile end inside it.  Shapes: one k-step
of rows a tile (33 mirrored points or fewer, 16 unmirrored ones) and several,
a centre row, ordinate runs of 16, 17 and 48 points over many layers, row
chunks; every work-group has four waves of atoms.  Against the oracle's direct
FP64 gradient, at the bar of the single-tile shapes (2e-5 of the largest
gradient per parameter kind), and bit for bit from call to call: the partial
sets and their order are fixed, so a difference is a wave reading what it
should not."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.refine import scattering_table
from oracle import oracle as O

pytestmark = pytest.mark.gpu
BAR = 2e-5


@pytest.fixture(scope="module")
def ctx():
    c = _lib.Context()
    yield c
    c.close()


@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
@pytest.mark.parametrize("shape,mirrored", [
    ((2, 16, 40), True), ((17, 48, 14), True), ((31, 17, 30), True), ((32, 16, 33), True), ((33, 16, 40), True),
    ((33, 17, 30), True), ((16, 17, 30), False), ((33, 16, 20), False), ((65, 16, 20), True), ((129, 17, 9), True),
    ((323, 16, 4), True)])
def test_many_tiles_a_range(ctx, prec, shape, mirrored):
    cr = X.orthorhombic(ncell=(6, 5, 4), seed=4)
    occ, bdw = X.refinement_parameters(cr, seed=5)
    cf = scattering_table(cr.scat)
    lo = [-0.04 * (n - 1) if mirrored else -0.031 * n for n in shape]
    eck, vi, inc = FR.grid_block(lo, [l + 0.08 * (n - 1) for l, n in zip(lo, shape)], shape)
    print(f"case adjoint walk {prec} mirrored={mirrored} {shape}", flush=True)
    F = O.model_f(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
    gi = np.random.default_rng(3).standard_normal(F.size)
    ref = O.model_grad(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten(), F, gi)
    d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
    ctx.set_precision(prec)
    try:
        for walk in (1, 32, 0):
            ctx.set_adjoint_walk(walk)
            g = ctx.model_vjp(d, F, gi)
            err = [np.abs(g[:, k] - ref[:, k]).max() / np.abs(ref[:, k]).max() for k in range(5)]
            assert max(err) <= BAR, (walk, err)
            for _ in range(4):
                assert np.array_equal(ctx.model_vjp(d, F, gi), g), walk
    finally:
        ctx.set_adjoint_walk(0)
        ctx.set_precision("fp32")
