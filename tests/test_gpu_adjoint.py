"""Reverse pass (dc_adjoint.hip) at the sizes where its layout changes, against
the oracle's direct FP64 gradient: row counts on both sides of a k-step of 16
pairs (a centre row taken apart, an even count, a single row, several row
chunks), grids whose rows are not mirrored about their centre (each row its
own pair), ordinate runs shorter than a column tile, a last tile of one
column, residuals of extreme size, and a population whose operand words are made
in more than one run of planes.  Bar: 2e-5 of the largest gradient per
parameter kind, the FP32 adjoint's own, in every precision."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.population import Population
from diffusecode_amd.refine import scattering_table
from oracle import oracle as O

pytestmark = pytest.mark.gpu
BAR = 2e-5


@pytest.fixture(scope="module")
def ctx():
    c = _lib.Context()
    yield c
    c.close()


def errors(g, ref):
    return [np.abs(g[:, k] - ref[:, k]).max() / max(np.abs(ref[:, k]).max(), 1e-300) for k in range(5)]


SHAPES = [(1, 5, 1), (2, 17, 3), (31, 4, 5), (32, 16, 2), (33, 33, 1), (65, 7, 3), (66, 1, 1),
          (97, 17, 1), (100, 3, 2), (163, 20, 1), (200, 2, 2), (323, 1, 1)]


@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
@pytest.mark.parametrize("mirrored", [True, False])
@pytest.mark.parametrize("shape", SHAPES)
def test_rows_and_columns(ctx, prec, mirrored, shape):
    cr = X.orthorhombic(ncell=(3, 3, 2), seed=4)
    occ, bdw = X.refinement_parameters(cr, seed=5)
    cf = scattering_table(cr.scat)
    lo = [-0.04 * (n - 1) if mirrored else -0.031 * n for n in shape]
    eck, vi, inc = FR.grid_block(lo, [l + 0.08 * (n - 1) for l, n in zip(lo, shape)], shape)
    print(f"case adjoint {prec} mirrored={mirrored} {shape}", flush=True)
    F = O.model_f(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
    gi = np.random.default_rng(3).standard_normal(F.size)
    ref = O.model_grad(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten(), F, gi)
    ctx.set_precision(prec)
    try:
        for b in (bdw, None) if not mirrored else (bdw,):
            if b is None:   # without B every grid's rows pair up
                F = O.model_f(cr.pos, cr.iscat, occ, None, cf, eck, vi, inc, cr.rten())
                ref = O.model_grad(cr.pos, cr.iscat, occ, np.zeros_like(occ), cf, eck, vi, inc, cr.rten(), F, gi)
            d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, b, cf, eck, vi, inc, cr.rten())
            g = ctx.model_vjp(d, F, gi)
            assert max(errors(g, ref)) <= BAR, b is None
    finally:
        ctx.set_precision("fp32")


@pytest.mark.parametrize("prec", ["fp32", "fp16x3"])
@pytest.mark.parametrize("scale", [1e-25, 1e25])
def test_extreme_residuals(ctx, prec, scale):
    """The gradient is linear in G over the range of FP32 Q planes."""
    cr = X.orthorhombic(ncell=(2, 2, 2), seed=4)
    occ, bdw = X.refinement_parameters(cr, seed=5)
    eck, vi, inc = FR.grid_block((-1.0, -1.0, -1.0), (1.0, 1.0, 1.0), (33, 9, 5))
    d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, bdw, scattering_table(cr.scat), eck, vi, inc, cr.rten())
    gi = np.random.default_rng(3).standard_normal(33 * 45)
    ctx.set_precision(prec)
    try:
        F = ctx.model_intensity(d)[1]
        one, big = ctx.model_vjp(d, F, gi), ctx.model_vjp(d, F, gi * scale)
    finally:
        ctx.set_precision("fp32")
    assert max(errors(big / scale, one)) <= 2e-6


def test_population_of_several_word_runs(ctx):
    """48 members of 8 atoms on 512^2 points: 1.2 GB or more of operand words,
    made in runs of 1 GiB; members of the first and last run against populations
    of their own."""
    crs = [X.orthorhombic(ncell=(1, 1, 1), seed=k) for k in range(48)]
    eck, vi, inc = FR.grid_block((-3.0, -3.0, 0.0), (3.0, 3.0, 0.0), (512, 512, 1))
    pop = Population.from_crystals(crs, eck, vi, inc, ctx=ctx, precision="fp32")
    nscat = pop.cfact.shape[1]
    assert 48 * nscat * 512 * 512 * 36 > 1.2 * 2**30
    T = np.asfortranarray(np.random.default_rng(1).uniform(1, 100, (pop.npixels, 48)))
    chi, _, g = pop.score(T)
    for m in (0, 47):
        one = Population.from_crystals(crs[m:m + 1], eck, vi, inc, seed=m, ctx=ctx, precision="fp32")
        chi1, _, g1 = one.score(np.asfortranarray(T[:, m:m + 1]))
        sl = slice(pop.atom_beg[m], pop.atom_beg[m + 1])
        assert max(errors(g[sl], g1)) <= 1e-5
