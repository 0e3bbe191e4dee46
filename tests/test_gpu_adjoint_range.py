"""Reverse pass of the split precisions (dc_adjoint.hip) where exp(-B s^2) and the
residuals leave the range of its FP16 operands: strong, negative and widely
spread B, on all pixels, on the outer half of s^2 and on the outer rows alone,
and residuals up to the end of FP32.  Gradients weighted to 1 / |F|, so that
the strongly damped pixels count.  l2 error of each parameter kind, in each third
of the atoms by B, against the oracle's FP64 gradient: operands of two 16-bit
parts hold 17 bits or more, 2 x 2^-17 = 1.5e-5 for the two of a product."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.refine import scattering_table
from oracle import oracle as O

pytestmark = pytest.mark.gpu
BAR = 1.5e-5
SHAPE = (65, 17, 9)


@pytest.fixture(scope="module")
def ctx():
    c = _lib.Context()
    yield c
    c.close()


@pytest.mark.parametrize("prec", ["bf16x3", "fp16x2"])
@pytest.mark.parametrize("mirrored", [True, False])
@pytest.mark.parametrize("b,spread", [(0.7, 0.3), (8.0, 1.0), (20.0, 2.0), (40.0, 4.0), (-8.0, 0.5), (8.0, 7.5)])
def test_damped_gradient(ctx, prec, mirrored, b, spread):
    cr = X.orthorhombic(ncell=(4, 4, 3), seed=4)
    occ, _ = X.refinement_parameters(cr, seed=5)
    bdw = b + spread * np.random.default_rng(2).uniform(-1.0, 1.0, cr.natoms)
    cf = scattering_table(cr.scat)
    lo = (-6.0, -6.0, -6.0) if mirrored else (-5.4, -6.0, -6.3)
    eck, vi, inc = FR.grid_block(lo, (6.0, 6.0, 6.0), SHAPE)
    F = O.model_f(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
    h = [np.linspace(l, 6.0, n) for l, n in zip(lo, SHAPE)]
    s2 = sum(np.meshgrid(*[cr.rten()[k, k] * h[k] ** 2 / 4.0 for k in range(3)], indexing="ij")).ravel(order="F")
    row = np.broadcast_to((h[0] ** 2)[:, None, None], SHAPE).ravel(order="F")
    g0 = np.random.default_rng(3).standard_normal(F.size) / np.abs(F.ravel(order="F"))
    d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
    thirds = np.array_split(np.argsort(bdw), 3)
    ctx.set_precision(prec)
    try:
        for name, mask in (("all", s2 >= 0.0), ("outer half", s2 > 0.5 * s2.max()), ("outer rows", row > 25.0)):
            gi = np.where(mask, g0, 0.0)
            ref = O.model_grad(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten(), F, gi)
            g = ctx.model_vjp(d, F, gi)
            err = max(np.linalg.norm(g[t, k] - ref[t, k]) / np.linalg.norm(ref[t, k]) for t in thirds for k in range(5))
            assert err <= BAR, name
    finally:
        ctx.set_precision("fp32")


@pytest.mark.parametrize("scale", [1e-34, 1e30])
def test_residuals_to_the_end_of_fp32(ctx, scale):
    """The gradient stays linear in G until the FP32 Q planes end."""
    cr = X.orthorhombic(ncell=(2, 2, 2), seed=4)
    occ, bdw = X.refinement_parameters(cr, seed=5)
    eck, vi, inc = FR.grid_block((-1.0, -1.0, -1.0), (1.0, 1.0, 1.0), (65, 9, 5))
    d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, bdw, scattering_table(cr.scat), eck, vi, inc, cr.rten())
    gi = np.random.default_rng(3).standard_normal(65 * 45)
    ctx.set_precision("bf16x3")
    try:
        F = ctx.model_intensity(d)[1]
        one, big = ctx.model_vjp(d, F, gi), ctx.model_vjp(d, F, gi * scale)
    finally:
        ctx.set_precision("fp32")
    for k in range(5):
        assert np.abs(big[:, k] / scale - one[:, k]).max() <= 2e-6 * np.abs(one[:, k]).max()
