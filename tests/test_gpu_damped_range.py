"""Forward sums with strong, negative and widely spread B, whose factor exp(-B s^2)
of a row or column leaves the range of FP16 operands (the models' and
populations' BF16X3 runs take FP16 products).  Relative error of F over all
pixels (l2, in s^2 shells so that the strongly damped ones count): hi and lo BF16
halves hold 17 bits of each of the two operands, so BF16X3 is held to 1.5e-5 =
2 x 2^-17; FP16X3, 22 bits, to 1e-6 on mirrored grids and 3e-6 on others."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.population import Population
from diffusecode_amd.refine import scattering_table
from oracle import oracle as O

pytestmark = pytest.mark.gpu
BS = [(0.7, 0.3), (8.0, 1.0), (20.0, 2.0), (60.0, 5.0), (-8.0, 0.5), (8.0, 7.5)]


@pytest.fixture(scope="module")
def ctx():
    c = _lib.Context()
    yield c
    c.close()


def model(b, spread, idle):
    cr = X.orthorhombic(ncell=(4, 4, 3), seed=4)
    occ, _ = X.refinement_parameters(cr, seed=5)
    bdw = b + spread * np.random.default_rng(2).uniform(-1.0, 1.0, cr.natoms)
    if idle:   # atoms that are not there do not set the range
        occ[::17], bdw[::17] = 0.0, 0.0
    return cr, occ, bdw


def grid(mirrored, shape=(65, 17, 9)):
    lo = (-6.0, -6.0, -6.0) if mirrored else (-5.4, -6.0, -6.3)
    return FR.grid_block(lo, (6.0, 6.0, 6.0), shape)


def shell_error(F, ref, eck, vi, inc, rten):
    e, v = np.asarray(eck, float).ravel()[:3], np.asarray(vi, float).reshape(3, 3)
    i = np.indices(inc).reshape(3, -1, order="F")
    h = e[:, None] + v.T @ i if np.allclose(v, np.diag(np.diag(v))) else None
    s2 = np.einsum("kp,kl,lp->p", h, rten, h) / 4.0
    out = 0.0
    for k in range(8):
        m = (s2 >= k / 8 * s2.max()) & (s2 <= (k + 1) / 8 * s2.max())
        out = max(out, np.linalg.norm(F[m] - ref[m]) / np.linalg.norm(ref[m]))
    return out


@pytest.mark.parametrize("prec,bar", [("bf16x3", 1.5e-5), ("fp16x3", 1e-6)])
@pytest.mark.parametrize("mirrored", [True, False])
@pytest.mark.parametrize("b,spread", BS)
def test_model_forward(ctx, prec, bar, mirrored, b, spread):
    if prec == "fp16x3" and not mirrored:
        bar = 3e-6   # general tiles: complex products, each of four roundings
    for idle in (False, True):
        cr, occ, bdw = model(b, spread, idle)
        cf = scattering_table(cr.scat)
        eck, vi, inc = grid(mirrored)
        ref = O.model_f(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten()).ravel(order="F")
        d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
        ctx.set_precision(prec)
        try:
            F = ctx.model_intensity(d)[1].ravel(order="F")
        finally:
            ctx.set_precision("fp32")
        assert shell_error(F, ref, eck, vi, inc, cr.rten()) <= bar, idle


@pytest.mark.parametrize("mirrored", [True, False])
def test_population_forward(ctx, mirrored):
    """Members of very different B in one launch."""
    members, refs = [], []
    eck, vi, inc = grid(mirrored, (65, 33, 1))
    for b, spread in BS:
        cr, occ, bdw = model(b, spread, False)
        cf = scattering_table(cr.scat)
        members.append({"pos": cr.pos, "types": cr.iscat, "occ": occ, "bdw": bdw, "cfact": cf, "rten": cr.rten()})
        F = O.model_f(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
        refs.append(np.abs(F.ravel(order="F")) ** 2)
    refs = np.asfortranarray(np.stack(refs, axis=1))
    ctx.set_precision("bf16x3")
    try:
        pop = Population(members, eck, vi, inc, ctx=ctx)
        _, I, _ = pop.score(np.zeros_like(refs), want_icalc=True, want_grad=False)
    finally:
        ctx.set_precision("fp32")
    for k, m in enumerate(members):
        assert shell_error(I[:, k], refs[:, k], eck, vi, inc, m["rten"]) <= 3e-5, BS[k]
