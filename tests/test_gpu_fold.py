"""Mirrored-pair tiles of the phase GEMM (dc_fold.h): every tile in the
precisions they are built for, on grids that fold the columns or the rows, odd and even point
counts, wrapping flattened axes, remainders of rows and pairs, against the
exact FP64 sum; and with per-atom B, where a side whose s^2 is not mirrored
about its centre must take the general tiles."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.refine import scattering_table
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# the bars of the direct sums
BAR = {"fp32": 1e-6, "bf16x3": 1e-5, "fp16x3": 1e-5}
TILE0 = 9


@pytest.fixture(scope="module")
def ctx():
    c = _lib.Context()
    yield c
    c.close()


def fold_tiles():
    return range(TILE0, TILE0 + 14)


@pytest.mark.parametrize("prec", ["fp32", "bf16x3", "fp16x3"])
@pytest.mark.parametrize("tile", fold_tiles())
def test_fold_tiles(ctx, prec, tile):
    """Shapes: one more and one fewer than a tile's pairs and rows, both
    parities on each side, wraps at 17 and 129 points, a single column."""
    assert tile < len(ctx.gemm_tiles())
    c = X.rocksalt(n=3, seed=5)
    pos = c.pos[c.iscat > 0]
    pairs = ctx.gemm_tiles()[tile][1]
    try:
        ctx.set_precision(prec)
        ctx.set_gemm_tile(tile)
        # a tile that FP32 is not built for falls back to the planned one
        for shape in ((129, pairs + 1, 1), (pairs - 1, 17, 9), (17, 18, pairs), (200, 1, 1), (6, 2, 2), (1, 1, 1)):
            print(f"case fold tile={tile} prec={prec} shape={shape}", flush=True)
            lo = [-0.05 * n + 0.013 for n in shape]
            eck, vi, num = FR.grid_block(lo, [l + (n - 1) * 0.1 for l, n in zip(lo, shape)], shape)
            st, lmn, off = O.fourier_lmn(eck, vi, num)
            corner = sum(int(m) * np.asarray(v) for m, v in
                         zip(lmn, [vi[:, 0], vi[:, 1], vi[:, 2], off[:, 0], off[:, 1], off[:, 2]]))
            F = ctx.strucf(pos, vi[:, 0], vi[:, 1], vi[:, 2], off, lmn, num)
            Fref = O.strucf_exact(pos, corner, vi[:, 0], vi[:, 1], vi[:, 2], num)
            # the bound of a sum of N unit terms; grids with a Bragg peak hold it on |F|^2 / max too
            assert float(np.abs(F - Fref).max()) <= BAR[prec] * len(pos)
    finally:
        ctx.set_gemm_tile(-1)
        ctx.set_precision("fp32")


@pytest.mark.parametrize("prec", ["fp32", "bf16x3", "fp16x3"])
@pytest.mark.parametrize("lo,n", [((-1.0, -1.2, -0.8), (21, 25, 17)), ((-1.0, 0.3, 0.1), (20, 15, 1)),
                                  ((0.2, -1.2, 0.0), (19, 24, 1)), ((0.2, 0.1, 0.3), (18, 17, 5))])
def test_fold_damped(ctx, prec, lo, n):
    """Per-atom B on grids centred on both, one or none of the foldable
    sides: F and I against the exact model."""
    print(f"case fold damped prec={prec} lo={lo} n={n}", flush=True)
    cr = X.orthorhombic(ncell=(4, 3, 4), seed=4)
    occ, bdw = X.refinement_parameters(cr, seed=5)
    cf = scattering_table(cr.scat)
    hi = [-l if l < 0 else l + 0.1 * (m - 1) for l, m in zip(lo, n)]
    eck, vi, inc = FR.grid_block(lo, hi, n)
    ctx.set_precision(prec)
    try:
        d, keep = ctx.model_desc(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten())
        icalc, fcalc = ctx.model_intensity(d)
    finally:
        ctx.set_precision("fp32")
    F = O.model_f(cr.pos, cr.iscat, occ, bdw, cf, eck, vi, inc, cr.rten()).reshape(icalc.shape, order="F")
    scale = sum(cf[0, t - 1].real * o for t, o in zip(cr.iscat, occ))      # sum of the terms at h = 0
    assert float(np.abs(fcalc - F).max()) <= BAR[prec] * scale
