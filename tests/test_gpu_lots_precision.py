"""FP16X3 lots against FP64: amplitude of the last lot, intensity, average amplitude and cross-lot
variance (relative l2, mean over three crystals).  Bars: the errors of the general tiles
(dc_gemm.hip) on the same runs, which the mirrored-pair tiles must not exceed --
their FP32 accumulators run over a slice of atoms, so the length of the slices of
small lots sets the error."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from oracle import oracle as O

pytestmark = pytest.mark.gpu
BARS = {"csf": 1.67e-7, "dsi": 1.28e-7, "fmean": 6.1e-8, "dvar": 7.0e-7}


def disordered(seed, cells=20, a=5.64):
    rng = np.random.default_rng(seed)
    pos, base = X.supercell(X.ROCKSALT_SITES, X.ROCKSALT_TYPES, (cells,) * 3)
    types = np.where(base == 1, 1, 2).astype(np.int32)
    swap = rng.random(types.size) < 0.3
    types[swap] = rng.integers(1, 3, int(swap.sum()))
    types[rng.random(types.size) < 0.03] = 0
    pos = pos + rng.normal(0.0, 0.05 / a, size=pos.shape)
    return X.Crystal(pos, types, (cells,) * 3, 8, (a, a, a, 90.0, 90.0, 90.0), X.random_form_factors(rng, 2), np.ones(2),
                     np.zeros(2))


def test_lots_fp16x3():
    eck, vi, inc = FR.grid_block((-10.0, -10.0, 0.0), (10.0, 10.0, 10.0), (151, 87, 2))
    err = {k: [] for k in BARS}
    with _lib.Context(precision="fp16x3") as ctx:
        for seed in (1, 2, 3):
            c = disordered(seed)
            lbeg = np.random.default_rng(seed + 1).integers(1, 21, (24, 3)).astype(np.int32)
            cf = FR.formtab(c)
            ref = O.four_run(c, eck, vi, inc, cf, ilots=2, ls=(6, 6, 6), lbeg=lbeg, want_var=True)
            ctx.crystal_set(c)
            desc, keep = ctx.run_desc(eck, vi, inc, c.rten(), cf, ilots=2, ls=(6, 6, 6), lbeg=lbeg)
            out = ctx.four_run(desc, want_var=True)
            for k in err:
                err[k].append(np.linalg.norm(out[k] - ref[k]) / np.linalg.norm(ref[k]))
    for k, bar in BARS.items():
        assert np.mean(err[k]) <= bar, (k, err[k])
