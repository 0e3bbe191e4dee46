"""Every forced GEMM tile (dc_set_gemm_tile) in every precision: a population
runs, with the tile where its scheme has it and with the planned one where it has
not, as single runs do.  Against the oracle at the population bars: chi^2 1e-4,
I 1e-6 of its largest value in FP32 and 1e-5 in the 3-product splits; FP16X2, one
side rounded to FP16 halves and the other to a single one, 2e-3."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.population import Population
from oracle import oracle as O

pytestmark = pytest.mark.gpu
NTILES = len(_lib.Context.gemm_tiles())


@pytest.fixture(scope="module")
def scored():
    crs = X.population(nmembers=3, nmin=300, nmax=1200, seed=5)
    eck, vi, inc = FR.grid_block((-3.0, -3.0, 0.0), (3.0, 3.0, 0.0), (35, 18, 1))
    pop = Population.from_crystals(crs, eck, vi, inc, precision="fp32")
    I = np.stack([np.abs(O.model_f(m["pos"], m["types"], m["occ"], m["bdw"], m["cfact"], eck, vi, inc, m["rten"])).ravel(order="F") ** 2
                  for m in pop.members], axis=1)
    T = I * np.random.default_rng(3).uniform(0.5, 1.5, I.shape)
    yield pop, np.asfortranarray(T), I
    pop.ctx.close()


@pytest.mark.parametrize("prec,bar", [("fp32", 1e-6), ("bf16x3", 1e-5), ("fp16x2", 2e-3), ("fp16x3", 1e-5)])
@pytest.mark.parametrize("tile", range(NTILES))
def test_forced_tile(scored, tile, prec, bar):
    pop, T, I = scored
    print(f"case batch tile {tile} {prec}", flush=True)
    pop.ctx.set_precision(prec)
    pop.ctx.check(_lib.lib().dc_set_gemm_tile(pop.ctx.h, tile))
    try:
        chi, ic, _ = pop.score(T, want_icalc=True, want_grad=False)
    finally:
        pop.ctx.check(_lib.lib().dc_set_gemm_tile(pop.ctx.h, -1))
        pop.ctx.set_precision("fp32")
    assert (np.abs(ic - I).max(axis=0) <= bar * I.max(axis=0)).all()
    ref = ((I - T) ** 2).sum(axis=0)
    assert (np.abs(chi - ref) <= max(1e-4, 10 * bar) * ref).all()
