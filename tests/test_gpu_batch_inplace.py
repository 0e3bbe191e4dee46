"""dc_batch_chi2_dev on arrays that overlap: an output that takes the place of
an input (or part of it) gives what the call on separate arrays gives, on
the first call of a shape, where the autotuner runs the step several times,
and on later ones, early-started.  chi^2 to 1e-4 relative and I and gradients to 1e-4 of
their largest value (the population's FP32 bars): the autotuner may choose another
order of summation in another context."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import crystal as X
from diffusecode_amd import fourier as FR
from diffusecode_amd.population import Population

pytestmark = pytest.mark.gpu


def close(a, b):
    return np.abs(a - b).max() <= 1e-4 * np.abs(b).max()


@pytest.mark.parametrize("case", ["icalc=target", "icalc=weight", "icalc inside target", "grad=pos", "grad over occ and bdw"])
def test_output_in_an_inputs_place(case):
    import torch
    dev = torch.device("cuda:0")
    crs = X.population(nmembers=4, nmin=300, nmax=1500, seed=5)
    eck, vi, inc = FR.grid_block((-3.0, -3.0, 0.0), (3.0, 3.0, 0.0), (65, 33, 1))
    ctx = _lib.Context(precision="fp32")
    try:
        pop = Population.from_crystals(crs, eck, vi, inc, ctx=ctx, precision="fp32")
        desc, keep = pop.desc()
        M, P, n = len(crs), pop.npixels, pop.natoms
        pos, occ, bdw = (torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in pop.params())
        rng = np.random.default_rng(2)
        T = torch.from_numpy(rng.uniform(1.0, 1e5, (M, P))).to(dev)
        W = torch.from_numpy(rng.uniform(0.5, 1.5, (M, P))).to(dev)
        grid = lambda: torch.zeros((M, P), dtype=torch.float64, device=dev)
        I, g = grid(), torch.zeros((n, 5), dtype=torch.float64, device=dev)
        torch.cuda.synchronize()
        chi = ctx.batch_chi2_dev(desc, pos, occ, bdw, T, W, icalc=I, grad=g)
        I, g = I.cpu().numpy(), g.cpu().numpy()
    finally:
        ctx.close()
    ctx = _lib.Context(precision="fp32")
    try:
        for call in range(3):
            p, o, b, t, w = (v.clone() for v in (pos, occ, bdw, T, W))
            i2, g2 = grid(), torch.zeros((n, 5), dtype=torch.float64, device=dev)
            if case == "icalc=target":
                i2 = t
            elif case == "icalc=weight":
                i2 = w
            elif case == "icalc inside target":
                big = torch.zeros(M * P + 7, dtype=torch.float64, device=dev)
                big[:M * P] = t.ravel()
                t, i2 = big[:M * P], big[7:]
            elif case == "grad=pos":
                g2 = torch.zeros((n, 5), dtype=torch.float64, device=dev)
                p = g2.view(-1)[:3 * n]
                p.copy_(pos.ravel())
            else:
                o, b = g2.view(-1)[n:2 * n], g2.view(-1)[3 * n:4 * n]
                o.copy_(occ)
                b.copy_(bdw)
            torch.cuda.synchronize()
            print(f"case in place {case} call {call}", flush=True)
            chi2 = ctx.batch_chi2_dev(desc, p, o, b, t, w, icalc=i2, grad=g2)
            assert np.abs(chi2 - chi).max() <= 1e-4 * chi.min(), call
            assert close(i2.cpu().numpy().reshape(M, P), I), call
            assert all(close(g2.cpu().numpy()[:, k], g[:, k]) for k in range(5)), call
    finally:
        ctx.close()


def test_pinned_host_arrays():
    """Arrays that are not memory of the context's device are copied, as inputs and as outputs."""
    import torch
    crs = X.population(nmembers=3, nmin=300, nmax=900, seed=6)
    eck, vi, inc = FR.grid_block((-3.0, -3.0, 0.0), (3.0, 3.0, 0.0), (35, 34, 1))
    ctx = _lib.Context(precision="fp32")
    try:
        ctx.set_autotune(False)
        pop = Population.from_crystals(crs, eck, vi, inc, ctx=ctx, precision="fp32")
        desc, keep = pop.desc()
        M, P, n = len(crs), pop.npixels, pop.natoms
        host = [torch.from_numpy(np.ascontiguousarray(v)).pin_memory() for v in pop.params()]
        T = torch.from_numpy(np.random.default_rng(2).uniform(1.0, 1e5, (M, P))).pin_memory()
        out = []
        for where in ("cuda:0", "cpu"):
            a = [v.to(where) for v in host]
            t = T.to(where)
            i = torch.zeros((M, P), dtype=torch.float64)
            g = torch.zeros((n, 5), dtype=torch.float64)
            i, g = (i.pin_memory(), g.pin_memory()) if where == "cpu" else (i.to(where), g.to(where))
            torch.cuda.synchronize()
            chi = ctx.batch_chi2_dev(desc, *a, t, icalc=i, grad=g)
            out.append((chi, i.cpu().numpy(), g.cpu().numpy()))
        assert all(np.array_equal(x, y) for x, y in zip(*out))
    finally:
        ctx.close()
