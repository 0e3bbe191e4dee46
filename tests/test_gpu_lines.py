"""Line transforms (dc_fft.h) in the calls that use them: the resolution
convolution at lengths of every radix, at squares and products of the large
ones, on both sides of the lengths where the work-group or the kernel changes
(256, 512), with one large prime factor (29 to 199), at the longest (600) and
beyond it or with a larger prime factor (the library's transforms), along each axis; and the run-level NUFFT on fine
grids of odd tile counts, even and odd mode counts, subsampled modes, points
on and beyond the cell's edges, against the direct sum.

Bars: 1e-12 of the largest value for the convolution (FP64 rounding of two
different transforms, as for the other post-processing tests); the NUFFT's own
1e-6 of the largest |F| at its tolerance of 1e-7."""
import numpy as np
import pytest

from diffusecode_amd import _lib
from diffusecode_amd import fourier as FR
from oracle import post as P

pytestmark = pytest.mark.gpu

TR = [0.7, 0.1, 0.0, -0.05, 0.9, 0.0, 0.0, 0.02, 1.1]
SIG = [1.0, 1.3, 0.8]
RTEN = (np.eye(3) / 5.64 ** 2).ravel(order="F")


@pytest.fixture(scope="module")
def ctx():
    c = _lib.Context()
    yield c
    c.close()


LENGTHS = [2, 3, 4, 5, 7, 8, 9, 11, 13, 17, 19, 23, 6, 121, 143, 161, 289, 437, 529, 81, 125, 128, 243, 256, 264, 343,
           486, 500, 512, 513, 567, 598, 600, 602, 29, 58, 31 * 8, 31 * 19, 37, 127, 254, 157, 199, 597, 211, 620]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", LENGTHS)
def test_conv_lengths(ctx, n, axis):
    num = {0: (n, 1, 1), 1: (5, n, 1), 2: (3, 4, n)}[axis]
    if axis == 0 and n < 3:
        num = (n, 9, 1)
    rng = np.random.default_rng(n)
    csf = rng.standard_normal(num) + 1j * rng.standard_normal(num)
    dsi = rng.random(num) + 0.1
    lo = [-(k // 2) * 0.1 for k in num]
    eck, vi, inc = FR.grid_block(lo, [l + (k - 1) * 0.1 for l, k in zip(lo, num)], num)
    print(f"case conv lengths {num}", flush=True)
    d = ctx.post_desc(num, eck, vi, RTEN, 1.0 / 180.0, fave=1.0, lots_off=True, res_sigma=SIG, res_tr=TR)
    c, s, _ = ctx.four_post(d, csf, dsi, want_dsi3d=False)
    rc, rs, _ = P.four_conv(num, SIG, TR, csf, dsi, lots_off=True, fave=1.0)
    assert np.abs(c - rc).max() <= 1e-12 * np.abs(rc).max()
    assert np.abs(s - rs).max() <= 1e-12 * np.abs(rs).max()


@pytest.mark.parametrize("inc,scales", [((5, 5, 5), (1, 1, 1)), ((9, 8, 11), (1, 1, 1)), ((17, 5, 6), (1, 3, 2)),
                                        ((41, 6, 27), (1, 1, 1)), ((6, 81, 9), (2, 1, 1)), ((128, 3, 4), (1, 4, 3)),
                                        ((150, 3, 3), (1, 3, 3)), ((3, 3, 280), (4, 4, 1)), ((301, 4, 4), (1, 2, 2))])
def test_strucf_nufft_shapes(ctx, inc, scales):
    """Fine grids of 16 points (the kernel's reach) up to 600 and beyond."""
    rng = np.random.default_rng(sum(inc))
    n = 300
    x = rng.uniform(-np.pi, np.pi, (3, n))
    x[:, 0] = 0.0
    x[:, 1] = -np.pi
    x[:, 2] = np.pi
    x[:, 3] = (7.0, -20.0, 1e3)          # periodic
    x[:, 4:40] = x[:, 4:5]               # many points of one bin
    print(f"case nufft shapes {inc} {scales}", flush=True)
    F = ctx.four_strucf_nufft(x, 0.75, inc, scales)
    k = [np.arange(inc[d]) * scales[d] - ((inc[d] - 1) * scales[d] + 1) // 2 for d in range(3)]
    e = [np.exp(1j * np.outer(k[d], x[d])) for d in range(3)]
    ref = 0.75 * np.einsum("an,bn,cn->abc", *e, optimize=True)
    F = np.asarray(F).reshape(inc, order="F") if np.asarray(F).shape != tuple(inc) else np.asarray(F)
    assert np.abs(F - ref).max() <= 1e-6 * np.abs(ref).max()
