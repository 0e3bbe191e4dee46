// dc_adjoint.hip -- reverse-mode derivative of the structure-factor path.
//
// Model (per atom n of scattering type t, fractional position x_n,
// occupancy o_n, isotropic displacement B_n):
//     F(p) = sum_n f_t(p) o_n exp(-B_n s_p^2) exp(2 pi i h_p . x_n),   I = |F|^2.
// For a loss L(I) with G_p = dL/dI_p put Q_t(p) = 2 G_p conj(F_p) f_t(p) and
// E_n(p) = exp(-B_n s_p^2) exp(2 pi i h_p . x_n).  Then
//     dL/do_n     = Re sum_p Q E
//     dL/dx_n,a   = -2 pi o_n Im sum_p h_p,a Q E
//     dL/dB_n     = -o_n Re sum_p s_p^2 Q E.
// REFINE obtains these by re-running the Fourier calculation for every
// parameter (finite differences, refine/prog/refine_run.f90:491-600); here
// they come from one pass that reuses the forward's phase generation.
//
// GEMM form (grid rows r = abscissa, columns c = (ordinate, top) flattened;
// the grid must be metric-orthogonal between rows and
// columns so that s^2 = s_r^2 + s_c^2 and E splits as A(r,n) B(c,n)):
//     Z_w(n, c) = sum_r w(r) A(r, n) Q(r, c),   w in {1, r - rc, s_r^2}
// on MFMA, then an epilogue contracts each Z with the column factor B(c, n)
// and the column weights (1, j - jc, m - mc, s_c^2).  h_p,a is affine in
// (r, j, m), so the three row weights and four column weights give every
// sum above; the weights are centred to keep the FP32 terms small.
//
// Mirrored rows.  About the centre of the rows A(+-j) = d_j (cos +- i sin),
// so that with S = wQ(+j) + wQ(-j) and D = wQ(+j) - wQ(-j)
//     sum over +-j of w A Q = d_j (cos S + i sin D):
// half the real products of the row-by-row sum, for every weight.  It needs
// d_j = exp(-B s_j^2) alike on both sides (s_r^2 mirrored, or no B); other
// grids run the same kernel with each row as its own pair, where the
// coefficients of cos and sin are Q and iQ.
//
// The coefficients (weights applied, S and D formed in FP32) are split once per
// call into 16-bit parts and stored as the words of the MFMA operand
// (adj_words_kernel): 3 parts and 6 products (hh, hm, mh, hl, lh, mm) in FP32,
// which keep 24 bits of both operands -- the dropped terms are below 2^-25 of a
// product, less than FP32's own rounding of it.  The split precisions take 2
// FP16 parts and 3 products, the coefficients of a column scaled by a power of
// two to FP16's range (22 bits against the largest; two BF16 parts
// hold 16, and S and D, being sums, then cost 1.4 times the row-by-row
// error).  FP16's range also has to hold the row factor exp(-B s_r^2): the atoms
// of a plane carry exp(-(B - Bref) s_r^2) and its coefficients exp(-Bref s_r^2)
// (adj_begin_kernel).  Either unit runs 16 times the FP32 rate.
#include <algorithm>
#include <atomic>

#include "dc_gemm_dev.h"

namespace dc {

namespace {

constexpr int AW = 4;               // waves of a work-group
constexpr int NT = 64 * AW;
constexpr int WA = 2;               // 16-atom tiles of a wave
constexpr int NA = 16 * WA * AW;    // atoms of a work-group
constexpr int CT = 16;              // grid columns of a tile
constexpr int KP = 16;              // row pairs of a k-step: one 16x16x32 product
constexpr int WALK_TILES = 256 / CT;   // tiles of one unit of the column walk
constexpr int MAX_WALK = 32;
constexpr int MAX_GROUPS = 64;      // column ranges, each a partial set
constexpr int RESYNC = 4;           // tiles between exact column phases
constexpr float LOG2E = 1.4426950408889634f;
// k-steps a wave keeps its A operands of in registers (24 VGPRs a step with 3
// parts, 16 with 2); longer grids are cut into row chunks, each a partial set.
constexpr int max_ksteps(int parts) { return parts == 3 ? 3 : 5; }

// (x, y) as NP pairs (x in the low half) whose sums are x and y: three BF16
// parts, exactly, or two FP16 parts, to 2^-23 (2^-25 where that is larger)
template <int NP>
__device__ __forceinline__ void split(float x, float y, uint32_t (&part)[NP]) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        if constexpr (NP == 3) {
            const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, bf16x2));
            part[p] = h;
            x -= __builtin_bit_cast(float, h << 16);
            y -= __builtin_bit_cast(float, h & 0xFFFF0000u);
        } else {
            const f16x2 h = __builtin_convertvector((f32x2){x, y}, f16x2);
            part[p] = __builtin_bit_cast(uint32_t, h);
            x -= (float)h[0];
            y -= (float)h[1];
        }
    }
}
template <int NP>
__device__ __forceinline__ f32x4 mfma(u32x4 x, u32x4 y, f32x4 c) {
    if constexpr (NP == 3)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), c, 0, 0, 0);
}

__device__ __forceinline__ float exp2i(int e) { return __builtin_bit_cast(float, (uint32_t)(e + 127) << 23); }
// e with 2^e <= x < 2^(e + 1), kept at -113 at least, so that 2^(13 - e) and its
// reciprocal are normal numbers (0 of zero)
__device__ __forceinline__ int exponent(float x) {
    return x == 0.0f ? 0 : min(127, max(-113, (int)(__builtin_bit_cast(uint32_t, x) >> 23 & 0xFF) - 127));
}
// Powers of two that bring the row weights to 1 at most (2 parts; 1 with 3).
template <int NP>
__device__ __forceinline__ void weight_scales(const AdjArgs &a, const float *__restrict__ sq, float (&sg)[3]) {
    sg[0] = sg[1] = sg[2] = 1.0f;
    if constexpr (NP == 2) {
        float m = 0.0f;
        for (int r = threadIdx.x & 63; r < a.R; r += 64) m = fmaxf(m, fabsf(sq[r]));
#pragma unroll
        for (int h = 1; h < 64; h *= 2) m = fmaxf(m, __shfl_xor(m, h));
        sg[1] = exp2i(-1 - exponent(fmaxf(a.rc, 0.5f)));
        sg[2] = exp2i(-1 - exponent(m));
    }
}

__device__ __forceinline__ float2 cis(uint64_t ph) {
    float c, s;
    sincos_turn_fine((uint32_t)((ph + 0x80000000ull) >> 32), c, s);
    return make_float2(c, s);
}
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Rows of pair p: r1 and, when folded, its mirror r0 (-1: none); false past the
// last pair.  a.center: the centre row is no pair, the epilogue adds it.
__device__ __forceinline__ bool pair_rows(const AdjArgs &a, int p, int &r1, int &r0) {
    r0 = -1;
    if (!a.fold) {
        r1 = p;
        return p < a.R;
    }
    const int h = a.R / 2;
    p += a.center;
    r1 = h + p;
    if (a.R & 1) {
        if (p > 0) r0 = h - p;
    } else {
        r0 = h - 1 - p;
    }
    return r1 < a.R;
}

// What a reverse pass starts with: the gradient array cleared (vacancies keep 0)
// and, for damped passes in 2 parts, Bref (times log2(e)) of every plane, a
// work-group each: the least B of the plane's atoms, whose row factors
// exp(-(B - Bref) s_r^2) are then at most 1 and hold 17 bits or more down to
// 2^-7; where B spreads further over the rows, Bref moves up, to factors of
// 2^14 at most (B may spread over 21 / s_r^2 in all).  Unlike in the forward sum
// a small factor is not small beside others: it is alone in its atom's gradient.
// Bound by latency: two dependent reads beside the clearing, which alone took a
// launch of its own before.
constexpr int BEGIN_THREADS = 1024;
__global__ void __launch_bounds__(BEGIN_THREADS) adj_begin_kernel(AdjArgs a, int nref, double *__restrict__ grad, long long ngrad) {
    __shared__ float red[3][BEGIN_THREADS / 64];
    if ((int)blockIdx.x >= nref) {
        for (long long k = (long long)(blockIdx.x - nref) * BEGIN_THREADS + threadIdx.x; k < ngrad;
             k += (long long)(gridDim.x - nref) * BEGIN_THREADS)
            grad[k] = 0.0;
        return;
    }
    const int plane = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int2 range = a.ranges[plane];
    float b0 = NO_B, b1 = -NO_B, s = 0.0f;
    for (long long k = range.x + (int)threadIdx.x; k < range.y; k += 8 * BEGIN_THREADS) {
        float b[8];                        // eight reads in flight
#pragma unroll
        for (int u = 0; u < 8; ++u) b[u] = a.rec[min(k + u * BEGIN_THREADS, (long long)range.y - 1)].pad;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            b0 = fminf(b0, b[u]);
            b1 = fmaxf(b1, b[u]);
        }
    }
    const float *sq = a.sq + (long long)(plane / a.planes_per_sq) * a.sq_stride;
    for (int r = threadIdx.x; r < a.R; r += BEGIN_THREADS) s = fmaxf(s, fabsf(sq[r]));
#pragma unroll
    for (int h = 1; h < 64; h *= 2) {
        b0 = fminf(b0, __shfl_xor(b0, h));
        b1 = fmaxf(b1, __shfl_xor(b1, h));
        s = fmaxf(s, __shfl_xor(s, h));
    }
    if (lane == 0) {
        red[0][wave] = b0;
        red[1][wave] = b1;
        red[2][wave] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < BEGIN_THREADS / 64; ++w) {
            b0 = fminf(b0, red[0][w]);
            b1 = fmaxf(b1, red[1][w]);
            s = fmaxf(s, red[2][w]);
        }
        a.ref[plane] = b0 > b1 || !(s > 0.0f) ? 0.0f
                       : LOG2E * b0 + fminf(fmaxf(LOG2E * (b1 - b0) - 7.0f / s, 0.0f), 14.0f / s);
    }
}

// Q planes -> operand words of one (plane, column tile, k-step): for weight w,
// component (re, im) and part, lane l holds column l % 16 of the tile and the
// (cos, sin) coefficients of pairs 4 (l / 16) .. + 3 of the step.
// One work-group per (plane, tile), a wave per k-step.  2 parts: the coefficients
// of each column, times the rows' exp(-Bref s_r^2), are scaled to below 2^15 (by
// column, since what the columns' own exp(-B s_c^2) leaves of them differs), and the
// scales noted: scales[plane][tile][column], then the tiles' least ones.
template <int NP>
__global__ void __launch_bounds__(256) adj_words_kernel(AdjArgs a, int plane0, int nplane, u32x4 *__restrict__ out) {
    constexpr int NW = 6 * NP;
    __shared__ float red[4][CT];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *scales = reinterpret_cast<float *>(out + (long long)nplane * a.ctiles * a.nkt * (NW * 64));
    float *tscales = scales + (long long)nplane * a.ctiles * CT;
    for (long long x = blockIdx.x; x < (long long)nplane * a.ctiles; x += gridDim.x) {
        const int ct = (int)(x % a.ctiles), pl = (int)(x / a.ctiles);
        const int c = ct * CT + (lane & 15);
        const bool in = c < a.C && c % a.C0 < a.f1;
        const float *sq = a.sq + (long long)((plane0 + pl) / a.planes_per_sq) * a.sq_stride;
        const float2 *q = a.q + (long long)(plane0 + pl) * a.plane + c;
        float sg[3], scale = 1.0f, bref = 0.0f;
        weight_scales<NP>(a, sq, sg);
        if constexpr (NP == 2) {
            if (a.damped) bref = a.ref[plane0 + pl];
            float m = 0.0f;
            if (in)
                for (int r = threadIdx.x >> 4; r < a.R; r += 16) {
                    const float2 v = q[(long long)a.C * r];
                    m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)) * damp_back(bref, sq[r]));
                }
            m = fmaxf(m, __shfl_xor(m, 16));
            m = fmaxf(m, __shfl_xor(m, 32));
            __syncthreads();   // the previous tile's maxima have been read
            if (lane < CT) red[wave][lane] = m;
            __syncthreads();
            const int col = lane & 15;
            m = fmaxf(fmaxf(red[0][col], red[1][col]), fmaxf(red[2][col], red[3][col]));
            scale = exp2i(13 - exponent(m));
#pragma unroll
            for (int h = 1; h < CT; h *= 2) m = fmaxf(m, __shfl_xor(m, h));
            if (threadIdx.x < CT) scales[x * CT + col] = scale;
            if (threadIdx.x == 0) tscales[x] = exp2i(13 - exponent(m));
        }
        for (int k = wave; k < a.nkt; k += 4) {
            u32x4 w[3][2][NP];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                int r1, r0;
                float2 q1 = make_float2(0.f, 0.f), q0 = q1;
                float w1[3] = {1.0f, 0.0f, 0.0f}, w0[3] = {1.0f, 0.0f, 0.0f};
                const bool pair = pair_rows(a, KP * k + 4 * (lane >> 4) + e, r1, r0);
                if (in && pair) {
                    q1 = q[(long long)a.C * r1];
                    w1[1] = ((float)r1 - a.rc) * sg[1];
                    w1[2] = sq[r1] * sg[2];
                    if (r0 >= 0) {
                        q0 = q[(long long)a.C * r0];
                        w0[1] = ((float)r0 - a.rc) * sg[1];
                        w0[2] = sq[r0] * sg[2];
                    }
                }
                if constexpr (NP == 2) {
                    // (one factor for both rows of a pair, as their s_r^2 is one)
                    const float f = in && pair ? damp_back(bref, sq[r1]) * scale : 0.0f;
                    q1 = make_float2(q1.x * f, q1.y * f);
                    q0 = make_float2(q0.x * f, q0.y * f);
                }
#pragma unroll
                for (int v = 0; v < 3; ++v) {
                    const float2 x1 = make_float2(q1.x * w1[v], q1.y * w1[v]), x0 = make_float2(q0.x * w0[v], q0.y * w0[v]);
                    uint32_t re[NP], im[NP];
                    split<NP>(x1.x + x0.x, x0.y - x1.y, re);   // S.re, -D.im
                    split<NP>(x1.y + x0.y, x1.x - x0.x, im);   // S.im, D.re
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        w[v][0][p][e] = re[p];
                        w[v][1][p][e] = im[p];
                    }
                }
            }
            u32x4 *o = out + (x * a.nkt + k) * (NW * 64) + lane;
#pragma unroll
            for (int v = 0; v < 6; ++v)
#pragma unroll
                for (int p = 0; p < NP; ++p) o[(v * NP + p) * 64] = w[v >> 1][v & 1][p];
        }
    }
}

// What bounds it: the matrix products (36 or 18 of 16x16x32 a k-step, wave and
// atom tile) with the epilogue's VALU work beside them.  A wave owns 32 atoms:
// their A operands of every k-step of the row chunk stay in registers, made
// once; the work-group's waves share the words of one (column tile, k-step)
// through LDS, double-buffered, the next step's loads in flight in registers
// while this one's products run (one barrier a step).  The words are the
// MFMA's rows and the atoms its columns, so a lane's 4 results of a tile
// belong to one atom: the epilogue sums them in the lane and keeps six FP64
// totals an atom over the whole column range, with no exchange until the end.
// (32x32x16 products, the same work, need twice the accumulators and spilled.)
// An odd row count whose centre row would open a k-step of its own (65 rows:
// 32 pairs and the centre) has it added by the epilogue instead, in FP32.
// Measured, 32,768 atoms on 65^3 points in FP32: 2.55 ms of FP32 products row
// by row -> 0.55 ms (0.25 ms of it matrix products at their peak) + 0.012 ms
// for the words; 24 members on 129^2 in the split precisions 0.595 -> 0.15 ms.
// The gradient's error against FP64 (relative to its norm; x, occ, B) went from
// 1.8e-7, 9e-8, 1.0e-7 to 1.2e-7, 5e-8, 6e-8 in FP32 and from 3.5e-6,
// 1.1e-6, 1.8e-6 to 1.4e-7, 6e-8, 7e-8 in the split precisions.
template <int NP, int NK>
__global__ void __launch_bounds__(NT, 2) adjoint_kernel(AdjArgs a, int tile0, int plane0, int nplane, int chunk0, const u32x4 *__restrict__ words) {
    constexpr int NW = 6 * NP, LD = (NW + AW - 1) / AW;
    __shared__ u32x4 sq_w[2][NW][64];
    // Values of a tile's columns: those of tile t + 1 are stored in the last
    // k-step of tile t, before that step's barrier.  With two k-steps or more the
    // barrier of the first one has let every wave out of the epilogue of tile t - 1,
    // whose slot they may take.  With one k-step a slower wave may still be in it:
    // three slots, of which tile t + 1 takes that of t - 2, whose epilogue every
    // wave left before the barrier that ended tile t - 1.
    constexpr int SLOTS = NK == 1 ? 3 : 2;
    __shared__ float4 col[SLOTS][CT];      // s_c^2, j - jc, m - mc, scaled s_c^2 of the tile's columns
    __shared__ float2 qcen[SLOTS][CT];     // Q of the centre row
    __shared__ float crel[SLOTS][CT];      // scale of the tile over that of the column (2 parts)
    auto slot_of = [](int ct) { return SLOTS == 2 ? ct & 1 : (int)((unsigned)ct % SLOTS); };
    const int4 tile = a.tiles[tile0 + blockIdx.y];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int li = lane & 15, lg = lane >> 4;
    const float *sq = a.sq + (long long)tile.w * a.sq_stride;
    const int group = blockIdx.x % a.groups, chunk = chunk0 + blockIdx.x / a.groups;
    const int ct0 = group * a.tpg, ct1 = min(a.ctiles, ct0 + a.tpg);
    const int k0 = chunk * NK;
    const int n0 = tile.x + wave * 16 * WA + li;
    const bool active = tile.x + wave * 16 * WA < tile.y;      // wave-uniform
    const bool center = a.center && chunk == 0;
    float sg[3];
    weight_scales<NP>(a, sq, sg);
    // scales of the columns and of the tiles (adj_words_kernel)
    const float *scales = reinterpret_cast<const float *>(words + (long long)nplane * a.ctiles * a.nkt * (NW * 64));
    const float *tscales = scales + (long long)nplane * a.ctiles * CT;
    float bref = 0.0f;
    if constexpr (NP == 2)
        if (a.damped) bref = a.ref[tile.z];
    scales += (long long)(tile.z - plane0) * a.ctiles * CT;
    tscales += (long long)(tile.z - plane0) * a.ctiles;
    const float s2c = sq[a.R / 2], s2cs = s2c * sg[2];

    // per atom: A operands, phase of the row origin, column factors: tl[v] of
    // the 4 columns a lane holds, rot of one tile, wrap of a step from the end
    // of one ordinate run to the next (runs are at least a tile long)
    u32x4 A[NK][WA][NP];
    uint64_t ph[WA], ca[WA], ca1[WA];
    float bl2[WA], cen[WA];
    float2 tl[WA][4], rot[WA], wrap[WA];
    const bool half = a.fold && !(a.R & 1);    // the centre lies half a step past row (R - 1) / 2
#pragma unroll
    for (int i = 0; i < WA; ++i) {
        AtomRec at{};
        if (n0 + 16 * i < tile.y) at = a.rec[n0 + 16 * i];
        const uint64_t hs = half ? at.ra >> 1 : 0;
        bl2[i] = -at.pad * LOG2E;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int p = KP * (k0 + k) + 4 * lg + e;
                int r1, r0;
                float2 v = make_float2(0.f, 0.f);
                if (pair_rows(a, p, r1, r0)) {
                    v = cis((uint64_t)(p + a.center) * at.ra + hs);
                    const float d = __builtin_amdgcn_exp2f((bl2[i] + bref) * sq[r1]);
                    v = make_float2(v.x * d, v.y * d);
                }
                uint32_t w[NP];
                split<NP>(v.x, v.y, w);
#pragma unroll
                for (int q = 0; q < NP; ++q) A[k][i][q][e] = w[q];
            }
        ph[i] = at.p0 + hs + (a.fold ? (uint64_t)((a.R - 1) / 2) * at.ra : 0);
        ca[i] = at.ca;
        ca1[i] = at.ca1;
        cen[i] = __builtin_amdgcn_exp2f(bl2[i] * s2c);
        rot[i] = cis(CT * at.ca);
        wrap[i] = cis(at.ca1 - (uint64_t)a.C0 * at.ca);
#pragma unroll
        for (int v = 0; v < 4; ++v) tl[i][v] = cis((uint64_t)v * at.ca);
    }
    const bool damp = __any(bl2[0] != 0.0f || bl2[1] != 0.0f);
    static_assert(WA == 2, "damp");

    double tot[WA][6];
#pragma unroll
    for (int i = 0; i < WA; ++i)
#pragma unroll
        for (int k = 0; k < 6; ++k) tot[i][k] = 0.0;
    // words of (column tile, k-step): contiguous over the chunk's steps, then a
    // jump over the other chunks' to the next column tile
    const u32x4 *src = words + (((long long)(tile.z - plane0) * a.ctiles + ct0) * a.nkt + k0) * (NW * 64);
    const long long jump = (long long)(a.nkt - NK + 1) * (NW * 64);
    u32x4 reg[LD];
    auto fetch = [&]() {
#pragma unroll
        for (int u = 0; u < LD; ++u)
            if (AW * (u + 1) <= NW || wave + AW * u < NW) reg[u] = src[(wave + AW * u) * 64 + lane];
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int u = 0; u < LD; ++u)
            if (AW * (u + 1) <= NW || wave + AW * u < NW) sq_w[buf][wave + AW * u][lane] = reg[u];
    };
    // the next tile's column values likewise, a tile ahead (threads 0..15)
    float csq = 0.0f, cr = 1.0f;
    float2 cq = make_float2(0.f, 0.f);
    int cj = 0, cm = 0;
    auto fetch_col = [&](int ct) {
        const int c = ct * CT + (int)threadIdx.x;
        cj = c % a.C0;
        cm = c / a.C0;
        const bool in = threadIdx.x < CT && c < a.C && cj < a.f1;
        csq = in ? sq[a.R + c] : 0.0f;
        cq = in && center ? a.q[tile.z * a.plane + c + (long long)a.C * (a.R / 2)] : make_float2(0.f, 0.f);
        if constexpr (NP == 2)
            if (in) {
                const float scale = scales[ct * CT + (int)threadIdx.x];
                cq = make_float2(cq.x * scale, cq.y * scale);
                cr = tscales[ct] / scale;      // powers of two
            }
    };
    auto put_col = [&](int ct) {
        if (threadIdx.x < CT) {
            col[slot_of(ct)][threadIdx.x] = make_float4(csq, (float)cj - a.jc, (float)cm - a.mc, csq * sg[2]);
            qcen[slot_of(ct)][threadIdx.x] = cq;
            if constexpr (NP == 2) crel[slot_of(ct)][threadIdx.x] = cr;
        }
    };
    if (ct0 < ct1) {
        fetch();
        fetch_col(ct0);
        put(0);
        put_col(ct0);
    }
    __syncthreads();
    int buf = 0;
    float2 th[WA];
    for (int ct = ct0; ct < ct1; ++ct) {
        f32x4 acc[6][WA];
#pragma unroll
        for (int x = 0; x < 6; ++x)
#pragma unroll
            for (int i = 0; i < WA; ++i) acc[x][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            // (the last step of the range fetches its own words again)
            src += k + 1 < NK ? NW * 64 : ct + 1 < ct1 ? jump : 0;
            fetch();
            if (k == 0) fetch_col(ct + 1);
            if (active) {
#pragma unroll
                for (int x = 0; x < 6; ++x) {
                    u32x4 w[NP];
#pragma unroll
                    for (int p = 0; p < NP; ++p) w[p] = sq_w[buf][x * NP + p][lane];
                    // the small products first
#pragma unroll
                    for (int s = NP - 1; s >= 0; --s)
#pragma unroll
                        for (int p = s; p >= 0; --p)
#pragma unroll
                            for (int i = 0; i < WA; ++i)
                                acc[x][i] = mfma<NP>(w[p], A[k][i][s - p], acc[x][i]);
                }
            }
            put(buf ^ 1);
            if (k == NK - 1) put_col(ct + 1);
            buf ^= 1;
            __syncthreads();
        }
        if (!active) continue;
        // contraction with the column factors: lane holds columns 4 lg + v
        const int cb = ct * CT + 4 * lg, j0 = cb % a.C0, m0 = cb / a.C0;
        if ((ct - ct0) % RESYNC == 0) {
#pragma unroll
            for (int i = 0; i < WA; ++i) th[i] = cis(ph[i] + (uint64_t)j0 * ca[i] + (uint64_t)m0 * ca1[i]);
        } else {
#pragma unroll
            for (int i = 0; i < WA; ++i) {
                th[i] = cmul(th[i], rot[i]);
                const float2 t = cmul(th[i], wrap[i]);
                th[i] = j0 < CT ? t : th[i];   // the lane's columns began a new run since the last tile
            }
        }
        double inv = 1.0;
        if constexpr (NP == 2) inv = (double)(1.0f / tscales[ct]);   // a power of two: exact
        float4 w[4];
        float2 qc[4];
        float d[WA][4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            w[v] = col[slot_of(ct)][4 * lg + v];
            qc[v] = qcen[slot_of(ct)][4 * lg + v];
#pragma unroll
            for (int i = 0; i < WA; ++i) d[i][v] = NP == 2 ? crel[slot_of(ct)][4 * lg + v] : 1.0f;
        }
        if (damp)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int i = 0; i < WA; ++i) d[i][v] *= __builtin_amdgcn_exp2f(bl2[i] * w[v].x);
#pragma unroll
        for (int i = 0; i < WA; ++i) {
            const float2 thw = cmul(th[i], wrap[i]);
            float s[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float2 b = cmul(j0 + v >= a.C0 ? thw : th[i], tl[i][v]);
                b = make_float2(b.x * d[i][v], b.y * d[i][v]);
                const float qr = cen[i] * qc[v].x, qi = cen[i] * qc[v].y;
                const float z0r = acc[0][i][v] + qr, z0i = acc[1][i][v] + qi;
                const float z2r = acc[4][i][v] + s2cs * qr, z2i = acc[5][i][v] + s2cs * qi;
                const float tr = z0r * b.x - z0i * b.y;
                const float ti = z0r * b.y + z0i * b.x;
                s[0] += tr;
                s[1] += ti;
                s[2] += acc[2][i][v] * b.y + acc[3][i][v] * b.x;
                s[3] += w[v].y * ti;
                s[4] += w[v].z * ti;
                s[5] += (z2r * b.x - z2i * b.y) + w[v].w * tr;
            }
#pragma unroll
            for (int k = 0; k < 6; ++k) tot[i][k] = NP == 2 ? __builtin_fma((double)s[k], inv, tot[i][k]) : tot[i][k] + (double)s[k];
        }
    }
    if (!active) return;
#pragma unroll
    for (int i = 0; i < WA; ++i) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            tot[i][k] += __shfl_xor(tot[i][k], 16);
            tot[i][k] += __shfl_xor(tot[i][k], 32);
        }
        tot[i][2] /= (double)sg[1];
        tot[i][5] /= (double)sg[2];
        if (lg == 0 && n0 + 16 * i < tile.y) {
            double *out = a.part + ((long long)blockIdx.x * a.natoms + n0 + 16 * i) * 6;
#pragma unroll
            for (int k = 0; k < 6; ++k) out[k] = chunk0 > 0 ? out[k] + tot[i][k] : tot[i][k];
        }
    }
}

// Partial sets -> gradients in the caller's atom order (FP64).
__global__ void adjoint_finish_kernel(AdjFinishArgs a) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= a.natoms) return;
    double s[6] = {0, 0, 0, 0, 0, 0};
    for (int t = 0; t < a.nset; ++t) {
        const double *p = a.part + ((long long)t * a.natoms + n) * 6;
        for (int k = 0; k < 6; ++k) s[k] += p[k];
    }
    const long long ci = a.idx[n];
    const double o = a.occ[ci];
    const double twopi = 6.283185307179586476925;
    double *g = a.grad + 5 * ci;
    for (int c = 0; c < 3; ++c)
        g[c] = -twopi * o * (a.hc[c] * s[1] + a.v[c] * s[2] + a.v[3 + c] * s[3] + a.v[6 + c] * s[4]);
    g[3] = s[0];
    g[4] = -o * s[5];
}

// Q planes: Q_t(p) = 2 G_p conj(F_p) f_t(bin p), column-fastest layout.
__global__ void model_q_kernel(QArgs a) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.g.P) return;
    const int i = (int)(p % a.g.f[0]);
    const long long q = p / a.g.f[0];
    const int j = (int)(q % a.g.f[1]), m = (int)(q / a.g.f[1]);
    int bin = istl_point(a.g, i, j, m);
    bin = bin >= a.ncfact ? a.ncfact - 1 : bin;
    const double fr = a.f[2 * p], fi = a.f[2 * p + 1], g2 = 2.0 * a.gi[p];
    const double rr = g2 * fr, ri = -g2 * fi;                 // 2 G conj(F)
    const long long o = (long long)j + (long long)a.C0 * m + (long long)a.C * i;
    for (int t = 0; t < a.nq; ++t) {
        const double2 u = a.cfact[(long long)a.qtype[t] * a.ncfact + bin];
        a.q[t * a.plane + o] = make_float2((float)(rr * u.x - ri * u.y), (float)(rr * u.y + ri * u.x));
    }
}

// G = 2 w (I - T) and per-block sums of w (I - T)^2 (FP64).
__global__ void chi2_resid_kernel(const double *icalc, const double *tgt, const double *wt, long long n, double *gi,
                                  double *blocksum) {
    __shared__ double red[256];
    double acc = 0.0;
    for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (long long)gridDim.x * blockDim.x) {
        const double w = wt ? wt[p] : 1.0;
        const double d = icalc[p] - tgt[p];
        gi[p] = 2.0 * w * d;
        acc += w * d * d;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) blocksum[blockIdx.x] = red[0];
}

// One member per blockIdx.y; grid-stride over the member's pixels.  A
// pixel's planes are loaded BR_BATCH at a time, all issued before they are
// summed (planes past the member's last slice repeat it, so every load is
// in bounds); CF_LDS: the pixel's form factor of each of the a.nscat
// (<= BR_LDS_TYPES) types is read once into LDS, so that the sums and the Q
// planes wait on no further global load.  Same arithmetic, same order, with
// or without.
constexpr int BR_BATCH = 8;
constexpr int BR_BLOCK = 256;
constexpr int BR_LDS_TYPES = 8;
template <bool CF_LDS>
__global__ __launch_bounds__(BR_BLOCK) void batch_reduce_kernel(BatchReduceArgs a) {
    __shared__ double red[BR_BLOCK];
    extern __shared__ double2 cf_lds[];   // CF_LDS: [type][thread]
    const int m = blockIdx.y;
    Grid g = a.g;
    for (int k = 0; k < 9; ++k) g.rten[k] = a.rten[9 * m + k];
    const long long P = g.P;
    const int s0 = a.mslice[m], s1 = a.mslice[m + 1];
    const double2 *cf = a.cfact + (long long)m * a.nscat * a.ncfact;
    double acc = 0.0;
    for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < P; p += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(p % g.f[0]);
        const long long q = p / g.f[0];
        const int j = (int)(q % g.f[1]), l = (int)(q / g.f[1]);
        int bin = istl_point(g, i, j, l);
        bin = bin >= a.ncfact ? a.ncfact - 1 : bin;
        const long long po = i * g.ps[0] + j * g.ps[1] + l * g.ps[2];
        if constexpr (CF_LDS)
            for (int t = 0; t < a.nscat; ++t) cf_lds[t * BR_BLOCK + threadIdx.x] = cf[(long long)t * a.ncfact + bin];
        auto cfv = [&](int t) {
            if constexpr (CF_LDS) return cf_lds[t * BR_BLOCK + threadIdx.x];
            else return cf[(long long)t * a.ncfact + bin];
        };
        // the member's slices come in runs of one type: sum a run's planes,
        // then apply that type's form factor once
        double fr = 0.0, fi = 0.0, sr = 0.0, si = 0.0;
        for (int sb = s0; sb < s1; sb += BR_BATCH) {
            // the batch's slice types first, then its planes: the sums wait
            // for the types without waiting for the planes behind them
            int tt[BR_BATCH + 1];
#pragma unroll
            for (int u = 0; u <= BR_BATCH; ++u) tt[u] = a.slice_type[min(sb + u, s1 - 1)];
            float2 v[BR_BATCH];
#pragma unroll
            for (int u = 0; u < BR_BATCH; ++u) v[u] = a.partial[(long long)min(sb + u, s1 - 1) * g.plane + po];
#pragma unroll
            for (int u = 0; u < BR_BATCH; ++u) {
                const int s = sb + u;
                if (s >= s1) break;
                sr += (double)v[u].x;
                si += (double)v[u].y;
                const int t = tt[u];
                if (s + 1 == s1 || tt[u + 1] != t) {
                    const double2 w = cfv(t);
                    fr += w.x * sr - w.y * si;
                    fi += w.x * si + w.y * sr;
                    sr = si = 0.0;
                }
            }
        }
        const long long mp = (long long)m * P + p;
        const double I = fr * fr + fi * fi;
        if (a.icalc) a.icalc[mp] = I;
        const double w = a.weight ? a.weight[mp] : 1.0;
        const double d = I - a.target[mp];
        acc += w * d * d;
        if (a.q) {
            const double g2 = 4.0 * w * d;                       // 2 G, G = 2 w (I - T)
            const double rr = g2 * fr, ri = -g2 * fi;
            const long long o = (long long)j + (long long)a.C0 * l + (long long)a.C * i;
            for (int t = 0; t < a.nscat; ++t) {
                const double2 u = cfv(t);
                a.q[((long long)m * a.nscat + t) * a.plane + o] =
                    make_float2((float)(rr * u.x - ri * u.y), (float)(rr * u.y + ri * u.x));
            }
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.chi_part[(long long)m * gridDim.x + blockIdx.x] = red[0];
}

__global__ void jvp_reduce_kernel(JvpArgs a) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= a.g.P) return;
    const Grid &g = a.g;
    const int i = (int)(p % g.f[0]);
    const long long q = p / g.f[0];
    const int j = (int)(q % g.f[1]), l = (int)(q / g.f[1]);
    int bin = istl_point(g, i, j, l);
    bin = bin >= a.ncfact ? a.ncfact - 1 : bin;
    double h[3];
    for (int k = 0; k < 3; ++k) h[k] = g.xm[k] + g.uin[k] * i + g.vin[k] * j + g.win[k] * l;
    double s2 = 0.0;
    for (int r = 0; r < 3; ++r)
        for (int k = 0; k < 3; ++k) s2 += h[r] * g.rten[r + 3 * k] * h[k];
    s2 *= 0.25;
    const long long po = i * g.ps[0] + j * g.ps[1] + l * g.ps[2];
    const double fr = a.f[2 * p], fi = a.f[2 * p + 1];
    const double twopi = 6.283185307179586476925;
    for (int d = 0; d < a.ndir; ++d) {
        double gr[5], gi[5];
        for (int c = 0; c < 5; ++c) {
            gr[c] = 0.0;
            gi[c] = 0.0;
            for (int sl = a.dslice[5 * d + c]; sl < a.dslice[5 * d + c + 1]; ++sl) {
                const float2 v = a.partial[(long long)sl * g.plane + po];
                const double2 u = a.cfact[(long long)a.slice_type[sl] * a.ncfact + bin];
                gr[c] += u.x * (double)v.x - u.y * (double)v.y;
                gi[c] += u.x * (double)v.y + u.y * (double)v.x;
            }
        }
        const double hr = h[0] * gr[1] + h[1] * gr[2] + h[2] * gr[3];
        const double hi = h[0] * gi[1] + h[1] * gi[2] + h[2] * gi[3];
        const double dr = gr[0] - twopi * hi - s2 * gr[4];
        const double di = gi[0] + twopi * hr - s2 * gi[4];
        a.di[(long long)d * g.P + p] = 2.0 * (fr * dr + fi * di);
        if (a.df) {
            a.df[2 * ((long long)d * g.P + p)] = dr;
            a.df[2 * ((long long)d * g.P + p) + 1] = di;
        }
    }
}

}  // namespace

hipError_t launch_batch_reduce(const BatchReduceArgs &a, int nblocks, hipStream_t st) {
    if (a.nmembers <= 0) return hipSuccess;
    if (a.nscat >= 1 && a.nscat <= BR_LDS_TYPES)
        batch_reduce_kernel<true>
            <<<dim3(nblocks, a.nmembers), BR_BLOCK, sizeof(double2) * BR_BLOCK * a.nscat, st>>>(a);
    else
        batch_reduce_kernel<false><<<dim3(nblocks, a.nmembers), BR_BLOCK, 0, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_jvp_reduce(const JvpArgs &a, hipStream_t st) {
    if (a.g.P <= 0 || a.ndir <= 0) return hipSuccess;
    jvp_reduce_kernel<<<(unsigned)((a.g.P + 255) / 256), 256, 0, st>>>(a);
    return hipGetLastError();
}

int adjoint_tile_atoms() { return NA; }
int adjoint_max_walk() { return MAX_WALK; }

int device_cu_count() {
    static std::atomic<int> cus[64];
    int dev = 0, ncu = 256;
    if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64) {
        ncu = cus[dev].load(std::memory_order_relaxed);
        if (ncu <= 0) {
            if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu <= 0)
                ncu = 256;
            cus[dev].store(ncu, std::memory_order_relaxed);
        }
    }
    return ncu;
}

void adjoint_plan(AdjArgs &a, int ntiles, bool split, int force) {
    a.parts = split ? 2 : 3;
    int pairs = a.fold ? (a.R + 1) / 2 : a.R;
    a.center = a.fold && (a.R & 1) && pairs > 1 && pairs % KP == 1;
    pairs -= a.center;
    const int ks = std::max(1, (pairs + KP - 1) / KP), maxk = max_ksteps(a.parts);
    a.chunks = (ks + maxk - 1) / maxk;
    a.nk = (ks + a.chunks - 1) / a.chunks;
    a.nkt = a.chunks * a.nk;
    a.ctiles = std::max(1, (a.C + CT - 1) / CT);
    a.tpg = a.ctiles;
    if (force > 0) {
        a.tpg = std::min(a.ctiles, force * WALK_TILES);
    } else if (ntiles > 0) {
        // Two work-groups fit a CU; a range costs its tiles and a prologue
        // (A operands, tables) worth about one tile.
        const long long slots = 2LL * device_cu_count(), items = (long long)ntiles * a.chunks;
        double best = 0.0;
        for (int g = 1; g <= std::min(a.ctiles, MAX_GROUPS); ++g) {
            const int tpg = (a.ctiles + g - 1) / g;
            if ((a.ctiles + tpg - 1) / tpg != g) continue;
            const double cost = (double)((items * g + slots - 1) / slots) * (tpg + 1.0);
            if (g == 1 || cost < best) {
                best = cost;
                a.tpg = tpg;
            }
        }
    }
    a.groups = (a.ctiles + a.tpg - 1) / a.tpg;
    // row chunks of later launches add to the sets of the first
    a.nchunk = (int)std::min<long long>(a.chunks, std::max<long long>(1, ADJ_PART_MAX / (48LL * a.groups * std::max(a.natoms, 1))));
    a.nset = a.groups * a.nchunk;
    a.walk = (a.tpg + WALK_TILES - 1) / WALK_TILES;
    a.plane_words = (long long)a.ctiles * a.nkt * 6 * a.parts * 64 + (a.ctiles * (CT + 1) + 3) / 4;   // and the scales
}

hipError_t launch_adj_begin(const AdjArgs &a, int nplanes, double *grad, long long ngrad, hipStream_t st) {
    const int nref = a.parts == 2 && a.damped ? nplanes : 0;
    if (nref > 0 && (!a.ranges || !a.ref || a.planes_per_sq < 1)) return hipErrorInvalidValue;
    const long long nz = std::min<long long>((std::max<long long>(ngrad, 0) + BEGIN_THREADS - 1) / BEGIN_THREADS, 1024);
    if (nref + nz <= 0) return hipSuccess;
    adj_begin_kernel<<<(unsigned)(nref + nz), BEGIN_THREADS, 0, st>>>(a, nref, grad, ngrad);
    return hipGetLastError();
}

hipError_t launch_adjoint(const AdjArgs &a, const AdjSpan &s, uint4 *words, hipStream_t st) {
    if (s.ntiles <= 0 || a.R <= 0 || a.C <= 0) return hipSuccess;
    if (!words || a.f1 < 1 || a.C0 < a.f1 || (a.C > a.C0 && a.C0 < CT) || a.nk < 1 || a.nk > max_ksteps(a.parts) ||
        a.nk * a.chunks != a.nkt || a.nchunk < 1 || a.nset != a.groups * a.nchunk || a.nkt * KP < (a.fold ? (a.R + 1) / 2 - a.center : a.R) || a.tpg < 1 ||
        a.groups * a.tpg < a.ctiles || a.planes_per_sq < 1 || s.ntiles > 65535)
        return hipErrorInvalidValue;
    u32x4 *w = reinterpret_cast<u32x4 *>(words);
    const unsigned nb = (unsigned)std::min<long long>((long long)s.nplanes * a.ctiles, 8192);
    auto run = [&](auto kernel) {
        for (int c = 0; c < a.chunks; c += a.nchunk) {
            const dim3 grid(a.groups * std::min(a.nchunk, a.chunks - c), s.ntiles);
            kernel<<<grid, NT, 0, st>>>(a, s.tile0, s.plane0, s.nplanes, c, w);
        }
    };
    if (a.parts == 2) {
        adj_words_kernel<2><<<nb, 256, 0, st>>>(a, s.plane0, s.nplanes, w);
        a.nk == 1 ? run(adjoint_kernel<2, 1>) : a.nk == 2 ? run(adjoint_kernel<2, 2>) : a.nk == 3 ? run(adjoint_kernel<2, 3>)
            : a.nk == 4 ? run(adjoint_kernel<2, 4>) : run(adjoint_kernel<2, 5>);
    } else {
        adj_words_kernel<3><<<nb, 256, 0, st>>>(a, s.plane0, s.nplanes, w);
        a.nk == 1 ? run(adjoint_kernel<3, 1>) : a.nk == 2 ? run(adjoint_kernel<3, 2>) : run(adjoint_kernel<3, 3>);
    }
    return hipGetLastError();
}

// Runs of planes whose words fit ADJ_WORDS_MAX together (one plane at least), with
// their tiles, which are in plane order; 65,535 tiles a launch at most.
std::vector<AdjSpan> adjoint_spans(const AdjArgs &a, const int *tiles, int ntiles) {
    std::vector<AdjSpan> out;
    const long long cap = std::max<long long>(1, ADJ_WORDS_MAX / (16 * std::max<long long>(a.plane_words, 1)));
    for (int t = 0; t < ntiles; ++t) {
        const int pl = tiles[4 * t + 2];
        if (out.empty() || pl - out.back().plane0 >= cap || out.back().ntiles == 65535) out.push_back({pl, 1, t, 0});
        out.back().nplanes = pl - out.back().plane0 + 1;
        ++out.back().ntiles;
    }
    return out;
}

hipError_t launch_adjoint_finish(const AdjFinishArgs &a, hipStream_t st) {
    if (a.natoms <= 0) return hipSuccess;
    adjoint_finish_kernel<<<(a.natoms + 255) / 256, 256, 0, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_model_q(const QArgs &a, hipStream_t st) {
    if (a.g.P <= 0) return hipSuccess;
    model_q_kernel<<<(unsigned)((a.g.P + 255) / 256), 256, 0, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_chi2_resid(const double *icalc, const double *tgt, const double *wt, long long n, double *gi,
                             double *blocksum, int nblocks, hipStream_t st) {
    chi2_resid_kernel<<<nblocks, 256, 0, st>>>(icalc, tgt, wt, n, gi, blocksum);
    return hipGetLastError();
}

}  // namespace dc
