// dc_fold.h -- the phase GEMM on mirrored column pairs (gfx950).
//
// One side of the grid ("columns", the abscissa or the last axis) is a single
// uniform run of NB points, so its points come in pairs mirrored about the
// run's centre: with theta_n the per-atom step and phi_n the phase at the
// centre,
//     F(r, +j) = X + iY,  F(r, -j) = X - iY,
//     X = sum_n A(r, n) w_n cos(t_nj),  Y = sum_n A(r, n) w_n sin(t_nj),
//     A(r, n) = exp(2 pi i (phi_n + phi_row_n(r))),  t_nj = 2 pi (j theta_n + delta_n)
// (delta_n: half a step when NB is even).  cos and sin are real, so the pair
// costs 4 real multiply-accumulates per atom where the complex product of
// dc_gemm.hip takes 8 -- half the matrix work, and half the column operands.
// Same results, sum over atoms in another order.
//
// Every atom's column operand of a split scheme carries a scale r_n in
// [K, 1], and its A operand K / r_n: the product is K times the
// term for every atom, undone in the epilogue, while the roundings of the two
// operands differ from atom to atom (a rotation, as dc_gemm.hip uses, would
// mix the mirrored columns).  Without it atoms of equal phase, a crystal at
// its Bragg peaks, would round identically and add their errors coherently;
// the spread of the hi halves over the 32 products of an MFMA also keeps
// equal terms from driving the accumulator's last bit in one direction.  Both
// scales stay at or below 1: scaled past it, cosines just under 1 lose the
// bit that their binade gives them (BF16X3 error of F 1.2 to 1.3 times as
// large).  Row l of a 16-row group carries a further scale of its own: rows r
// and -r of a grid centred on the origin hold conjugate operands, whose equal
// roundings would add in sums over the grid (gradients of centred models:
// error 1.2 to 1.4 times as large).  The tables are rotated by +psi2 / -psi2 in their two factors, so
// the sin/cos polynomial differs per atom as well.
//
// Work split.  A work-group of 8 waves owns RT = 128 WR rows x 8 WC column
// pairs; wave w owns rows [16 WR w, 16 WR (w+1)) and every column, so its A
// operands are formed in the registers the MFMAs read them from: a lane's
// A fragment is 8 consecutive atoms of one row, the product of two table rows
// (TH[row / 16] * TL_d[row % 16], as in dc_gemm.hip).  Only the tables and
// the column operands (cos and sin interleaved: 8 pairs per 16-column MFMA
// tile) go through LDS.  A stage is 32 atoms, one K of
// v_mfma_f32_16x16x32; in stage s the waves build the tables of stage s+2,
// the columns of stage s+1 and run the MFMAs of stage s.  Waves 0..3 form
// their A operands before their MFMAs and waves 4..7 after (for the next
// stage), so of the two waves of a SIMD one generates while the other
// multiplies; the tables therefore live for three stages.
//
// FP32 operands are split into three BF16 parts, which hold all 24 bits, and
// multiplied in six products; what is left out (second times third parts and
// smaller) is below 2^-25 of a product, FP32's own rounding of it.  Six products on the BF16 units
// take 3/8 of the time of the FP32 ones (v_mfma_f32_16x16x4_f32 before: 0.62 ->
// 0.41 ms for 62,000 atoms x 33 x 65 x 65, now bound by the VALU work; error of F
// against FP64 4.2e-8 -> 3.1e-8 on a 4,000-atom line, 5.1e-8 -> 4.0e-8 there).
//
// Bound: half matrix cores, half the VALU work of forming operands, which
// overlaps with them only in part (256 x 176: matrix cores busy 42% of the time in
// FP16X3, 47% in BF16X3, 3.0 and 3.3 other VALU instructions per MFMA; FP32
// 128 x 96 37% and 7.3).  Measured against dc_gemm.hip:
// 256,000 atoms x 81 x 161 x 161, FP16X3 10.06 -> 6.75 ms (6.7 to 7.2 from box to
// box); 62,000 atoms x 33 x 65 x 65, FP32 1.38 -> 0.39 ms; an 8,000-atom
// 101^2 layer, FP32 174 -> 15 us (with slices cut to fill the device); a
// population of 96 (1.8M atoms, 256^2, damped) 2.66 -> 1.5 ms.
//
// Epilogue: an even lane holds X and its neighbour Y of the same pair, so
// one quad permute gives each lane one finished column.
#pragma once
#include "dc_gemm_dev.h"

namespace dc {

constexpr int FKS = 32;           // atoms per stage

template <int WR_, int WC_>
struct FoldCfg {
    static constexpr int WR = WR_, WC = WC_, NW = 8, NT = 64 * NW;
    static constexpr int RT = 16 * WR * NW;        // rows of the tile
    static constexpr int CT = 16 * WC;             // operand columns = output columns
    static constexpr int JT = 8 * WC;              // column pairs
    static constexpr int RH = RT / 16, CH = WC;    // 16-row groups, 8-pair groups
};

// Fold tiles (WR, WC), in the order of their tile indices.  The WC of one row
// block are close enough together that 25 pairs or more fill 77% of their
// tiles at least and 92% on the average (9 to 24 pairs: 82%); those of two row
// blocks start at 4, since few columns leave their row operands, formed anew
// for every tile of columns, too little to multiply with (49 pairs or more: 83%
// at least).  What a half-empty tile costs: 33 pairs in 48 instead of 40, 0.456
// -> 0.426 ms a call (62,000 atoms x 33 x 65 x 65, FP32); 101 in 128
// instead of 112, 0.474 -> 0.444 ms (GEMM of 32 lots, 804 rows, FP16X3).
#define DC_FOLD_TILES(X) \
    X(0, 2, 11) X(1, 1, 11) X(2, 2, 8) X(3, 1, 8) X(4, 2, 6) X(5, 1, 6) X(6, 2, 4) X(7, 1, 4) X(8, 1, 2) X(9, 2, 9) X(10, 1, 9) \
    X(11, 1, 5) X(12, 1, 3) X(13, 2, 7)
// FP32 holds FP64 sums beside its accumulators: 24 WR WC registers
constexpr bool fold_built(int scheme, int wr, int wc) {
    return split3(scheme) || (scheme == SCH_FP32 && wr == 1 && wc <= 6);
}

// Geometry of a folded launch: side A (rows, period PA), side B (NB points).
struct FoldGeom {
    int NA, PA, NB;
    int swap;            // side A from the records' column phases, side B from the row phases
    int sr, sc;          // output strides of a row / a column (one of them 1)
};

// Low tables: [atom pair q][row l] as float4 (two atoms), q stride padded by
// one so that a wave's stores of one row and loads of 16 rows are spread over
// the banks.  High tables: [group][atom].
struct alignas(16) FoldLow {
    float4 v[16 * 17];
};
template <class T>
struct alignas(16) FoldTables {
    FoldLow al[2];                          // side A, wrap state 0 / 1
    alignas(16) float2 ah[T::RH * FKS];
    alignas(16) float4 bl[16 * 9];          // side B, 8 pairs
    alignas(16) float2 bh[T::CH * FKS];
    alignas(16) float dmp[FKS];             // (B_n - the slice's reference) log2(e) (damped variant)
};
template <int SCHEME, class T>
struct alignas(16) FoldB {
    alignas(16) uint32_t hi[T::CT * 16];    // two FP16/BF16 atoms per word, pk_off
    alignas(16) uint32_t lo[T::CT * 16];
};
template <class T>
struct alignas(16) FoldB<SCH_FP32, T> {
    alignas(16) uint32_t p[3][T::CT * 16];  // three BF16 parts, pk_off
};
template <int SCHEME, class T>
struct alignas(16) FoldSmem {
    FoldB<SCHEME, T> b[2];
    FoldTables<T> t[3];
    int k16[T::RH], wpos[T::RH];
    float s_b[T::JT];
    float wmax[T::NW];
    float bmin[T::NW];                      // damped FP16: least B by wave, factors put back (damp_back2)
    alignas(16) float2 back_a[T::RT];       // and the scales of the row and the slice
    float2 back_b[T::JT];
    int item;
};

// K of the operand scales, and its reciprocal to 1e-12: a range of 64 steps of
// an FP16 hi half, of 20 of a BF16 one (over 8 steps the lo halves of the two
// operands, whose product is fixed, stay correlated: BF16X3 sums of equal
// terms came out 4.5e-6 low).
template <int SCHEME>
constexpr float fscale_k() {
    return f16ops(SCHEME) ? 0x1.f001f8p-1f : 0x1.d86bd4p-1f;
}
template <int SCHEME>
constexpr float fscale_undo() {
    return f16ops(SCHEME) ? 0x1.084104p+0f : 0x1.157284p+0f;
}
// Scale of row l of a group: frow_m(l % 4) * frow_j(l / 4), and the
// reciprocals of both (each product with its scale is 1 to 1e-11).
__device__ __forceinline__ float pick4(int k, float a, float b, float c, float d) {
    return k < 2 ? (k == 0 ? a : b) : (k == 2 ? c : d);
}
__device__ __forceinline__ float frow_m(int k) { return pick4(k, 1.0f, 0x1.eb736ep-1f, 0x1.f594e6p-1f, 0x1.e16a4ap-1f); }
__device__ __forceinline__ float frow_m_undo(int k) { return pick4(k, 1.0f, 0x1.0ab444p+0f, 0x1.055140p+0f, 0x1.104392p+0f); }
__device__ __forceinline__ float frow_j(int k) { return pick4(k, 1.0f, 0x1.f001f8p-1f, 0x1.fd5eb2p-1f, 0x1.f9781ap-1f); }
__device__ __forceinline__ float frow_j_undo(int k) { return pick4(k, 1.0f, 0x1.084104p+0f, 0x1.015264p+0f, 0x1.034ec0p+0f); }

// FP32: frame of the MFMA chain g (64 atoms) of a slice, a pseudo-random turn.
__device__ __forceinline__ uint64_t fold_frame(int slice, int g, uint32_t salt) {
    return dither_turn32((uint32_t)slice * 0x9E3779B9u + (uint32_t)g, salt);
}

__device__ __forceinline__ float2 cis_fine(uint64_t ph) {
    float c, s;
    sincos_turn_fine(phase_top(ph), c, s);
    return make_float2(c, s);
}
template <int SCHEME>
__device__ __forceinline__ float2 fold_cis(uint64_t ph) {
    if constexpr (SCHEME == SCH_FP32)
        return cis_fine(ph);
    else
        return cis(ph);
}

template <int SCHEME, class T>
__device__ __forceinline__ void fold_tables(FoldTables<T> &tb, const int *__restrict__ k16s, uint64_t p0, uint64_t sA,
                                            uint64_t s1A, uint64_t sB, float w, float pad, bool live, int a0, int hi0,
                                            const FoldGeom &fg, int pair0, int wave, int lane, uint32_t hash,
                                            uint64_t frame, float bref) {
    const int a16 = lane & 15, m = lane >> 4, a = 16 * (wave & 1) + a16;
    const uint64_t psi2 = (uint64_t)hash * 0xD6E8FEB86659FD93ull;
    const uint64_t wrp = s1A - (uint64_t)fg.PA * sA;
    // Who builds what.  Evaluations of sin/cos a lane, by wave pair: FP32 4 | 4 | 3
    // | 3 (128 x 96), split schemes 3 and their exchange | 5 | 3 | 3 (256 x 176).
    // The column operands go to the first waves in FP32 and to the last ones in
    // the split schemes (fold_b).  Measured, both orders of both: FP32 65^3 0.412 ms, with the split
    // schemes' order 0.47, with both row tables on the first pair 0.42;
    // FP16X3 161^3 (on the fastest box) 6.1 ms, with the columns on the first waves 6.5, with
    // the high groups spread as in FP32 6.5.
    constexpr bool F32 = SCHEME == SCH_FP32;
    if (wave == 0 || wave == 1) {
        if (m == 0) tb.dmp[a] = live && w != 0.0f ? (pad - bref) * 1.4426950408889634f : 0.0f;
    }
    if (wave < (F32 ? 4 : 2)) {
        float2 *t0 = reinterpret_cast<float2 *>(tb.al[0].v) + (a & 1);
        float2 *t1 = reinterpret_cast<float2 *>(tb.al[1].v) + (a & 1);
        const int q = 17 * (a >> 1);
        if constexpr (F32) {
            const bool wrapped = wave >= 2;
            if (wrapped && fg.PA >= fg.NA) return;
            float2 *t = wrapped ? t1 : t0;
            const uint64_t base = psi2 + (wrapped ? wrp : 0ull);
#pragma unroll
            for (int j = 0; j < 4; ++j) t[2 * (q + m + 4 * j)] = fold_cis<SCHEME>((uint64_t)(m + 4 * j) * sA + base);
        } else {
            // helper m evaluates fold_cis<SCHEME>(m s + psi2), fold_cis<SCHEME>(4m s) and fold_cis<SCHEME>(4m s + w); the
            // four helpers of an atom exchange the last two (see dc_gemm.hip)
            float2 base = fold_cis<SCHEME>((uint64_t)m * sA + psi2);
            const uint64_t hs = (uint64_t)(4 * m) * sA;
            float2 g0 = fold_cis<SCHEME>(hs), g1 = fold_cis<SCHEME>(hs + wrp);
            const float fm = frow_m(m), fj = frow_j(m);
            base = make_float2(base.x * fm, base.y * fm);
            g0 = make_float2(g0.x * fj, g0.y * fj);
            g1 = make_float2(g1.x * fj, g1.y * fj);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int src = a16 + 16 * j;
                const float2 h0 = make_float2(__shfl(g0.x, src), __shfl(g0.y, src));
                const float2 h1 = make_float2(__shfl(g1.x, src), __shfl(g1.y, src));
                t0[2 * (q + m + 4 * j)] = cmul(base, h0);
                t1[2 * (q + m + 4 * j)] = cmul(base, h1);
            }
        }
        return;
    }
    const uint64_t half = (fg.NB & 1) ? 0ull : sB >> 1;
    const int first = F32 ? 2 : 1;             // the wave pair with the low table of side B
    if ((wave >> 1) == first) {
        float2 *t = reinterpret_cast<float2 *>(tb.bl) + (a & 1);
        const int q = 9 * (a >> 1);
        t[2 * (q + m)] = fold_cis<SCHEME>((uint64_t)m * sB + half + psi2);
        t[2 * (q + m + 4)] = fold_cis<SCHEME>((uint64_t)(m + 4) * sB + half + psi2);
    }
    const float r = SCHEME == SCH_FP32 ? 1.0f : 1.0f - (1.0f - fscale_k<SCHEME>()) * ((float)(hash & 0xFFFFFFu) * 0x1p-24f);
    const float ampA = SCHEME == SCH_FP32 ? 1.0f : fscale_k<SCHEME>() / r;
    const float ampB = live ? w * r : 0.0f;
    const uint64_t pa = p0 + (uint64_t)(fg.NB / 2) * sB - half + (uint64_t)a0 * sA + (uint64_t)hi0 * s1A - psi2 + frame;
    // FP32: that pair takes one high group a lane, the last one the rest
    const int step = !F32 ? 12 : (wave >> 1) == first ? T::RH + T::CH : 4;
    for (int q = ((wave >> 1) - first) * 4 + m; q < T::RH + T::CH; q += step) {
        const bool isb = q >= T::RH;
        const int h = isb ? q - T::RH : q;
        const uint64_t ph = isb ? (uint64_t)(pair0 + 8 * h) * sB - psi2
                                : pa + (uint64_t)(16 * h) * sA + (uint64_t)(uint32_t)k16s[h] * wrp;
        const float2 v = fold_cis<SCHEME>(ph);
        const float amp = isb ? ampB : ampA;
        (isb ? tb.bh : tb.ah)[h * FKS + a] = make_float2(v.x * amp, v.y * amp);
    }
}

// 8 values (atoms 8g .. 8g+7 of one row or column) as packed hi / lo halves
template <int SCHEME>
__device__ __forceinline__ void split8(const float (&x)[8], u32x4 &hi, u32x4 &lo) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        hi[q] = pack2<SCHEME>(x[2 * q], x[2 * q + 1]);
        if constexpr (f16ops(SCHEME)) {
            lo[q] = lo_halves_f16(hi[q], x[2 * q], x[2 * q + 1]);
        } else {
            const f32x2 h = unpack2<SCHEME>(hi[q]);
            lo[q] = pack2<SCHEME>(x[2 * q] - h.x, x[2 * q + 1] - h.y);
        }
    }
}

// FP32 values as three BF16 parts whose sum they are, exactly.
__device__ __forceinline__ void split8_3(const float (&x)[8], u32x4 (&p)[3]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float a = x[2 * q], b = x[2 * q + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            p[k][q] = pack2<SCH_BF16X3>(a, b);
            const f32x2 h = unpack2<SCH_BF16X3>(p[k][q]);
            a -= h.x;
            b -= h.y;
        }
    }
}

// Elements of 8 atoms: products of two rows of tables (4 float4 each).
template <bool DAMP>
__device__ __forceinline__ void elems8(const float4 *tl, int tstep, const float4 *th, const float *dmp, float sv,
                                       float (&re)[8], float (&im)[8]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 x = tl[q * tstep], y = th[q];
        const float2 u = cmul(make_float2(x.x, x.y), make_float2(y.x, y.y));
        const float2 v = cmul(make_float2(x.z, x.w), make_float2(y.z, y.w));
        re[2 * q] = u.x;
        im[2 * q] = u.y;
        re[2 * q + 1] = v.x;
        im[2 * q + 1] = v.y;
    }
    if constexpr (DAMP) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float f = __builtin_amdgcn_exp2f(-dmp[k] * sv);
            re[k] *= f;
            im[k] *= f;
        }
    }
}

// A operands of one stage, in the MFMA's own layout: lane (li = row, lg) holds
// atoms 8 lg .. 8 lg + 7.
template <int SCHEME, int WR>
struct FoldA {
    u32x4 rh[WR], rl[WR], ih[WR], il[WR];
};
template <int WR>
struct FoldA<SCH_FP32, WR> {
    u32x4 re[WR][3], im[WR][3];
};

template <int SCHEME, class T, bool DAMP>
__device__ __forceinline__ void fold_a(FoldA<SCHEME, T::WR> &A, const FoldTables<T> &tb, const int (&dsel)[T::WR],
                                       const float (&sv)[T::WR], int wave, int li, int lg) {
#pragma unroll
    for (int i = 0; i < T::WR; ++i) {
        const float4 *tl = tb.al[0].v + dsel[i] + 17 * 4 * lg + li;
        const float4 *th = reinterpret_cast<const float4 *>(tb.ah + (wave * T::WR + i) * FKS + 8 * lg);
        float re[8], im[8];
        elems8<DAMP>(tl, 17, th, tb.dmp + 8 * lg, sv[i], re, im);
        if constexpr (SCHEME == SCH_FP32) {
            split8_3(re, A.re[i]);
            split8_3(im, A.im[i]);
        } else {
            split8<SCHEME>(re, A.rh[i], A.rl[i]);
            split8<SCHEME>(im, A.ih[i], A.il[i]);
        }
    }
}

// Column operands of one stage: half a wave forms 8 pairs x 32 atoms; the
// two halves store cos and sin in opposite order so that together they fill
// both bank halves.
template <int SCHEME, class T, bool DAMP>
__device__ __forceinline__ void fold_b(FoldB<SCHEME, T> &bb, const FoldTables<T> &tb, const float *__restrict__ s_b,
                                       int wave, int lane) {
    const int l = lane & 7, g = (lane >> 3) & 3, hs = lane >> 5;
    for (int jp = SCHEME == SCH_FP32 ? wave : T::NW - 1 - wave; jp < (T::CH + 1) / 2; jp += T::NW) {
        const int h = 2 * jp + hs;
        if (h < T::CH) {
            float re[8], im[8];
            const float sv = DAMP ? s_b[8 * h + l] : 0.0f;
            elems8<DAMP>(tb.bl + 9 * 4 * g + l, 9, reinterpret_cast<const float4 *>(tb.bh + h * FKS + 8 * g),
                         tb.dmp + 8 * g, sv, re, im);
            const int c0 = 16 * h + 2 * l;
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                const bool sn = (o ^ hs) != 0;
                float x[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) x[k] = sn ? im[k] : re[k];
                const int col = c0 + (sn ? 1 : 0);
                if constexpr (SCHEME == SCH_FP32) {
                    u32x4 p[3];
                    split8_3(x, p);
#pragma unroll
                    for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4 *>(&bb.p[q][pk_off(col, g)]) = p[q];
                } else {
                    u32x4 hi, lo;
                    split8<SCHEME>(x, hi, lo);
                    *reinterpret_cast<u32x4 *>(&bb.hi[pk_off(col, g)]) = hi;
                    *reinterpret_cast<u32x4 *>(&bb.lo[pk_off(col, g)]) = lo;
                }
            }
        }
    }
}

template <int SCHEME>
__device__ __forceinline__ f32x4 mfma_k32(u32x4 a, u32x4 b, f32x4 c) {
    if constexpr (f16ops(SCHEME))
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// MFMAs of one stage; the columns of tile j+1 are read while tile j multiplies.
template <int SCHEME, class T>
__device__ __forceinline__ void fold_mfma(const FoldB<SCHEME, T> &bb, const FoldA<SCHEME, T::WR> &A,
                                          f32x4 (&accR)[T::WR][T::WC], f32x4 (&accI)[T::WR][T::WC], int li, int lg) {
    if constexpr (SCHEME == SCH_FP32) {
        u32x4 y[3], n[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) y[q] = *reinterpret_cast<const u32x4 *>(&bb.p[q][pk_off(li, lg)]);
#pragma unroll
        for (int j = 0; j < T::WC; ++j) {
            if (j + 1 < T::WC)
#pragma unroll
                for (int q = 0; q < 3; ++q) n[q] = *reinterpret_cast<const u32x4 *>(&bb.p[q][pk_off(16 * (j + 1) + li, lg)]);
            __builtin_amdgcn_sched_barrier(0);
            // the small products first: those of the second and third parts are below FP32's rounding
#pragma unroll
            for (int s = 2; s >= 0; --s)
#pragma unroll
                for (int q = s; q >= 0; --q)
#pragma unroll
                    for (int i = 0; i < T::WR; ++i) {
                        accR[i][j] = mfma_k32<SCH_BF16X3>(A.re[i][s - q], y[q], accR[i][j]);
                        accI[i][j] = mfma_k32<SCH_BF16X3>(A.im[i][s - q], y[q], accI[i][j]);
                    }
#pragma unroll
            for (int q = 0; q < 3; ++q) y[q] = n[q];
        }
    } else {
        u32x4 yh = *reinterpret_cast<const u32x4 *>(&bb.hi[pk_off(li, lg)]);
        u32x4 yl = *reinterpret_cast<const u32x4 *>(&bb.lo[pk_off(li, lg)]);
#pragma unroll
        for (int j = 0; j < T::WC; ++j) {
            const int on = pk_off(16 * (j + 1 < T::WC ? j + 1 : j) + li, lg);
            u32x4 nh = yh, nl = yl;
            if (j + 1 < T::WC) {
                nh = *reinterpret_cast<const u32x4 *>(&bb.hi[on]);
                nl = *reinterpret_cast<const u32x4 *>(&bb.lo[on]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < T::WR; ++i) {
                accR[i][j] = mfma_k32<SCHEME>(A.rh[i], yh, accR[i][j]);
                accI[i][j] = mfma_k32<SCHEME>(A.ih[i], yh, accI[i][j]);
            }
#pragma unroll
            for (int i = 0; i < T::WR; ++i) {
                accR[i][j] = mfma_k32<SCHEME>(A.rh[i], yl, accR[i][j]);
                accI[i][j] = mfma_k32<SCHEME>(A.ih[i], yl, accI[i][j]);
            }
#pragma unroll
            for (int i = 0; i < T::WR; ++i) {
                accR[i][j] = mfma_k32<SCHEME>(A.rl[i], yh, accR[i][j]);
                accI[i][j] = mfma_k32<SCHEME>(A.il[i], yh, accI[i][j]);
            }
            yh = nh;
            yl = nl;
        }
    }
}

// value of the lane's neighbour (lane ^ 1)
__device__ __forceinline__ float pair_swap(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, true));
}

template <int SCHEME, class T, bool DAMP>
__global__ void __launch_bounds__(T::NT)
fold_gemm_kernel(const AtomRec *__restrict__ rec, const int *__restrict__ slice_beg, float2 *__restrict__ partial,
                 const float *__restrict__ sq, const int *__restrict__ slice_sq, GemmGeom g, FoldGeom fg, int slice0,
                 int nitems) {
    __shared__ FoldSmem<SCHEME, T> sm;
    constexpr int WR = T::WR, WC = T::WC;
    const int J = (fg.NB + 1) / 2;
    const int nct = (J + T::JT - 1) / T::JT, nrt = (fg.NA + T::RT - 1) / T::RT;
    const bool padh = !DAMP && g.pad_hash != 0;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
    // work items and their order: see dc_gemm.hip
    int item0 = blockIdx.x;
    if (!g.queue && !g.order && (int)gridDim.x == nitems) {
        constexpr int NX = 8;
        const int q = nitems / NX, r = nitems % NX, x = blockIdx.x % NX, k = blockIdx.x / NX;
        item0 = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + k;
    }
    auto next_item = [&](int cur) -> int {
        if (!g.queue) return cur + (int)gridDim.x;
        __syncthreads();
        if (threadIdx.x == 0) sm.item = atomicAdd(g.queue, 1);
        __syncthreads();
        return sm.item;
    };
    for (int item = g.queue ? next_item(0) : item0; item < nitems; item = next_item(item)) {
        __syncthreads();   // the previous item's tables and bookkeeping are done with
        const int si = item / (nct * nrt);
        const int slice = slice0 + (g.order ? g.order[si] : si);
        const int kbeg = slice_beg[slice], kend = slice_beg[slice + 1];
        const int row0 = ((item / nct) % nrt) * T::RT, pair0 = (item % nct) * T::JT;
        const int wr0 = row0 + 16 * WR * wave;
        const bool active = wr0 < fg.NA;                 // this wave's rows touch the grid
        const int a0 = row0 % fg.PA, hi0 = row0 / fg.PA;
        for (int h = threadIdx.x; h < T::RH; h += T::NT) {
            const int x = a0 + 16 * h;
            sm.k16[h] = x / fg.PA;
            sm.wpos[h] = fg.PA - (x % fg.PA);
        }
        float sv[WR];
#pragma unroll
        for (int i = 0; i < WR; ++i) sv[i] = 0.0f;
        constexpr bool SCALED = DAMP && f16ops(SCHEME);   // damp_back
        float bref = 0.0f;
        if constexpr (DAMP) {
            const float *sqs = sq + (slice_sq ? slice_sq[slice] : 0);
            const float *sa = sqs + (fg.swap ? g.R : 0), *sb = sqs + (fg.swap ? 0 : g.R);
#pragma unroll
            for (int i = 0; i < WR; ++i) {
                const int r = wr0 + 16 * i + li;
                sv[i] = r < fg.NA ? sa[r] : 0.0f;
            }
            for (int x = threadIdx.x; x < T::JT; x += T::NT)
                sm.s_b[x] = pair0 + x < J ? sb[fg.NB / 2 + pair0 + x] : 0.0f;
        }

        f32x4 accR[WR][WC], accI[WR][WC];
#pragma unroll
        for (int i = 0; i < WR; ++i)
#pragma unroll
            for (int j = 0; j < WC; ++j) {
                accR[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                accI[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        // FP32: the MFMA rounds its accumulator after every product, so chains
        // of 64 atoms are added into FP64 sums.  Equal terms would round the
        // same way in every chain: the A operands of a chain carry a turn of
        // its own (fold_frame), undone before it is added (64,000 atoms, 65^3:
        // error of I 6.5e-8 with one frame for all).
        constexpr bool TWO = SCHEME == SCH_FP32;
        double sumR[TWO ? WR : 1][TWO ? WC : 1][4], sumI[TWO ? WR : 1][TWO ? WC : 1][4];
        if constexpr (TWO) {
#pragma unroll
            for (int i = 0; i < WR; ++i)
#pragma unroll
                for (int j = 0; j < WC; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) sumR[i][j][v] = sumI[i][j][v] = 0.0;
        }

        const int nst = (kend - kbeg + FKS - 1) / FKS;
        const int at = 16 * (wave & 1) + (lane & 15);
        auto fetch = [&](int st) {
            const int k = kbeg + st * FKS + at;
            return rec[k < kend ? k : kend - 1];
        };
        auto tables = [&](int st, const AtomRec &r) {
            const int k = kbeg + st * FKS + at;
            const uint32_t hash = g.dither == 0 ? 0u : padh ? __builtin_bit_cast(uint32_t, r.pad) : dither_hash32((uint32_t)k, g.dither);
            const uint64_t frame = TWO ? fold_frame(slice, st >> 1, g.dither) : 0;
            fold_tables<SCHEME, T>(sm.t[st % 3], sm.k16, r.p0, fg.swap ? r.ca : r.ra, fg.swap ? r.ca1 : r.ra1,
                                   fg.swap ? r.ra : r.ca, r.w * sm.wmax[0], r.pad, k < kend, a0, hi0, fg, pair0, wave, lane,
                                   hash, frame, bref);
        };
        const AtomRec r0 = fetch(0), r1 = fetch(nst > 1 ? 1 : 0);
        AtomRec rn = fetch(nst > 2 ? 2 : 0);
        // FP16 schemes: amplitudes scaled by a power of two, undone in the epilogue
        float wscale = 1.0f, wunscale = 1.0f;
        if constexpr (f16ops(SCHEME)) {
            float m = 0.0f, b = NO_B;
            for (int k = kbeg + (int)threadIdx.x; k < kend; k += T::NT) {
                const float wk = rec[k].w;
                m = fmaxf(m, fabsf(wk));
                if constexpr (SCALED) b = wk != 0.0f ? fminf(b, rec[k].pad) : b;
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                m = fmaxf(m, __shfl_xor(m, o));
                if constexpr (SCALED) b = fminf(b, __shfl_xor(b, o));
            }
            if (lane == 0) {
                sm.wmax[wave] = m;
                if constexpr (SCALED) sm.bmin[wave] = b;
            }
            __syncthreads();
            m = 0.0f;
#pragma unroll
            for (int w = 0; w < T::NW; ++w) m = fmaxf(m, sm.wmax[w]);
            if constexpr (SCALED) {
#pragma unroll
                for (int w = 0; w < T::NW; ++w) b = fminf(b, sm.bmin[w]);
                bref = damp_ref(b);
            }
            if (m > 0.0f && m <= 3.0e38f) {
                int e = 0;
                (void)frexpf(m, &e);
                wscale = ldexpf(1.0f, -e);
                wunscale = ldexpf(1.0f, e);
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) sm.wmax[0] = wscale;
        __syncthreads();
        int dsel[WR];
#pragma unroll
        for (int i = 0; i < WR; ++i)
            dsel[i] = fg.PA < fg.NA && li >= sm.wpos[wave * WR + i] ? (int)(sizeof(FoldLow) / sizeof(float4)) : 0;
        FoldA<SCHEME, WR> A{};
        const bool mfma_first = ((wave >> 2) & 1) != 0;
        if constexpr (SCALED) {
            // what the floats of sq leave of s^2 lies behind them
            const float *lo = sq + (slice_sq ? slice_sq[slice] : 0) + g.R + g.C;
            const float *la = lo + (fg.swap ? g.R : 0), *lb = lo + (fg.swap ? 0 : g.R) + fg.NB / 2 + pair0;
#pragma unroll
            for (int i = 0; i < WR; ++i) {
                const int r = wr0 + 16 * i + li;
                if (lg == 0)
                    sm.back_a[16 * (wave * WR + i) + li] =
                        damp_back2(bref, sv[i], r < fg.NA ? la[r] : 0.0f,
                                   (double)frow_j_undo(li >> 2) * frow_m_undo(li & 3) * fscale_undo<SCHEME>() * wunscale);
            }
            for (int x = threadIdx.x; x < T::JT; x += T::NT)
                sm.back_b[x] = damp_back2(bref, sm.s_b[x], pair0 + x < J ? lb[x] : 0.0f, 1.0);
        }
        tables(0, r0);
        __syncthreads();
        if (nst > 1) tables(1, r1);
        fold_b<SCHEME, T, DAMP>(sm.b[0], sm.t[0], sm.s_b, wave, lane);
        if (mfma_first) fold_a<SCHEME, T, DAMP>(A, sm.t[0], dsel, sv, wave, li, lg);
        __syncthreads();
        int tc = 0;   // s % 3
        for (int s = 0; s < nst; ++s) {
            const int tn = tc == 2 ? 0 : tc + 1;
            auto generate = [&](const FoldTables<T> &ta, bool form_a) {
                if (s + 2 < nst) tables(s + 2, rn);
                if (s + 1 < nst) fold_b<SCHEME, T, DAMP>(sm.b[(s + 1) & 1], sm.t[tn], sm.s_b, wave, lane);
                if (form_a) fold_a<SCHEME, T, DAMP>(A, ta, dsel, sv, wave, li, lg);
            };
            if (!mfma_first) generate(sm.t[tc], true);
            __builtin_amdgcn_s_setprio(1);
            fold_mfma<SCHEME, T>(sm.b[s & 1], A, accR, accI, li, lg);
            __builtin_amdgcn_s_setprio(0);
            if (mfma_first) generate(sm.t[tn], s + 1 < nst);
            if constexpr (TWO) {
                if ((s & 1) || s + 1 == nst) {
                    const float2 back = cis_fine(0 - fold_frame(slice, s >> 1, g.dither));
#pragma unroll
                    for (int i = 0; i < WR; ++i)
#pragma unroll
                        for (int j = 0; j < WC; ++j) {
#pragma unroll
                            for (int v = 0; v < 4; ++v) {
                                const float xr = accR[i][j][v], xi = accI[i][j][v];
                                sumR[i][j][v] += (double)__builtin_fmaf(back.x, xr, -back.y * xi);
                                sumI[i][j][v] += (double)__builtin_fmaf(back.x, xi, back.y * xr);
                            }
                            accR[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                            accI[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                        }
                }
            }
            rn = fetch(s + 3 < nst ? s + 3 : 0);
            __syncthreads();
            tc = tn;
        }
        if constexpr (TWO) {
#pragma unroll
            for (int i = 0; i < WR; ++i)
#pragma unroll
                for (int j = 0; j < WC; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        accR[i][j][v] = (float)sumR[i][j][v];
                        accI[i][j][v] = (float)sumI[i][j][v];
                    }
        }

        // lane li of a 16-column tile holds operand column li: cos (even) or
        // sin (odd) of pair li / 2, rows 4 lg + v; even lanes finish the
        // column right of the centre, odd lanes its mirror image
        float2 *out = partial + (long long)(slice - slice0) * g.P;
        const bool odd = (li & 1) != 0;
        // row 4 lg + v of a group: scales frow_m(v) frow_j(lg)
        const float undo = SCHEME == SCH_FP32 ? 1.0f : frow_j_undo(lg), last = SCHEME == SCH_FP32 ? 1.0f : wunscale * fscale_undo<SCHEME>();
        const bool wide = fg.sr == 1 && (fg.sc & 1) == 0;
        if (active) {
#pragma unroll
            for (int i = 0; i < WR; ++i) {
                float2 backa[4];
                if constexpr (SCALED)
#pragma unroll
                    for (int v = 0; v < 4; ++v) backa[v] = sm.back_a[16 * (wave * WR + i) + 4 * lg + v];
#pragma unroll
                for (int j = 0; j < WC; ++j) {
                    const int pr = pair0 + 8 * j + (li >> 1);
                    float2 f[4];
                    const float2 backb = SCALED ? sm.back_b[8 * j + (li >> 1)] : make_float2(1.0f, 0.0f);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float xr = accR[i][j][v], xi = accI[i][j][v];
                        const float yr = pair_swap(xr), yi = pair_swap(xi);
                        const float re = odd ? yr + xi : xr - yi, im = odd ? yi - xr : xi + yr;
                        if constexpr (SCHEME == SCH_FP32) {
                            f[v] = make_float2(re, im);
                        } else if constexpr (SCALED) {
                            const float2 b = mul2(backa[v], backb);
                            f[v] = make_float2(__builtin_fmaf(re, b.x, re * b.y), __builtin_fmaf(im, b.x, im * b.y));
                        } else {
                            const float um = frow_m_undo(v);
                            f[v] = make_float2(re * undo * um * last, im * undo * um * last);
                        }
                    }
                    // odd NB: pair 0 is the centre column, stored by the even lane
                    if (pr >= J || (odd && pr == 0 && (fg.NB & 1))) continue;
                    const int col = odd ? (fg.NB - 1) / 2 - pr : fg.NB / 2 + pr;
                    const int r4 = wr0 + 16 * i + 4 * lg;
                    float2 *p = out + (long long)r4 * fg.sr + (long long)col * fg.sc;
                    if (wide && r4 + 3 < fg.NA) {
                        reinterpret_cast<float4 *>(p)[0] = make_float4(f[0].x, f[0].y, f[1].x, f[1].y);
                        reinterpret_cast<float4 *>(p)[1] = make_float4(f[2].x, f[2].y, f[3].x, f[3].y);
                    } else {
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            if (r4 + v < fg.NA) p[(long long)v * fg.sr] = f[v];
                    }
                }
            }
        }
    }
}

template <int SCHEME, class T>
static hipError_t fold_launch(const AtomRec *rec, const int *slice_beg, float2 *partial, const float *sq,
                              const int *slice_sq, const GemmGeom &g, const FoldGeom &fg, int slice0, int nslice, int nwg,
                              hipStream_t st) {
    const int J = (fg.NB + 1) / 2;
    const long long items = (long long)((J + T::JT - 1) / T::JT) * ((fg.NA + T::RT - 1) / T::RT) * nslice;
    const int grid = (int)(nwg > 0 && nwg < items ? nwg : items);
    if (sq)
        fold_gemm_kernel<SCHEME, T, true><<<grid, dim3(T::NT), 0, st>>>(rec, slice_beg, partial, sq, slice_sq, g, fg, slice0, (int)items);
    else
        fold_gemm_kernel<SCHEME, T, false><<<grid, dim3(T::NT), 0, st>>>(rec, slice_beg, partial, sq, slice_sq, g, fg, slice0, (int)items);
    return hipGetLastError();
}

// Launch of tile t of DC_FOLD_TILES.
template <int SCHEME>
static hipError_t fold_dispatch(int t, const AtomRec *rec, const int *slice_beg, float2 *partial, const float *sq,
                                const int *slice_sq, const GemmGeom &g, const FoldGeom &fg, int slice0, int nslice, int nwg,
                                hipStream_t st) {
    switch (t) {
#define X(i, wr, wc)                                                                                                    \
    case i:                                                                                                             \
        if constexpr (fold_built(SCHEME, wr, wc))                                                                       \
            return fold_launch<SCHEME, FoldCfg<wr, wc>>(rec, slice_beg, partial, sq, slice_sq, g, fg, slice0, nslice, nwg, st); \
        else                                                                                                            \
            return hipErrorInvalidValue;
        DC_FOLD_TILES(X)
#undef X
    default: return hipErrorInvalidValue;
    }
}

}  // namespace dc
