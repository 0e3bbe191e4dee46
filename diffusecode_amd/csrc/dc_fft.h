// dc_fft.h -- FP64 transforms of many lines, a few lines per work-group in LDS.
//
// A work-group holds LINES lines of n points and runs the whole transform of
// them between one read and one write of global memory, so that what comes
// before and after a transform (index maps, spectra, pruning, a second
// transform of the same lines) costs no pass of its own.  Element i of line l
// sits at LDS position i * LINES + l: consecutive lanes hold the lines of one element, so
// every LDS access is of whole 128-byte rows whatever the radix, and global
// accesses of strided axes take 128 bytes at a time.
//
// Lengths of grids are not ours to choose: primes up to 23 (161 = 7 x 23) are
// butterflies in registers, one larger prime up to FFT_MAXP a direct sum over LDS
// (P multiply-adds a point: at P = 157 half the time of a convolution of twice
// the length).  Self-sorting radix passes in place: each thread
// reads its butterflies, the work-group synchronises, and they are written
// to their places (Stockham's ordering); odd radices fold x_j +- x_{P-j}, a
// quarter of the plain sum's products, with their roots in scalar registers
// (read from the twiddle table inside each pass: as literals the compiler
// holds those of every radix at once).  The transform is forward; the backward one
// swaps real and imaginary parts at both ends.
//
// Bound: memory, 16 bytes a point each way (26 us a pass of 161^3 points at the
// rate of a copy), and the latency of the passes in LDS, which the work-groups
// of a CU cover for each other: 80 registers, 6 waves a SIMD (4 where a radix
// above 9 needs 128: one wave of four runs the 23-point butterflies of 8
// lines).  Measured 33 to 47 us; the vendor library's 161-point transforms are
// convolutions of length 320 or more with a transpose between axes, 121 us.
#pragma once
#include "dc_internal.h"

namespace dc {

constexpr int FFT_LINES = 8;
constexpr int FFT_MAXN = 600;          // 86 KB of LDS
constexpr int FFT_COMMON = 512;        // longer lengths, and radices above 9, take the kernels with more registers
constexpr int FFT_MAXPASS = 10;
constexpr int FFT_MAXP = 199;          // largest prime factor
constexpr int FFT_KB = 6;              // outputs (and mirrors) a thread of the direct sum at most

struct FftLen {
    int n, npass;
    int kind;                          // kernel: 0, 1 (longer than FFT_COMMON or a radix above 9), 2 (a direct sum)
    int radix[FFT_MAXPASS];
    uint32_t magic[FFT_MAXPASS];       // ceil(2^32 / Ns), Ns the product of the radices before (Ns > 1)
    const double2 *tw;                 // exp(-2 pi i k / n), on the device
};

// Threads of a work-group: 5 to 10 points each.
constexpr int FFT_SMALL = 256;         // lengths of 256 threads
inline int fft_threads(const FftLen &f) { return f.n <= FFT_SMALL ? 256 : 512; }
// Outputs a thread of the direct sum takes: of nb sums over P values, (P + 1) / 2
// outputs with their mirrors each, on NT / FFT_LINES threads a line.
__host__ __device__ inline int fft_direct_kb(int p, int nb, int nt) {
    const int h = (p + 1) / 2, slots = nt / FFT_LINES;
    for (int kb = 1; kb <= FFT_KB; ++kb)
        if (nb * ((h + kb - 1) / kb) <= slots) return kb;
    return 0;
}

// Radices of a length; false if it has a larger prime factor or is too long.
inline bool fft_length(long long n, FftLen &f) {
    f = FftLen{};
    if (n < 2 || n > FFT_MAXN) return false;
    f.n = (int)n;
    f.kind = n > FFT_COMMON;
    long long ns = 1;
    auto take = [&](int p) {
        if (f.npass == FFT_MAXPASS) return false;
        f.kind = std::max(f.kind, p > 23 ? 2 : p > 9 ? 1 : 0);
        f.radix[f.npass] = p;
        f.magic[f.npass++] = ns > 1 ? (uint32_t)((0x100000000ull + ns - 1) / ns) : 0u;
        ns *= p;
        n /= p;
        return true;
    };
    long long big = n;                 // the factor of primes above 23
    for (int p : {2, 3, 5, 7, 11, 13, 17, 19, 23})
        while (big % p == 0) big /= p;
    if (big > 1) {                     // below 29^2, so a prime
        if (big > FFT_MAXP || big >= 29 * 29 || !fft_direct_kb((int)big, (int)(n / big), fft_threads(f)) || !take((int)big)) return false;
    }
    for (int p : {23, 19, 17, 13, 11, 9, 8, 7, 5, 4, 3, 2})
        while (n % p == 0)
            if (!take(p)) return false;
    return n == 1;
}
inline size_t fft_lds(const FftLen &f) { return sizeof(double2) * (size_t)f.n * (FFT_LINES + 1); }

__device__ __forceinline__ double2 operator+(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 operator-(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 zmul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ double2 mul_mi(double2 a) { return make_double2(a.y, -a.x); }   // -i a

// Forward DFT of P values, in two halves: dft_begin leaves in v the sums that
// dft_out makes output r of (so that outputs need not be held with the
// inputs: 23 values and their 22 sums are 180 registers).
template <int P>
__device__ __forceinline__ void dft_begin(double2 (&v)[P]) {
    if constexpr (P == 2) {
        const double2 a = v[0] + v[1], b = v[0] - v[1];
        v[0] = a;
        v[1] = b;
    } else if constexpr (P == 4) {
        const double2 a = v[0] + v[2], b = v[0] - v[2], c = v[1] + v[3], d = mul_mi(v[1] - v[3]);
        v[0] = a + c;
        v[1] = b + d;
        v[2] = a - c;
        v[3] = b - d;
    } else if constexpr (P == 8) {
        double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        dft_begin<4>(e);
        dft_begin<4>(o);
        const double h = 0.70710678118654752440;
        const double2 o1 = make_double2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
        const double2 o2 = mul_mi(o[2]);
        const double2 o3 = make_double2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));
        v[0] = e[0] + o[0];
        v[4] = e[0] - o[0];
        v[1] = e[1] + o1;
        v[5] = e[1] - o1;
        v[2] = e[2] + o2;
        v[6] = e[2] - o2;
        v[3] = e[3] + o3;
        v[7] = e[3] - o3;
    } else {
        static_assert(P & 1, "radix");
#pragma unroll
        for (int j = 1; j <= (P - 1) / 2; ++j) {
            const double2 t = v[j] + v[P - j], d = v[j] - v[P - j];
            v[j] = t;
            v[P - j] = d;
        }
    }
}
// Outputs in the order that write(r, value) takes them.
typedef const __attribute__((address_space(4))) double *RootPtr;   // scalar loads
template <int P>
struct DftRoots {
    static constexpr int H = P & 1 ? (P - 1) / 2 : 1;
    double c[H], s[H];
    __device__ __forceinline__ DftRoots(const double2 *tw, int n) {
        const RootPtr t = (RootPtr)(uintptr_t)tw;
        const int q = __builtin_amdgcn_readfirstlane(n / P);
        if constexpr (P & 1)
#pragma unroll
            for (int m = 0; m < H; ++m) {
                c[m] = t[2 * (m + 1) * q];
                s[m] = -t[2 * (m + 1) * q + 1];
            }
    }
    // of m P-ths of a turn
    __device__ __forceinline__ double cosine(int m) const { return m == 0 ? 1.0 : c[(m <= H ? m : P - m) - 1]; }
    __device__ __forceinline__ double sine(int m) const { return m == 0 ? 0.0 : m <= H ? s[m - 1] : -s[P - m - 1]; }
};
template <int P, class W>
__device__ __forceinline__ void dft_out(const double2 (&v)[P], const DftRoots<P> &w, const W &write) {
    if constexpr (!(P & 1)) {
#pragma unroll
        for (int r = 0; r < P; ++r) write(r, v[r]);
    } else {
        constexpr int H = (P - 1) / 2;
        double2 sum = v[0];
#pragma unroll
        for (int j = 1; j <= H; ++j) sum = sum + v[j];
        write(0, sum);
#pragma unroll
        for (int k = 1; k <= H; ++k) {
            double ar = v[0].x, ai = v[0].y, br = 0.0, bi = 0.0;
#pragma unroll
            for (int j = 1; j <= H; ++j) {
                const double c = w.cosine(j * k % P), s = w.sine(j * k % P);
                ar = __builtin_fma(v[j].x, c, ar);
                ai = __builtin_fma(v[j].y, c, ai);
                br = __builtin_fma(v[P - j].x, s, br);
                bi = __builtin_fma(v[P - j].y, s, bi);
            }
            // a - i b and a + i b
            write(k, make_double2(ar + bi, ai - br));
            write(P - k, make_double2(ar - bi, ai + br));
            if (P > 9) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// One radix-P pass in place; R butterflies a thread at most.
template <int NT, int P, int R>
__device__ __forceinline__ void fft_pass(double2 *buf, const double2 *tw, const FftLen &f, int ns, uint32_t magic) {
    int n = f.n, tid = threadIdx.x;
    // nothing of a pass is the same in the next one: without this the compiler
    // keeps the addresses of every radix across the loop over the passes
    asm volatile("" : "+s"(n), "+v"(tid));
    const int nb = n / P, l = tid % FFT_LINES, step = nb / ns;
    double2 v[R][P];
    int base[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int j = tid / FFT_LINES + q * (NT / FFT_LINES);
        base[q] = -1;
        if (j < nb) {
            const int jq = ns > 1 ? (int)__umulhi((uint32_t)j, magic) : j, k = j - jq * ns;
            base[q] = jq * ns * P + k;
#pragma unroll
            for (int r = 0; r < P; ++r) v[q][r] = buf[(j + r * nb) * FFT_LINES + l];
            if (ns > 1)
#pragma unroll
                for (int r = 1; r < P; ++r) {
                    v[q][r] = zmul(v[q][r], tw[r * k * step]);
                    if (r % 4 == 0) __builtin_amdgcn_sched_barrier(0);   // bounds the twiddles in registers
                }
            dft_begin<P>(v[q]);
        }
    }
    __syncthreads();
    const DftRoots<P> roots(f.tw, n);
#pragma unroll
    for (int q = 0; q < R; ++q)
        if (base[q] >= 0) dft_out<P>(v[q], roots, [&](int r, double2 x) { buf[(base[q] + r * ns) * FFT_LINES + l] = x; });
    __syncthreads();
}

template <int NT, int P, int KIND>
__device__ __forceinline__ void fft_pass_any(double2 *buf, const double2 *tw, const FftLen &f, int ns, uint32_t magic) {
    constexpr int PER = NT / FFT_LINES;                // butterflies of a line a round
    constexpr int RMAX = ((NT == 256 ? FFT_SMALL : KIND ? FFT_MAXN : FFT_COMMON) / P + PER - 1) / PER;
    const int rounds = (f.n / P + PER - 1) / PER;
    if (rounds <= 1 || RMAX == 1) fft_pass<NT, P, 1>(buf, tw, f, ns, magic);
    else if (rounds == 2 || RMAX == 2) fft_pass<NT, P, RMAX < 2 ? 1 : 2>(buf, tw, f, ns, magic);
    else fft_pass<NT, P, RMAX>(buf, tw, f, ns, magic);
}

// First pass of a length with a prime factor P above 23: direct sums.  The
// values become x_r + x_{P-r} and x_r - x_{P-r} in place; a thread then sums KB
// outputs and their mirrors of one butterfly, the sums read once for all of
// them, the roots from the twiddle table.
template <int NT, int KB>
__device__ __forceinline__ void fft_direct(double2 *buf, const double2 *tw, int n, int P) {
    const int nb = n / P, H = (P - 1) / 2, l = threadIdx.x % FFT_LINES, slot = threadIdx.x / FFT_LINES;
    for (int x = slot; x < nb * H; x += NT / FFT_LINES) {
        const int r = x / nb + 1, j = x - (r - 1) * nb;
        double2 &a = buf[(j + r * nb) * FFT_LINES + l], &b = buf[(j + (P - r) * nb) * FFT_LINES + l];
        const double2 t = a + b, d = a - b;
        a = t;
        b = d;
    }
    __syncthreads();
    const int nblk = (H + KB) / KB, j = slot / nblk, k0 = slot - j * nblk;
    const bool in = j < nb;
    double ar[KB], ai[KB], br[KB], bi[KB];
    int at[KB];
    if (in) {
        const double2 x0 = buf[j * FFT_LINES + l];
#pragma unroll
        for (int q = 0; q < KB; ++q) {
            ar[q] = x0.x;
            ai[q] = x0.y;
            br[q] = bi[q] = 0.0;
            at[q] = 0;
        }
        for (int r = 1; r <= H; ++r) {
            const double2 t = buf[(j + r * nb) * FFT_LINES + l], d = buf[(j + (P - r) * nb) * FFT_LINES + l];
#pragma unroll
            for (int q = 0; q < KB; ++q) {
                const int k = k0 + q * nblk;                 // past H: a sum that is not written
                at[q] += k <= H ? k : 0;
                at[q] -= at[q] >= P ? P : 0;
                const double2 w = tw[at[q] * nb];            // cos, -sin
                ar[q] = __builtin_fma(t.x, w.x, ar[q]);
                ai[q] = __builtin_fma(t.y, w.x, ai[q]);
                br[q] = __builtin_fma(-d.x, w.y, br[q]);
                bi[q] = __builtin_fma(-d.y, w.y, bi[q]);
            }
        }
    }
    __syncthreads();
    if (in)
#pragma unroll
        for (int q = 0; q < KB; ++q) {
            const int k = k0 + q * nblk;
            if (k > H) continue;
            buf[(j * P + k) * FFT_LINES + l] = make_double2(ar[q] + bi[q], ai[q] - br[q]);
            if (k) buf[(j * P + P - k) * FFT_LINES + l] = make_double2(ar[q] - bi[q], ai[q] + br[q]);
        }
    __syncthreads();
}

// Forward transform of the FFT_LINES lines in buf, in place, natural order
// (the caller has synchronised buf and tw; synchronised on return).
template <int NT, int KIND>
__device__ __forceinline__ void fft_lines(double2 *buf, const double2 *tw, const FftLen &f) {
    int ns = 1;
    for (int p = 0; p < f.npass; ++p) {
        const uint32_t mg = f.magic[p];
        switch (f.radix[p]) {
        case 2: fft_pass_any<NT, 2, KIND>(buf, tw, f, ns, mg); break;
        case 3: fft_pass_any<NT, 3, KIND>(buf, tw, f, ns, mg); break;
        case 4: fft_pass_any<NT, 4, KIND>(buf, tw, f, ns, mg); break;
        case 5: fft_pass_any<NT, 5, KIND>(buf, tw, f, ns, mg); break;
        case 7: fft_pass_any<NT, 7, KIND>(buf, tw, f, ns, mg); break;
        case 8: fft_pass_any<NT, 8, KIND>(buf, tw, f, ns, mg); break;
        case 9: fft_pass_any<NT, 9, KIND>(buf, tw, f, ns, mg); break;
        default:
            if constexpr (KIND > 0) {
                switch (f.radix[p]) {
                case 11: fft_pass_any<NT, 11, KIND>(buf, tw, f, ns, mg); break;
                case 13: fft_pass_any<NT, 13, KIND>(buf, tw, f, ns, mg); break;
                case 17: fft_pass_any<NT, 17, KIND>(buf, tw, f, ns, mg); break;
                case 19: fft_pass_any<NT, 19, KIND>(buf, tw, f, ns, mg); break;
                case 23: fft_pass_any<NT, 23, KIND>(buf, tw, f, ns, mg); break;
                default:
                    if constexpr (KIND == 2) switch (fft_direct_kb(f.radix[p], f.n / f.radix[p], NT)) {
                    case 1: fft_direct<NT, 1>(buf, tw, f.n, f.radix[p]); break;
                    case 2: fft_direct<NT, 2>(buf, tw, f.n, f.radix[p]); break;
                    case 3: fft_direct<NT, 3>(buf, tw, f.n, f.radix[p]); break;
                    case 4: fft_direct<NT, 4>(buf, tw, f.n, f.radix[p]); break;
                    case 5: fft_direct<NT, 5>(buf, tw, f.n, f.radix[p]); break;
                    default: fft_direct<NT, FFT_KB>(buf, tw, f.n, f.radix[p]); break;
                    }
                }
            }
        }
        ns *= f.radix[p];
    }
}

// put(i, get(i)) of the thread's elements i of its line, B at a time so that their
// loads are in flight together.
template <int NT, int B, class Get, class Put>
__device__ __forceinline__ void fft_each(int n, const Get &get, const Put &put) {
    for (int i0 = threadIdx.x / FFT_LINES; i0 < n; i0 += B * (NT / FFT_LINES)) {
        double2 v[B];
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (i0 + u * (NT / FFT_LINES) < n) v[u] = get(i0 + u * (NT / FFT_LINES));
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (i0 + u * (NT / FFT_LINES) < n) put(i0 + u * (NT / FFT_LINES), v[u]);
    }
}

// One pass over an array of lines.  op.line(group, l) gives the thread's line,
// with load(i), store(i, v) and, for TWICE, mid(i, v) between two transforms;
// past the last line it loads zeros and stores nothing.
template <class Op, int NT, int KIND>
__global__ void __launch_bounds__(NT, KIND ? 4 : 6) fft_kernel(FftLen f, Op op) {
    extern __shared__ double2 fft_smem[];
    double2 *buf = fft_smem, *tw = fft_smem + (size_t)f.n * FFT_LINES;
    const int l = threadIdx.x % FFT_LINES;
    const auto line = op.line((long long)blockIdx.x, l);
    for (int k = threadIdx.x; k < f.n; k += NT) tw[k] = f.tw[k];
    fft_each<NT, 6>(f.n, [&](int i) { return line.load(i); }, [&](int i, double2 v) { buf[i * FFT_LINES + l] = v; });
    __syncthreads();
    for (int rep = 0;; ++rep) {
        fft_lines<NT, KIND>(buf, tw, f);
        if (!Op::TWICE || rep == 1) break;
        if constexpr (Op::TWICE)
            fft_each<NT, 2>(f.n, [&](int i) { return line.mid(i, buf[i * FFT_LINES + l]); },
                         [&](int i, double2 v) { buf[i * FFT_LINES + l] = v; });
        __syncthreads();
    }
    fft_each<NT, 2>(f.n, [&](int i) { return buf[i * FFT_LINES + l]; }, [&](int i, double2 v) { line.store(i, v); });
}

template <class Op>
hipError_t fft_launch(const FftLen &f, const Op &op, long long groups, hipStream_t st) {
    if (groups <= 0) return hipSuccess;
    if (groups > 0x7FFFFFFF || !f.tw) return hipErrorInvalidValue;
    const unsigned nb = (unsigned)groups;
    const size_t lds = fft_lds(f);
    if (fft_threads(f) == 256) {
        if (f.kind == 0) fft_kernel<Op, 256, 0><<<nb, 256, lds, st>>>(f, op);
        else if (f.kind == 1) fft_kernel<Op, 256, 1><<<nb, 256, lds, st>>>(f, op);
        else fft_kernel<Op, 256, 2><<<nb, 256, lds, st>>>(f, op);
    } else {
        if (f.kind == 0) fft_kernel<Op, 512, 0><<<nb, 512, lds, st>>>(f, op);
        else if (f.kind == 1) fft_kernel<Op, 512, 1><<<nb, 512, lds, st>>>(f, op);
        else fft_kernel<Op, 512, 2><<<nb, 512, lds, st>>>(f, op);
    }
    return hipGetLastError();
}

}  // namespace dc
