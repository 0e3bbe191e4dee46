// dc_host.h -- host-side state and helpers shared by the C-ABI translation
// units (dc_api.hip: the Fourier run, dc_refine.hip: the refinement model).
#pragma once
#include <algorithm>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "../../include/diffuse_turbo.h"
#include "dc_internal.h"

struct BatchState;   // dc_batch.hip
struct PostState;    // dc_post.hip
struct NufftState;   // dc_nufft.hip
namespace dc {
struct FftLen;       // dc_fft.h
}

struct DevBuf {
    void *p = nullptr;
    size_t n = 0;
};
// pinned host memory, readable and writable by kernels at the same address
struct PinBuf {
    unsigned char *p = nullptr;
    size_t n = 0;
};

struct dc_ctx {
    int device = 0;
    hipStream_t st = nullptr;
    int prec = DC_PREC_FP32;
    int tile = -1;                  // forced GEMM tile configuration, -1 = planned
    int autotune = 1;               // batch: time tile shapes on the first call of a shape
    int graphs = 1;                 // batch: capture the population step as a hipGraph
    int adj_walk = 0;               // adjoint column walk: 0 planned, else forced
    int dither = 1;                 // per-atom phase rotation of the phase GEMM (dither_turn)
    int slice_atoms = 0;            // forced atoms per GEMM slice, 0 = planned
    BatchState *batch = nullptr;    // cached plan / buffers / graph of the last batch shape
    PostState *post = nullptr;      // FFT plans and buffers of the post-processing calls
    NufftState *nufft = nullptr;    // fine grid, plans and buffers of the NUFFT technique
    std::map<int, DevBuf> fft_tw;   // twiddles of the transform lengths used (dc_fft.h; 600 lengths, 10 KB each at most)
    std::string err;
    int err_typ = DC_ER_NONE;
    const volatile int *cancel = nullptr;
    hipEvent_t ev[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    dc_stats stats{};
    // timed spans of the current call whose events the host has not waited
    // for: (start, end, stats field the elapsed ms are added to); tev is the
    // pool their events come from (tev_used in use)
    struct Span {
        hipEvent_t a, b;
        double *dst;
    };
    std::vector<Span> spans;
    std::vector<hipEvent_t> tev;
    size_t tev_used = 0;
    // device buffers of the Fourier run
    DevBuf rec, slice_beg, slice_order, slice_type, lot_slice, partial, cfact, istl, idx, oid, offs, xat, w;
    DevBuf acsf, dsi, csf, wm, wv, lat, out_tcsf, out[5];
    // device buffers of the refinement model
    DevBuf m_pos, m_w, m_b, m_sq, m_q, m_part, m_grad, m_tiles, m_gi, m_f, m_qt, m_qs, m_jw, m_dsl, m_di, m_rng, m_ref;
    // crystal
    bool have_crystal = false;
    DevBuf pos, iscat;
    std::vector<double> h_pos;
    std::vector<int> h_iscat;
    int64_t natoms = 0;
    int icc[3] = {1, 1, 1};
    int ncatoms = 1, nscat = 0;
    double dim0[3] = {0, 0, 0}, dim_lo[3] = {0, 0, 0};
    std::vector<int> type_beg;      // per type offsets into d type list
    DevBuf type_idx;
    // lot gather (DISCUS-ordered crystals, natoms == cells x sites): per type,
    // the atoms in (cell, site) order on the device (tc_idx, type t from
    // type_beg[t]) and per type the first position of every cell in that list
    // (tc_start[t * (ncell + 1) + cell], host), so that a run of consecutive
    // cells of a lot is one contiguous range
    std::vector<int> tc_start;
    DevBuf runs;
    // Staging of a call's small host arrays (see stage): packed into h_arena and
    // copied to arena by one kernel; outputs of host entry points that fit
    // come back through h_out.  Both belong to the context, whose calls wait
    // for their stream, and are reused by the next call.
    PinBuf h_arena, h_out;
    DevBuf arena;
    size_t arena_n = 0, arena_done = 0;   // bytes packed / already copied in this call
    size_t arena_want = 0;                // bytes this call asked for
    bool arena_busy = false;              // a copy was launched and not waited for
    // this device's dc_scratch array (dc_noalloc.hip), looked up at creation
    void *scratch = nullptr;
    // rec's records carry the rotation hash in AtomRec::pad (PrepArgs::hash_salt):
    // set by the Fourier run's prep, cleared by the refinement's, whose
    // adjoints read pad as B
    bool rec_hash = false;

    std::vector<DevBuf *> buffers() {
        return {&rec, &slice_beg, &slice_order, &slice_type, &lot_slice, &partial, &cfact, &istl, &idx, &oid, &offs, &xat, &w,
                &acsf, &dsi, &csf, &wm, &wv, &lat, &out_tcsf, &out[0], &out[1], &out[2], &out[3], &out[4],
                &m_pos, &m_w, &m_b, &m_sq, &m_q, &m_part, &m_grad, &m_tiles, &m_gi, &m_f, &m_qt, &m_qs, &m_jw, &m_dsl, &m_di, &m_rng, &m_ref,
                &pos, &iscat, &type_idx, &runs, &arena};
    }
};

namespace dc {

inline int set_err(dc_ctx *c, int code, int typ, const std::string &msg) {
    if (c) {
        c->err = msg;
        c->err_typ = typ;
    }
    return code;
}

inline int hip_err(dc_ctx *c, hipError_t e, const char *where) {
    return set_err(c, e == hipErrorOutOfMemory ? DC_ERR_NOMEM : DC_ERR_DEVICE, DC_ER_LIB,
                   std::string(where) + ": " + hipGetErrorString(e));
}

#define HIPCHK(call)                                        \
    do {                                                    \
        hipError_t e_ = (call);                             \
        if (e_ != hipSuccess) return hip_err(c, e_, #call); \
    } while (0)

// Grow-only device buffer (reallocation synchronises the context stream).
inline int ensure(dc_ctx *c, DevBuf &b, size_t bytes) {
    if (bytes == 0) bytes = 16;
    if (b.n >= bytes) return 0;
    if (b.p) {
        hipError_t e = hipStreamSynchronize(c->st);
        if (e != hipSuccess) return hip_err(c, e, "sync before realloc");
        (void)hipFree(b.p);
        b.p = nullptr;
        b.n = 0;
    }
    size_t n = bytes + bytes / 8;
    hipError_t e = hipMalloc(&b.p, n);
    if (e != hipSuccess) {
        b.p = nullptr;
        return hip_err(c, e, "hipMalloc");
    }
    b.n = n;
    return 0;
}

template <class T>
T *ptr(DevBuf &b) {
    return reinterpret_cast<T *>(b.p);
}

template <class T>
int upload(dc_ctx *c, DevBuf &b, const T *src, size_t count) {
    int st = ensure(c, b, sizeof(T) * count);
    if (st) return st;
    if (count) HIPCHK(hipMemcpyAsync(b.p, src, sizeof(T) * count, hipMemcpyHostToDevice, c->st));
    return 0;
}

// Staging.  A call's tables (slice boundaries and types, form-factor rows, lot
// runs) are a few kilobytes each; copied one by one from pageable memory they
// cost about 15 us of host time apiece, which is most of a small call.  They
// are packed into pinned memory instead and one kernel copies them.
// stage_begin starts a call, stage returns the device address of a packed copy
// (falling back to upload into b when the arena is full: it grows with the
// next call, up to ARENA_MAX), stage_flush launches
// the copy of what has been packed; every launch that reads staged data comes
// after a flush.
constexpr size_t ARENA_MIN = 256u << 10, ARENA_MAX = 8u << 20;
hipError_t launch_stage_copy(const void *src, void *dst, size_t bytes, hipStream_t st);   // dc_lot.hip

inline int pin_ensure(dc_ctx *c, PinBuf &b, size_t bytes) {
    if (b.n >= bytes) return 0;
    if (b.p) (void)hipHostFree(b.p);
    b.p = nullptr;
    b.n = 0;
    void *p = nullptr;
    hipError_t e = hipHostMalloc(&p, bytes, hipHostMallocDefault);
    if (e != hipSuccess) return hip_err(c, e, "hipHostMalloc");
    b.p = static_cast<unsigned char *>(p);
    b.n = bytes;
    return 0;
}
inline int stage_begin(dc_ctx *c) {
    int st;
    if (c->arena_busy) HIPCHK(hipStreamSynchronize(c->st));   // an earlier call ended early
    c->arena_busy = false;
    size_t n = ARENA_MIN;
    while (n < c->arena_want && n < ARENA_MAX) n *= 2;
    n = std::max(n, c->h_arena.n);
    c->arena_n = c->arena_done = c->arena_want = 0;
    if ((st = pin_ensure(c, c->h_arena, n))) return st;
    return ensure(c, c->arena, n);
}
template <class T>
int stage(dc_ctx *c, DevBuf &b, const T *src, size_t count, T *&dev) {
    const size_t bytes = sizeof(T) * count;
    const size_t room = (bytes + 255) & ~(size_t)255;
    c->arena_want += room;
    if (room > c->h_arena.n - c->arena_n) {
        int st = upload(c, b, src, count);
        dev = ptr<T>(b);
        return st;
    }
    if (bytes) std::memcpy(c->h_arena.p + c->arena_n, src, bytes);
    dev = reinterpret_cast<T *>(static_cast<unsigned char *>(c->arena.p) + c->arena_n);
    c->arena_n += room;
    return 0;
}
inline int stage_flush(dc_ctx *c) {
    if (c->arena_n == c->arena_done) return 0;
    HIPCHK(launch_stage_copy(c->h_arena.p + c->arena_done, static_cast<unsigned char *>(c->arena.p) + c->arena_done,
                             c->arena_n - c->arena_done, c->st));
    c->arena_done = c->arena_n;
    c->arena_busy = true;
    return 0;
}
// Form-factor rows 0 .. rows-1 of the nscat columns of a (ncfact, nscat) table.
inline int stage_cfact(dc_ctx *c, const double *cfact, int ncfact, int nscat, int rows, double2 *&dev) {
    if (rows == ncfact) return stage(c, c->cfact, reinterpret_cast<const double2 *>(cfact), (size_t)ncfact * nscat, dev);
    std::vector<double2> v((size_t)rows * nscat);
    for (int t = 0; t < nscat; ++t)
        std::memcpy(v.data() + (size_t)rows * t, cfact + 2 * (size_t)ncfact * t, sizeof(double2) * rows);
    return stage(c, c->cfact, v.data(), v.size(), dev);
}
// Rows of the form-factor table a grid reaches: its largest bin lies at a
// corner; two rows more cover bins that round up beside it.
inline int cfact_rows(int corner_bin, int ncfact) { return std::min(ncfact, corner_bin + 3); }

// Outputs of a host entry point up to this size are written by the last
// kernel into pinned memory and copied to the caller's arrays from there.
constexpr size_t HOST_OUT_BYTES = 8u << 20;

// Deferred timing: mark() records a pool event on the context stream;
// span() files (start, end) to be added to a stats field once the host has
// waited for the stream, so that timing a kernel does not stall the host
// between launches.  stats_begin() starts a call's statistics (dropping the
// spans of an earlier call), resolve_spans() waits for the last span and
// adds every span's elapsed time.
inline int mark(dc_ctx *c, hipEvent_t &e) {
    if (c->tev_used == c->tev.size()) {
        hipEvent_t n = nullptr;
        HIPCHK(hipEventCreate(&n));
        c->tev.push_back(n);
    }
    e = c->tev[c->tev_used++];
    HIPCHK(hipEventRecord(e, c->st));
    return 0;
}
inline void span(dc_ctx *c, hipEvent_t a, hipEvent_t b, double *dst) { c->spans.push_back({a, b, dst}); }
inline void stats_begin(dc_ctx *c) {
    c->stats = dc_stats{};
    c->spans.clear();
    c->tev_used = 0;
}
inline int resolve_spans(dc_ctx *c) {
    if (c->spans.empty()) return 0;
    HIPCHK(hipEventSynchronize(c->spans.back().b));
    for (const auto &s : c->spans) {
        float ms = 0.f;
        HIPCHK(hipEventElapsedTime(&ms, s.a, s.b));
        *s.dst += ms;
    }
    c->spans.clear();
    c->tev_used = 0;
    return 0;
}

inline bool cancelled(dc_ctx *c) { return c->cancel && *c->cancel; }

// GEMM plan of a grid region (dc_api.hip).
struct Plan {
    GemmGeom gg{};
    int mapping = 0;
    int tile = 0;
    int scheme = 0;              // GEMM scheme the plan is for (DC_PREC_* or SCHEME_FP32_ACC64)
};

// Slices over a list of (type, count) segments laid out consecutively.
struct SliceSet {
    std::vector<int> beg;        // nslice + 1 atom offsets
    std::vector<int> type;       // per slice
    std::vector<int> lot;        // lot boundaries (slice ids), nlots + 1
    std::vector<int> seg_first;  // first slice of each segment
};

long long padded(long long n, long long t);
int max_corner_bin(const Grid &g);   // largest sin(theta)/lambda bin over the grid corners
// Work items per slice of a tile on a geometry (gg.fold names the folded
// side of a mirrored-pair tile), and the better side a mask allows (0: none).
int gemm_items(const GemmGeom &gg, int tile);
int fold_side(const GemmGeom &gg, int fold_mask, int tile);
// fold_mask: sides that the mirrored-pair tiles may fold (FOLD_COLS |
// FOLD_ROWS); a damped launch needs s^2 mirrored about the side's centre.
Plan plan_gemm(Grid &g, int forced, int only_mapping = -1, int prec = 1, long long natoms = 0,
               int fold_mask = FOLD_COLS | FOLD_ROWS);
// Geometry of mapping 0, which no tile changes.
GemmGeom mapping0_geom(const Grid &g);
// Slice length of a fold tile for a launch's segments, and its predicted time.
int fold_slices(const GemmGeom &gg, int tile, const std::vector<std::pair<int, int>> &segs, int prec, double &best_us,
                bool lots = false);
// the sides whose s^2 parts (R row values, then C column values) are mirrored
int mirrored_sides(const GemmGeom &gg, const float *sq);
int kchunk_for(const Plan &pl, long long natoms_batch, int prec);
int kchunk_for(const Plan &pl, const std::vector<std::pair<int, int>> &segs, int prec, bool lots = false);
void add_segments(SliceSet &s, const std::vector<std::pair<int, int>> &segs, int kchunk, int &atom_off);
// beg: the slices' atom offsets (nslice + 1), d_beg: the same on the device
int run_gemm(dc_ctx *c, const Plan &pl, const std::vector<int> &beg, const int *d_beg, float2 *partial,
             const float *sq = nullptr);
// atoms per slice: the context's forced length (dc_set_slice_atoms) or the planned one
inline int slice_len(const dc_ctx *c, int planned) { return c->slice_atoms > 0 ? c->slice_atoms : planned; }
// the plan's geometry with the context's dither salt
inline GemmGeom launch_geom(const dc_ctx *c, const GemmGeom &g) {
    GemmGeom r = g;
    r.dither = c->dither ? 0x2545F491u : 0u;
    return r;
}
void batch_release(dc_ctx *c);   // frees the cached batch plan, buffers and graph
void post_release(dc_ctx *c);    // frees the FFT plans and buffers of the post-processing calls
int fft_table(dc_ctx *c, FftLen &f);   // f.tw, made on a length's first use
void fft_release(dc_ctx *c);
void nufft_release(dc_ctx *c);   // frees the NUFFT fine grid, plans and buffers
int noalloc_attach(dc_ctx *c);   // device address of this device's dc_scratch (dc_noalloc.hip)
PrepArgs base_prep(const Grid &g, int mapping);
// Products of the refinement model's and the populations' forward sums: a
// gradient amplifies the error of F, so BF16X3 runs the FP16X3 products there
// (the same MFMA rate), as the Bragg-subtracted runs do.
inline int model_scheme(int prec) { return prec == DC_PREC_BF16X3 ? DC_PREC_FP16X3 : prec; }
// s^2 of a grid (metric rten, corner eck, increments vi) as the sum of a part of
// the R rows and one of the C columns (f1 valid of each period of C0, the others
// 0), R + C floats.  For the schemes with FP16 operands (sq_floats: twice as many)
// the least row part is moved to the columns -- on a grid whose rows and columns are
// orthogonal both parts are then >= 0, and neither factor of exp(-B s^2) exceeds 1
// for B >= 0 -- and behind the floats lie what they leave of the parts (damp_back2).
inline bool f16_scheme(int scheme) { return scheme == DC_PREC_FP16X2 || scheme == DC_PREC_FP16X3; }
inline int sq_floats(const GemmGeom &gg, bool f16) { return (gg.R + gg.C) * (f16 ? 2 : 1); }
void split_sq(const double *rten, const double *eck, const double *vi, const GemmGeom &gg, int f1, bool f16, float *out);

}  // namespace dc
