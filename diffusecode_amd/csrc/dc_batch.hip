// dc_batch.hip -- population scoring: chi^2 (and its gradient) of many trial
// structures against their own target grids in one pass.
//
// DIFFEV evaluates a generation by running one DISCUS macro per member over
// its MPI farm (diffev/prog/diffev_kdo.f90:676, lib_f90/with_mpi.f90:281-609).
// Here every member's atoms become GEMM slices of ONE persistent phase-GEMM
// launch (uneven member sizes are balanced by slicing), one fused reduction
// forms F, I, chi^2 and the adjoint's Q planes for all members, and one
// adjoint launch gives the gradients.  The whole step is captured once per
// batch shape as a hipGraph and replayed for every later generation; the
// GEMM tile shape and persistent grid size are chosen by timing the
// candidates on the batch itself (autotuner).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "dc_host.h"

using namespace dc;

struct BatchState {
    // key: the shape of the batch
    int nmembers = 0, nscat = 0, ncfact = 0, prec = -1, tile_forced = -2, autotune = -1, graphs = -1;
    int slice_atoms = -1, dither = -1;
    int fold_mask = 0;                       // sides the mirrored-pair tiles may fold (dc_fold.h)
    bool want_grad = false, want_icalc = false, have_weight = false, any_b = false;
    std::vector<int64_t> atom_beg;
    std::vector<int> type;
    double eck[12] = {}, vi[9] = {};
    int inc[3] = {0, 0, 0};
    // plan
    Grid g{};
    Plan pl;
    int nwg = 0;
    std::vector<int> order;
    std::vector<std::pair<int, int>> segs;   // (type, atoms) per member and type, member-major
    std::vector<int> seg_member;
    int kchunk = 0;                          // atoms per GEMM slice
    int sq_stride = 0;                       // floats of a member's s^2 parts
    int nsorted = 0, nslice = 0, ntiles = 0, nblk = 0;
    AdjArgs adj{};                       // plan of the reverse pass, and its launches
    std::vector<AdjSpan> spans;
    int walk_req = 0;                    // the context's adjoint walk setting at planning
    int64_t natoms = 0;
    int rows = 0;                        // form-factor rows on the device (the bins the metrics reach, and a margin)
    PinBuf h_cf, h_sq, h_chi;            // pinned: form-factor rows, s^2 parts, chi^2 of the members
    DevBuf pos, occ, bdw, idx, rec, sbeg, stype, ssq, msl, sorder, partial, cfact, rten, sq, target, weight, icalc,
        chi, q, qs, atiles, aranges, aref, part, grad, wq;
    bool queue = false;                  // GEMM items from a device counter (autotuner's choice)
    bool primed = false;                 // records built and autotuned once
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    float tune_best_ms = 0.f;

    std::vector<DevBuf *> buffers() {
        return {&pos, &occ, &bdw, &idx, &rec, &sbeg, &stype, &ssq, &msl, &sorder, &partial, &cfact, &rten, &sq,
                &target, &weight, &icalc, &chi, &q, &qs, &atiles, &aranges, &aref, &part, &grad, &wq};
    }
};

namespace dc {

void batch_release(dc_ctx *c) {
    BatchState *b = c->batch;
    if (!b) return;
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    for (DevBuf *d : b->buffers())
        if (d->p) (void)hipFree(d->p);
    for (PinBuf *p : {&b->h_cf, &b->h_sq, &b->h_chi})
        if (p->p) (void)hipHostFree(p->p);
    delete b;
    c->batch = nullptr;
}

}  // namespace dc

namespace {

double dotg(const double *a, const double *g, const double *b) {
    double s = 0.0;
    for (int r = 0; r < 3; ++r)
        for (int k = 0; k < 3; ++k) s += a[r] * g[r + 3 * k] * b[k];
    return s;
}

// The cached state fits the call, its atom types apart (same_types).
bool same_shape(const BatchState *b, const dc_ctx *c, const dc_batch_desc *d, bool want_grad, bool want_icalc,
                bool have_weight, bool any_b) {
    if (!b) return false;
    if (b->nmembers != d->nmembers || b->nscat != d->nscat || b->ncfact != d->ncfact || b->prec != c->prec ||
        b->tile_forced != c->tile || b->autotune != c->autotune || b->graphs != c->graphs ||
        b->want_grad != want_grad || b->want_icalc != want_icalc || b->have_weight != have_weight ||
        b->any_b != any_b || b->walk_req != c->adj_walk || b->slice_atoms != c->slice_atoms || b->dither != c->dither)
        return false;
    if (std::memcmp(b->eck, d->eck, sizeof(b->eck)) || std::memcmp(b->vi, d->vi, sizeof(b->vi)) ||
        std::memcmp(b->inc, d->inc, sizeof(b->inc)))
        return false;
    return std::equal(b->atom_beg.begin(), b->atom_beg.end(), d->atom_beg);
}
bool same_types(const BatchState &b, const dc_batch_desc *d) {
    return std::memcmp(b.type.data(), d->type, sizeof(int) * b.type.size()) == 0;
}

int check_desc(dc_ctx *c, const dc_batch_desc *d) {
    if (!d || d->nmembers < 1 || !d->atom_beg || !d->pos || !d->type || !d->occ || !d->cfact || !d->rten ||
        d->nscat < 1 || d->ncfact < 1)
        return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: null pointer or bad size");
    if (d->atom_beg[0] != 0) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: atom_beg[0] must be 0");
    for (int m = 0; m < d->nmembers; ++m)
        if (d->atom_beg[m + 1] < d->atom_beg[m]) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: atom_beg decreasing");
    const int64_t n = d->atom_beg[d->nmembers];
    if (n > INT32_MAX / 8) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: too many atoms");
    for (int k = 0; k < 3; ++k)
        if (d->inc[k] < 1) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: bad inc");
    return 0;
}
int check_types(dc_ctx *c, const dc_batch_desc *d) {
    const int64_t n = d->atom_beg[d->nmembers];
    for (int64_t k = 0; k < n; ++k)
        if (d->type[k] < 0 || d->type[k] > d->nscat) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: type outside 0..nscat");
    return 0;
}

// s^2 row / column parts for every member's metric; errors on grids that are
// not metric-orthogonal between rows and columns when B or gradients need it.
int member_sq(dc_ctx *c, const Grid &g, const GemmGeom &gg, const dc_batch_desc *d, std::vector<float> &sq, bool need_sep,
              int &top_bin) {
    top_bin = 0;
    const bool f16 = f16_scheme(model_scheme(c->prec));
    const int stride = sq_floats(gg, f16);
    sq.resize((size_t)stride * d->nmembers);
    const double *v1 = d->vi;
    for (int m = 0; m < d->nmembers; ++m) {
        const double *G = d->rten + 9 * m;
        if (need_sep) {
            const double n1 = std::sqrt(std::fabs(dotg(v1, G, v1)));
            for (int ax = 1; ax < 3; ++ax) {
                if (d->inc[ax] <= 1) continue;
                const double *v = d->vi + 3 * ax;
                const double nv = std::sqrt(std::fabs(dotg(v, G, v)));
                if (std::fabs(dotg(v1, G, v)) > 1e-12 * std::max(1.0, n1 * nv))
                    return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: vi(:,1) not metric-orthogonal to vi(:,2), vi(:,3)");
            }
        }
        split_sq(G, d->eck, d->vi, gg, g.f[1], f16, sq.data() + (size_t)stride * m);
        Grid gm = g;
        for (int k = 0; k < 9; ++k) gm.rten[k] = G[k];
        top_bin = std::max(top_bin, max_corner_bin(gm));
        if (top_bin >= d->ncfact) return set_err(c, DC_ERR_ISTL, DC_ER_FOUR, "sin(theta)/lambda beyond table");
    }
    return 0;
}

// GEMM slices of at most kchunk atoms over the member-major, type-sorted
// segments: slice tables, each member's slice range and metric offset, the
// launch order and the plane buffer.
int make_slices(dc_ctx *c, BatchState &b, int kchunk) {
    const GemmGeom &gg = b.pl.gg;
    SliceSet ss;
    std::vector<int> mslice, slice_sq;
    int off = 0;
    size_t sg = 0;
    for (int m = 0; m < b.nmembers; ++m) {
        mslice.push_back((int)ss.type.size());
        for (; sg < b.segs.size() && b.seg_member[sg] == m; ++sg) {
            add_segments(ss, {b.segs[sg]}, kchunk, off);
            while ((int)slice_sq.size() < (int)ss.type.size()) slice_sq.push_back(m * b.sq_stride);
        }
    }
    mslice.push_back((int)ss.type.size());
    if (ss.beg.empty()) ss.beg.push_back(0);
    b.nslice = (int)ss.type.size();
    b.kchunk = kchunk;
    int st;
    if ((st = upload(c, b.sbeg, ss.beg.data(), ss.beg.size()))) return st;
    if ((st = upload(c, b.stype, ss.type.data(), ss.type.size()))) return st;
    if ((st = upload(c, b.ssq, slice_sq.data(), slice_sq.size()))) return st;
    if ((st = upload(c, b.msl, mslice.data(), mslice.size()))) return st;
    // GEMM launch order of the slices: longest first.  Members of uneven size
    // give slices of uneven length, and in member order a long slice can
    // start in the launch's last round of work-groups and run alone
    std::vector<int> sorder(std::max(b.nslice, 1), 0);
    for (int s = 0; s < b.nslice; ++s) sorder[s] = s;
    std::stable_sort(sorder.begin(), sorder.begin() + b.nslice,
                     [&](int x, int y) { return ss.beg[x + 1] - ss.beg[x] > ss.beg[y + 1] - ss.beg[y]; });
    if ((st = upload(c, b.sorder, sorder.data(), sorder.size()))) return st;
    return ensure(c, b.partial, sizeof(float2) * gg.P * std::max(b.nslice, 1));
}

Grid batch_grid(const dc_batch_desc *d) {
    Grid g{};
    for (int k = 0; k < 3; ++k) {
        g.n[k] = g.f[k] = d->inc[k];
        g.xm[k] = d->eck[k];
        g.uin[k] = d->vi[k];
        g.vin[k] = d->vi[3 + k];
        g.win[k] = d->vi[6 + k];
    }
    g.P = (long long)g.f[0] * g.f[1] * g.f[2];
    return g;
}

int build_state(dc_ctx *c, const dc_batch_desc *d, BatchState &b) {
    b.nmembers = d->nmembers;
    b.nscat = d->nscat;
    b.ncfact = d->ncfact;
    b.prec = c->prec;
    b.walk_req = c->adj_walk;
    b.tile_forced = c->tile;
    b.slice_atoms = c->slice_atoms;
    b.dither = c->dither;
    b.autotune = c->autotune;
    b.graphs = c->graphs;
    b.natoms = d->atom_beg[d->nmembers];
    b.atom_beg.assign(d->atom_beg, d->atom_beg + d->nmembers + 1);
    b.type.assign(d->type, d->type + b.natoms);
    std::memcpy(b.eck, d->eck, sizeof(b.eck));
    std::memcpy(b.vi, d->vi, sizeof(b.vi));
    std::memcpy(b.inc, d->inc, sizeof(b.inc));
    Grid &g = b.g;
    g = batch_grid(d);
    b.pl = plan_gemm(g, c->tile, 0, model_scheme(c->prec), d->atom_beg[d->nmembers], b.fold_mask);
    const GemmGeom &gg = b.pl.gg;
    b.sq_stride = sq_floats(gg, f16_scheme(b.pl.scheme));

    // member-major, type-sorted atom order; adjoint tiles; slices
    std::vector<int> tiles;
    std::vector<std::pair<int, int>> &segs_all = b.segs;
    std::vector<int> &seg_member = b.seg_member;
    segs_all.clear();
    seg_member.clear();
    b.order.clear();
    for (int m = 0; m < d->nmembers; ++m) {
        std::vector<int> cnt(d->nscat + 1, 0);
        for (int64_t k = d->atom_beg[m]; k < d->atom_beg[m + 1]; ++k) cnt[d->type[k]]++;
        for (int t = 1; t <= d->nscat; ++t) {
            if (!cnt[t]) continue;
            for (int64_t k = d->atom_beg[m]; k < d->atom_beg[m + 1]; ++k)
                if (d->type[k] == t) b.order.push_back((int)k);
            segs_all.push_back({t - 1, cnt[t]});
            seg_member.push_back(m);
        }
    }
    b.nsorted = (int)b.order.size();
    int off = 0;
    const int na = adjoint_tile_atoms();
    std::vector<int2> ranges((size_t)d->nmembers * d->nscat, make_int2(0, 0));
    for (size_t sg = 0; sg < segs_all.size(); ++sg) {
        const int m = seg_member[sg];
        ranges[(size_t)m * d->nscat + segs_all[sg].first] = make_int2(off, off + segs_all[sg].second);
        for (int k = 0; k < segs_all[sg].second; k += na)
            tiles.insert(tiles.end(), {off + k, off + std::min(segs_all[sg].second, k + na),
                                       m * d->nscat + segs_all[sg].first, m});
        off += segs_all[sg].second;
    }
    b.ntiles = (int)tiles.size() / 4;
    b.adj = AdjArgs{};
    b.adj.R = gg.R;
    b.adj.C = gg.C;
    b.adj.C0 = gg.C0;
    b.adj.f1 = g.f[1];
    b.adj.fold = (b.fold_mask & FOLD_ROWS) != 0;
    b.adj.damped = b.any_b;
    b.adj.natoms = b.nsorted;
    adjoint_plan(b.adj, b.ntiles, b.prec != DC_PREC_FP32, c->adj_walk);
    b.spans = adjoint_spans(b.adj, tiles.data(), b.ntiles);
    b.nblk = (int)std::min<long long>((g.P + 255) / 256, 256);

    int st;
    const size_t M = (size_t)d->nmembers;
    if ((st = upload(c, b.idx, b.order.data(), b.order.size()))) return st;
    if ((st = make_slices(c, b, slice_len(c, kchunk_for(b.pl, b.segs, b.pl.scheme))))) return st;
    if ((st = upload(c, b.atiles, tiles.data(), tiles.size()))) return st;
    if ((st = upload(c, b.aranges, ranges.data(), ranges.size()))) return st;
    if ((st = ensure(c, b.aref, sizeof(float) * ranges.size()))) return st;
    if ((st = ensure(c, b.rec, sizeof(AtomRec) * std::max(b.nsorted, 1)))) return st;
    if ((st = ensure(c, b.cfact, sizeof(double) * 2 * (size_t)b.rows * d->nscat * M))) return st;
    if ((st = pin_ensure(c, b.h_cf, sizeof(double) * (2 * (size_t)b.rows * d->nscat + 9) * M))) return st;
    if ((st = pin_ensure(c, b.h_sq, sizeof(float) * (size_t)b.sq_stride * M))) return st;
    if ((st = pin_ensure(c, b.h_chi, sizeof(double) * M))) return st;
    if ((st = ensure(c, b.rten, sizeof(double) * 9 * M))) return st;
    if ((st = ensure(c, b.sq, sizeof(float) * (size_t)b.sq_stride * M))) return st;
    if ((st = ensure(c, b.chi, sizeof(double) * (size_t)b.nblk * M))) return st;
    if (b.want_grad) {
        if ((st = ensure(c, b.q, sizeof(float2) * gg.P * d->nscat * M))) return st;
        if ((st = ensure(c, b.part, sizeof(double) * 6 * (size_t)b.adj.nset * std::max(b.nsorted, 1)))) return st;
        long long most = 0;
        for (const AdjSpan &s : b.spans) most = std::max<long long>(most, s.nplanes);
        if ((st = ensure(c, b.qs, sizeof(uint4) * (size_t)(b.adj.plane_words * most)))) return st;
    }
    return 0;
}

// Arrays of one step: the state's own (host entry point, replayed graph) or the
// caller's device arrays.
struct StepIO {
    const double *pos, *occ, *bdw, *target, *weight;
    double *icalc, *grad;
};
StepIO own_io(BatchState &b) {
    return {ptr<double>(b.pos), ptr<double>(b.occ), b.any_b ? ptr<double>(b.bdw) : nullptr, ptr<double>(b.target),
            b.have_weight ? ptr<double>(b.weight) : nullptr, b.want_icalc ? ptr<double>(b.icalc) : nullptr,
            b.want_grad ? ptr<double>(b.grad) : nullptr};
}

// chi^2 of every member from the reduction's block sums, into pinned memory.
__global__ void chi_finish_kernel(const double *__restrict__ part, int nblk, double *__restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int k = threadIdx.x; k < nblk; k += 256) s += part[(size_t)blockIdx.x * nblk + k];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// The reduction of the slice planes: every member's I, its chi^2 partial sums
// and, when gradients are wanted, the Q planes.
int reduce_planes(dc_ctx *c, BatchState &b, const StepIO &io) {
    const GemmGeom &gg = b.pl.gg;
    BatchReduceArgs ra{};
    ra.g = b.g;
    ra.R = gg.R;
    ra.C = gg.C;
    ra.C0 = gg.C0;
    ra.plane = gg.P;
    ra.partial = ptr<float2>(b.partial);
    ra.mslice = ptr<int>(b.msl);
    ra.slice_type = ptr<int>(b.stype);
    ra.cfact = ptr<double2>(b.cfact);
    ra.ncfact = b.rows;
    ra.nscat = b.nscat;
    ra.nmembers = b.nmembers;
    ra.rten = ptr<double>(b.rten);
    ra.target = io.target;
    ra.weight = io.weight;
    ra.icalc = io.icalc;
    ra.chi_part = ptr<double>(b.chi);
    ra.q = b.want_grad ? ptr<float2>(b.q) : nullptr;
    HIPCHK(launch_batch_reduce(ra, b.nblk, c->st));
    return 0;
}

// Kernels of one population step, in stream order (captured into the graph).
// part: STEP_GEMM = records (prep) and GEMM, STEP_REST = the reduction (I,
// chi^2, Q planes) and the adjoint when gradients are wanted.
constexpr int STEP_GEMM = 1, STEP_REST = 2;
__global__ void zero_counter_kernel(int *p) {
    if (threadIdx.x == 0) *p = 0;
}

int enqueue(dc_ctx *c, BatchState &b, const StepIO &io, int tile, int nwg, bool prep, int part, bool queue) {
    const GemmGeom &gg = b.pl.gg;
    int st;
    if (prep) {
        PrepArgs pa = base_prep(b.g, 0);
        pa.src = io.pos;
        pa.src_ld = 0;
        pa.idx = ptr<int>(b.idx);
        pa.occ_src = io.occ;
        pa.bdw_src = io.bdw;
        pa.n = b.nsorted;
        if (b.nsorted > 0) HIPCHK(launch_prep(pa, ptr<AtomRec>(b.rec), c->st));
    }
    if (part & STEP_GEMM) {
        GemmGeom lg = launch_geom(c, gg);
        lg.fold = fold_side(gg, b.fold_mask, tile);
        lg.order = ptr<int>(b.sorder);
        if (queue) {
            if ((st = ensure(c, b.wq, 256))) return st;
            zero_counter_kernel<<<1, 64, 0, c->st>>>(ptr<int>(b.wq));
            HIPCHK(hipGetLastError());
            lg.queue = ptr<int>(b.wq);
        }
        HIPCHK(launch_phase_gemm(b.pl.scheme, tile, ptr<AtomRec>(b.rec), ptr<int>(b.sbeg), ptr<float2>(b.partial),
                                 b.any_b ? ptr<float>(b.sq) : nullptr, lg, 0, b.nslice, c->st, nwg, ptr<int>(b.ssq)));
    }
    if (!(part & STEP_REST)) return 0;
    if ((st = reduce_planes(c, b, io))) return st;
    chi_finish_kernel<<<b.nmembers, 256, 0, c->st>>>(ptr<double>(b.chi), b.nblk, reinterpret_cast<double *>(b.h_chi.p));
    HIPCHK(hipGetLastError());
    if (b.want_grad) {
        AdjArgs aa = b.adj;
        aa.rec = ptr<AtomRec>(b.rec);
        aa.tiles = ptr<int4>(b.atiles);
        aa.q = ptr<float2>(b.q);
        aa.sq = ptr<float>(b.sq);
        aa.sq_stride = b.sq_stride;
        aa.planes_per_sq = b.nscat;
        aa.part = ptr<double>(b.part);
        aa.plane = gg.P;
        aa.natoms = b.nsorted;
        aa.rc = 0.5f * (float)(b.g.f[0] - 1);
        aa.jc = 0.5f * (float)(b.g.f[1] - 1);
        aa.mc = 0.5f * (float)(b.g.f[2] - 1);
        aa.ranges = ptr<int2>(b.aranges);
        aa.ref = ptr<float>(b.aref);
        HIPCHK(launch_adj_begin(aa, b.nmembers * b.nscat, io.grad, 5 * b.natoms, c->st));
        for (const AdjSpan &s : b.spans) HIPCHK(launch_adjoint(aa, s, ptr<uint4>(b.qs), c->st));
        AdjFinishArgs fa{};
        fa.part = ptr<double>(b.part);
        fa.nset = b.adj.nset;
        fa.natoms = b.nsorted;
        fa.idx = ptr<int>(b.idx);
        fa.occ = io.occ;
        for (int k = 0; k < 3; ++k)
            fa.hc[k] = b.eck[k] + (double)aa.rc * b.vi[k] + (double)aa.jc * b.vi[3 + k] + (double)aa.mc * b.vi[6 + k];
        for (int k = 0; k < 9; ++k) fa.v[k] = b.vi[k];
        fa.grad = io.grad;
        HIPCHK(launch_adjoint_finish(fa, c->st));
    }
    return 0;
}

// Time every tile configuration on this batch at the planned slice length,
// each with one work-group per item, #CU or 2 #CU persistent work-groups
// (static item assignment), or #CU work-groups taking items from a device
// counter (longest first, each as it finishes one: the cfg 5 population's
// GEMM 2.49 -> 2.43 ms and a steadier step); then the best tile at half and
// at twice that length, with the same four launch forms.  A candidate costs its GEMM plus the
// reduction of its slice planes, whose number the slice length sets: longer
// slices mean fewer planes to write and reduce, shorter ones more, smaller
// work items to balance over the CUs.  Another length must beat the planned
// one by 2%, more than the spread of these short timings: the slice length
// changes the FP32 summation order, so a choice made on noise would change
// the results' last bits from one context to the next for nothing (on the
// 96-member population the planned length wins).
int autotune(dc_ctx *c, BatchState &b, const StepIO &io) {
    const bool fp32_only = b.prec == DC_PREC_FP32;    // tiles built without an FP32 variant are skipped
    auto built = [&](int t) {
        const TileInfo ti = gemm_tile_info(t);
        return !(fp32_only && ti.no_fp32) && !(ti.fold && !(scheme_folds(b.pl.scheme) && fold_side(b.pl.gg, b.fold_mask, t)));
    };
    // predicted cost: microseconds of the planner's model where a side can be
    // folded (the fold tiles alone are candidates then), else padded work
    const bool folds = b.pl.gg.fold != 0;
    auto candidate = [&](int t) { return built(t) && (gemm_tile_info(t).fold != 0) == folds; };
    auto cost = [&](int t) {
        GemmGeom gg = b.pl.gg;
        gg.fold = fold_side(gg, b.fold_mask, t);
        const TileInfo ti = gemm_tile_info(t);
        double us;
        if (!folds) return (double)gemm_items(gg, t) * ti.rt * ti.ct;
        (void)fold_slices(gg, t, b.segs, b.pl.scheme, us);
        return us;
    };
    if (c->tile >= 0 && built(c->tile)) b.pl.tile = c->tile;
    b.nwg = 0;
    if (c->tile >= 0 || !c->autotune || b.nslice == 0) return 0;
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, c->device));
    const int ncu = prop.multiProcessorCount;
    // mean of 2 launches after a warm-up: the GEMM of (tile, nwg), or the reduction
    auto time_ms = [&](int t, int nwg, bool reduce, float &ms) -> int {
        const bool qu = nwg < 0;
        const int n = qu ? -nwg : nwg;
        int st = reduce ? reduce_planes(c, b, io) : enqueue(c, b, io, t, n, false, STEP_GEMM, qu);
        if (st) return st;
        HIPCHK(hipEventRecord(c->ev[2], c->st));
        for (int r = 0; r < 2; ++r)
            if ((st = reduce ? reduce_planes(c, b, io) : enqueue(c, b, io, t, n, false, STEP_GEMM, qu))) return st;
        HIPCHK(hipEventRecord(c->ev[3], c->st));
        HIPCHK(hipEventSynchronize(c->ev[3]));
        HIPCHK(hipEventElapsedTime(&ms, c->ev[2], c->ev[3]));
        ms *= 0.5f;
        return 0;
    };
    float best = 1e30f, best_gemm = 0.f, red = 0.f;
    int bt = b.pl.tile, bn = 0, bk = b.kchunk;
    int st = time_ms(0, 0, true, red);
    if (st) return st;
    // candidates: tiles whose padded work is within 1.5x of the least padded
    // one, or whose predicted time is within 1.2x of the shortest
    double wmin = 1e300;
    for (int t = 0; t < gemm_num_tiles(); ++t)
        if (candidate(t)) wmin = std::min(wmin, cost(t));
    for (int t = 0; t < gemm_num_tiles(); ++t) {
        if (!candidate(t) || cost(t) > (folds ? 1.2 : 1.5) * wmin) continue;
        for (int nwg : {0, ncu, 2 * ncu, -ncu}) {
            float g = 0.f;
            if ((st = time_ms(t, nwg, false, g))) return st;
            if (g + red < best) {
                best = g + red;
                best_gemm = g;
                bt = t;
                bn = nwg;
            }
        }
    }
    // slice length, on the best tile (a forced length is kept)
    if (c->slice_atoms <= 0) {
        const int k0 = b.kchunk;
        for (int kc : {(k0 / 2 + 15) / 16 * 16, 2 * k0}) {
            if (kc < 256 || kc == k0) continue;
            if ((st = make_slices(c, b, kc))) return st;
            if ((st = time_ms(0, 0, true, red))) return st;
            for (int nwg : {0, ncu, 2 * ncu, -ncu}) {
                float g = 0.f;
                if ((st = time_ms(bt, nwg, false, g))) return st;
                if (g + red < (bk == k0 ? 0.98f : 1.0f) * best) {
                    best = g + red;
                    best_gemm = g;
                    bn = nwg;
                    bk = kc;
                }
            }
        }
        if (b.kchunk != bk && (st = make_slices(c, b, bk))) return st;
    }
    b.pl.tile = bt;
    b.queue = bn < 0;
    b.nwg = bn < 0 ? -bn : bn;
    b.tune_best_ms = best_gemm;
    return 0;
}

}  // namespace

extern "C" {

int dc_set_autotune(dc_ctx *c, int on) {
    if (!c) return DC_ERR_ARG;
    c->autotune = on ? 1 : 0;
    return DC_OK;
}

int dc_set_graphs(dc_ctx *c, int on) {
    if (!c) return DC_ERR_ARG;
    c->graphs = on ? 1 : 0;
    return DC_OK;
}

int dc_batch_info(const dc_ctx *c, int *tile, int *nwg, int *graph, double *tune_ms) {
    if (!c || !c->batch) return DC_ERR_STATE;
    if (tile) *tile = c->batch->pl.tile;
    if (nwg) *nwg = c->batch->queue ? -c->batch->nwg : c->batch->nwg;
    if (graph) *graph = c->batch->exec != nullptr;
    if (tune_ms) *tune_ms = c->batch->tune_best_ms;
    return DC_OK;
}

}  // extern "C"

namespace {

// Whether the kernels of a step may work on the caller's arrays (pointer and
// bytes of each; the first nin are inputs): memory of the context's device, and no output
// that shares bytes with another array -- the reduction writes I before it
// reads the target, several times over when the autotuner runs.
struct Span {
    const void *p;
    size_t bytes;
};
bool in_place(const dc_ctx *c, const Span *s, int n, int nin) {
    for (int x = 0; x < n; ++x) {
        if (!s[x].p || !s[x].bytes) continue;
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, s[x].p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        if (at.type != hipMemoryTypeDevice || at.device != c->device) return false;
        const uintptr_t b = (uintptr_t)s[x].p, e = b + s[x].bytes;
        for (int y = std::max(x + 1, nin); y < n; ++y)
            if (s[y].p && b < (uintptr_t)s[y].p + s[y].bytes && (uintptr_t)s[y].p < e) return false;
    }
    return true;
}

// One population step.  dev = false: pos/occ/bdw of d, target, weight, icalc
// and grad are host arrays, copied to and from the buffers that the replayed
// graph works on.  dev = true: they are device arrays, and a non-null bdw counts
// as per-atom B; the kernels of the step, launched one by one, read and write
// them in place (96 members, 1.8M atoms: the copies moved 400 MB) where in_place
// allows it, else they go through the state's buffers as host arrays do, all inputs
// copied before the first kernel and the outputs after the last.
int batch_chi2(dc_ctx *c, const dc_batch_desc *d, const double *target, const double *weight, double *chi2,
               double *icalc, double *grad, bool dev) {
    if (!c) return DC_ERR_ARG;
    c->err.clear();
    c->err_typ = DC_ER_NONE;
    int st;
    if ((st = check_desc(c, d))) return st;
    if (!target || !chi2) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "batch: null target or chi2");
    if (cancelled(c)) return set_err(c, DC_ERR_CANCEL, DC_ER_COMM, "cancelled");
    HIPCHK(hipSetDevice(c->device));
    stats_begin(c);
    const int64_t natoms = d->atom_beg[d->nmembers];
    bool any_b = dev && d->bdw != nullptr;
    if (d->bdw && !dev)
        for (int64_t k = 0; k < natoms && !any_b; ++k) any_b = d->type[k] > 0 && d->bdw[k] != 0.0;
    const bool want_grad = grad != nullptr, want_icalc = icalc != nullptr, have_weight = weight != nullptr;
    // s^2 of this call's metrics; with per-atom B the mirrored-pair tiles fold
    // a side only where every member's s^2 is mirrored about its centre
    std::vector<float> sq;
    int fold_mask = FOLD_COLS | FOLD_ROWS, top_bin = 0;
    {
        const Grid g = batch_grid(d);
        const GemmGeom gg = mapping0_geom(g);
        if ((st = member_sq(c, g, gg, d, sq, any_b || want_grad, top_bin))) return st;
        for (int m = 0; m < d->nmembers && any_b; ++m) fold_mask &= mirrored_sides(gg, sq.data() + sq.size() / d->nmembers * m);
    }
    const bool shape = same_shape(c->batch, c, d, want_grad, want_icalc, have_weight, any_b) &&
                       c->batch->fold_mask == fold_mask && cfact_rows(top_bin, d->ncfact) <= c->batch->rows;
    // Device arrays and a state of this shape: the records and the GEMM start
    // on the cached plan while the host compares the atom types with the
    // plan's (1.8M atoms: 0.5 ms) and packs the form factors; other types
    // discard what was started.  Everything that was started stays inside the
    // state's buffers, whose sizes the shape fixes.
    const size_t nd = sizeof(double), grid_bytes = nd * (size_t)d->nmembers * d->inc[0] * d->inc[1] * d->inc[2];
    const Span spans[] = {{d->pos, 3 * nd * natoms}, {d->occ, nd * natoms}, {any_b ? d->bdw : nullptr, nd * natoms},
                          {target, grid_bytes}, {weight, grid_bytes}, {icalc, grid_bytes}, {grad, 5 * nd * natoms}};
    const bool direct = dev && in_place(c, spans, 7, 5);
    const bool early = direct && shape && c->batch->primed;
    const StepIO io_dev{d->pos, d->occ, any_b ? d->bdw : nullptr, target, weight, icalc, grad};
    auto send_sq = [&](BatchState &b) -> int {
        std::memcpy(b.h_sq.p, sq.data(), sizeof(float) * sq.size());
        HIPCHK(hipMemcpyAsync(b.sq.p, b.h_sq.p, sizeof(float) * sq.size(), hipMemcpyHostToDevice, c->st));
        return 0;
    };
    if (early) {
        BatchState &b = *c->batch;
        HIPCHK(hipEventRecord(c->ev[0], c->st));
        if ((st = send_sq(b))) return st;
        HIPCHK(hipEventRecord(c->ev[4], c->st));
        if ((st = enqueue(c, b, io_dev, b.pl.tile, b.nwg, true, STEP_GEMM, b.queue))) return st;
    }
    bool fits = shape && same_types(*c->batch, d);
    if (!fits) {
        if ((st = check_types(c, d))) {
            (void)hipStreamSynchronize(c->st);
            return st;
        }
        HIPCHK(hipStreamSynchronize(c->st));
        batch_release(c);
        c->batch = new BatchState();
        c->batch->want_grad = want_grad;
        c->batch->want_icalc = want_icalc;
        c->batch->have_weight = have_weight;
        c->batch->any_b = any_b;
        c->batch->fold_mask = fold_mask;
        // a margin for the metrics of later generations
        c->batch->rows = std::min(d->ncfact, cfact_rows(top_bin, d->ncfact) + top_bin / 4 + 16);
        if ((st = build_state(c, d, *c->batch))) {
            batch_release(c);
            return st;
        }
    }
    BatchState &b = *c->batch;
    const bool started = early && fits;
    const size_t P = (size_t)b.g.P, M = (size_t)d->nmembers;
    if (!direct) {
        const size_t T = (size_t)std::max<int64_t>(natoms, 1);
        if ((st = ensure(c, b.pos, sizeof(double) * 3 * T))) return st;
        if ((st = ensure(c, b.occ, sizeof(double) * T))) return st;
        if ((st = ensure(c, b.bdw, sizeof(double) * T))) return st;
        if ((st = ensure(c, b.target, sizeof(double) * P * M))) return st;
        if (weight && (st = ensure(c, b.weight, sizeof(double) * P * M))) return st;
        if (want_icalc && (st = ensure(c, b.icalc, sizeof(double) * P * M))) return st;
        if (want_grad && (st = ensure(c, b.grad, sizeof(double) * 5 * T))) return st;
    }
    const StepIO io = direct ? io_dev : own_io(b);
    const hipMemcpyKind in = dev ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    const hipMemcpyKind out = dev ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    if (!started) {
        HIPCHK(hipEventRecord(c->ev[0], c->st));
        if (!direct) {
            HIPCHK(hipMemcpyAsync(b.pos.p, d->pos, sizeof(double) * 3 * natoms, in, c->st));
            HIPCHK(hipMemcpyAsync(b.occ.p, d->occ, sizeof(double) * natoms, in, c->st));
            if (any_b) HIPCHK(hipMemcpyAsync(b.bdw.p, d->bdw, sizeof(double) * natoms, in, c->st));
            HIPCHK(hipMemcpyAsync(b.target.p, target, sizeof(double) * P * M, in, c->st));
            if (weight) HIPCHK(hipMemcpyAsync(b.weight.p, weight, sizeof(double) * P * M, in, c->st));
        }
        if ((st = send_sq(b))) return st;
    }
    for (size_t q = 0; q < (size_t)d->nscat * M; ++q)
        std::memcpy(b.h_cf.p + sizeof(double) * 2 * b.rows * q, d->cfact + 2 * (size_t)d->ncfact * q, sizeof(double) * 2 * b.rows);
    HIPCHK(hipMemcpyAsync(b.cfact.p, b.h_cf.p, sizeof(double) * 2 * b.rows * d->nscat * M, hipMemcpyHostToDevice, c->st));
    unsigned char *h_rten = b.h_cf.p + sizeof(double) * 2 * b.rows * d->nscat * M;
    std::memcpy(h_rten, d->rten, sizeof(double) * 9 * M);
    HIPCHK(hipMemcpyAsync(b.rten.p, h_rten, sizeof(double) * 9 * M, hipMemcpyHostToDevice, c->st));

    if (!b.primed) {
        // records of this call, then the tile / grid-size choice, then the graph
        if ((st = enqueue(c, b, io, b.pl.tile, 0, true, STEP_GEMM, false))) return st;
        if ((st = autotune(c, b, io))) return st;
        b.primed = true;
    }
    if (!direct && c->graphs && !b.exec) {
        HIPCHK(hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
        st = enqueue(c, b, io, b.pl.tile, b.nwg, true, STEP_GEMM | STEP_REST, b.queue);
        hipGraph_t graph = nullptr;
        hipError_t e = hipStreamEndCapture(c->st, &graph);
        if (st) {
            if (graph) (void)hipGraphDestroy(graph);
            return st;
        }
        HIPCHK(e);
        b.graph = graph;
        HIPCHK(hipGraphInstantiate(&b.exec, b.graph, nullptr, nullptr, 0));
    }
    if (!started) HIPCHK(hipEventRecord(c->ev[4], c->st));
    if (!direct && b.exec) {
        HIPCHK(hipGraphLaunch(b.exec, c->st));
    } else {
        if ((st = enqueue(c, b, io, b.pl.tile, b.nwg, !started, started ? STEP_REST : STEP_GEMM | STEP_REST, b.queue))) return st;
    }
    HIPCHK(hipEventRecord(c->ev[5], c->st));
    if (!direct && icalc) HIPCHK(hipMemcpyAsync(icalc, b.icalc.p, sizeof(double) * P * M, out, c->st));
    if (!direct && grad) HIPCHK(hipMemcpyAsync(grad, b.grad.p, sizeof(double) * 5 * natoms, out, c->st));
    HIPCHK(hipEventRecord(c->ev[1], c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    std::memcpy(chi2, b.h_chi.p, sizeof(double) * M);
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, c->ev[4], c->ev[5]));
    c->stats.forward_ms = ms;          // the whole population step (forward + adjoint when requested)
    HIPCHK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    c->stats.total_ms = ms;
    c->stats.pairs = (double)b.nsorted * (double)P;
    c->stats.slices = b.nslice;
    c->stats.gemm_launches = 1;
    c->stats.gemm_scheme = b.pl.scheme;
    c->stats.gemm_ms = b.tune_best_ms;
    c->stats.adjoint_walk = want_grad ? b.adj.walk : 0;
    return DC_OK;
}

}  // namespace

extern "C" {

int dc_batch_chi2(dc_ctx *c, const dc_batch_desc *d, const double *target, const double *weight, double *chi2,
                  double *icalc, double *grad) {
    return batch_chi2(c, d, target, weight, chi2, icalc, grad, false);
}

int dc_batch_chi2_dev(dc_ctx *c, const dc_batch_desc *d, const double *target, const double *weight, double *chi2,
                      double *icalc, double *grad) {
    return batch_chi2(c, d, target, weight, chi2, icalc, grad, true);
}

}  // extern "C"
