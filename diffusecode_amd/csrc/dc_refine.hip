// dc_refine.hip -- C ABI of the refinement model: intensity of a structure
// with per-atom occupancies and displacement parameters, and the reverse-mode
// derivative of a loss of that intensity (include/diffuse_turbo.h).
//
// REFINE (refine/prog/refine_run.f90:491-600) differentiates the Fourier
// calculation by re-running it once per parameter; the adjoint here costs a
// small multiple of one forward pass for all 5N parameters together.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "dc_host.h"

using namespace dc;

namespace {

constexpr int CHI2_BLOCKS = 1024;
constexpr double JVP_PARTIAL_BUDGET = 4.0e9;   // bytes of slice planes per batch of directions

struct ModelPlan {
    Grid g{};
    Plan pl;
    std::vector<int> order;                   // sorted atom -> caller index
    std::vector<std::pair<int, int>> segs;    // (type 0-based, count) in sorted order
    std::vector<float> sq;                    // s^2 row parts (R) then column parts (C)
    bool separable = true;
    bool any_b = false;
    int nsorted = 0;
    int rows = 0;                             // form-factor rows the grid reaches
    // staged device copies
    const int *idx = nullptr;
    const float *d_sq = nullptr;
    const double2 *cfact = nullptr;
    const double *pos = nullptr, *occ = nullptr, *bdw = nullptr;   // caller order (staged, or the caller's device arrays)
};

double dotg(const double *a, const double *g, const double *b) {
    double s = 0.0;
    for (int r = 0; r < 3; ++r)
        for (int k = 0; k < 3; ++k) s += a[r] * g[r + 3 * k] * b[k];
    return s;
}

int check_model(dc_ctx *c, const dc_model_desc *m) {
    if (!m || !m->pos || !m->type || !m->occ || !m->cfact || m->natoms < 0 || m->nscat < 1 || m->ncfact < 1)
        return set_err(c, DC_ERR_ARG, DC_ER_LIB, "model: null pointer or bad size");
    if (m->natoms > INT32_MAX / 8) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "model: too many atoms");
    for (int k = 0; k < 3; ++k)
        if (m->inc[k] < 1) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "model: bad inc");
    for (int64_t n = 0; n < m->natoms; ++n)
        if (m->type[n] < 0 || m->type[n] > m->nscat) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "model: type outside 0..nscat");
    return 0;
}

// Grid, GEMM plan (rows = abscissa), type-sorted atom order and the s^2 parts.
// dev: pos, occ and bdw are device arrays, a non-null bdw counts as per-atom B.
int plan_model(dc_ctx *c, const dc_model_desc *m, ModelPlan &mp, bool dev) {
    Grid &g = mp.g;
    for (int k = 0; k < 3; ++k) {
        g.n[k] = g.f[k] = m->inc[k];
        g.xm[k] = m->eck[k];
        g.uin[k] = m->vi[k];
        g.vin[k] = m->vi[3 + k];
        g.win[k] = m->vi[6 + k];
    }
    for (int k = 0; k < 9; ++k) g.rten[k] = m->rten[k];
    g.P = (long long)g.f[0] * g.f[1] * g.f[2];
    const GemmGeom gg = mapping0_geom(g);

    // metric orthogonality of the abscissa against the other axes
    const double *v1 = m->vi;
    const double n1 = std::sqrt(std::fabs(dotg(v1, m->rten, v1)));
    for (int ax = 1; ax < 3; ++ax) {
        if (m->inc[ax] <= 1) continue;
        const double *v = m->vi + 3 * ax;
        const double nv = std::sqrt(std::fabs(dotg(v, m->rten, v)));
        if (std::fabs(dotg(v1, m->rten, v)) > 1e-12 * std::max(1.0, n1 * nv)) mp.separable = false;
    }
    const bool f16 = f16_scheme(model_scheme(c->prec));
    mp.sq.resize((size_t)sq_floats(gg, f16));
    split_sq(m->rten, m->eck, m->vi, gg, g.f[1], f16, mp.sq.data());

    // counting sort by type, vacancies dropped
    std::vector<int> cnt(m->nscat + 1, 0);
    for (int64_t n = 0; n < m->natoms; ++n) cnt[m->type[n]]++;
    std::vector<int> beg(m->nscat + 2, 0);
    for (int t = 1; t <= m->nscat; ++t) beg[t + 1] = beg[t] + cnt[t];
    mp.nsorted = beg[m->nscat + 1];
    mp.order.assign(mp.nsorted, 0);
    std::vector<int> fill(beg.begin(), beg.end());
    for (int64_t n = 0; n < m->natoms; ++n) {
        const int t = m->type[n];
        if (t > 0) mp.order[fill[t]++] = (int)n;
        if (!dev && t > 0 && m->bdw && m->bdw[n] != 0.0) mp.any_b = true;
    }
    if (dev) mp.any_b = m->bdw != nullptr;
    for (int t = 1; t <= m->nscat; ++t)
        if (cnt[t] > 0) mp.segs.push_back({t - 1, cnt[t]});
    // the planes of mapping 0 are the same for every tile; with per-atom B a
    // side is folded only where its s^2 is mirrored
    mp.pl = plan_gemm(g, c->tile, 0, model_scheme(c->prec), m->natoms,
                      mp.any_b ? mirrored_sides(gg, mp.sq.data()) : FOLD_COLS | FOLD_ROWS);
    if (mp.any_b && !mp.separable)
        return set_err(c, DC_ERR_ARG, DC_ER_LIB, "model: per-atom B needs vi(:,1) metric-orthogonal to vi(:,2), vi(:,3)");
    const int top_bin = max_corner_bin(g);
    if (top_bin >= m->ncfact)
        return set_err(c, DC_ERR_ISTL, DC_ER_FOUR, "sin(theta)/lambda beyond table");
    mp.rows = cfact_rows(top_bin, m->ncfact);
    return 0;
}

// Per-atom inputs and tables on the device and the GEMM records (corner phases).
int upload_model(dc_ctx *c, const dc_model_desc *m, ModelPlan &mp, bool dev) {
    int st;
    const int ns = mp.nsorted;
    const size_t n = (size_t)m->natoms;
    const double *pos = m->pos, *occ = m->occ, *bdw = m->bdw;
    if (!dev) {
        double *d_pos, *d_occ, *d_bdw = nullptr;
        if ((st = stage(c, c->m_pos, m->pos, 3 * n, d_pos))) return st;
        if ((st = stage(c, c->m_w, m->occ, n, d_occ))) return st;
        if (m->bdw && (st = stage(c, c->m_b, m->bdw, n, d_bdw))) return st;
        pos = d_pos;
        occ = d_occ;
        bdw = d_bdw;
    }
    int *d_idx;
    float *d_sq;
    double2 *d_cf;
    if ((st = stage(c, c->idx, mp.order.data(), mp.order.size(), d_idx))) return st;
    if ((st = stage(c, c->m_sq, mp.sq.data(), mp.sq.size(), d_sq))) return st;
    if ((st = stage_cfact(c, m->cfact, m->ncfact, m->nscat, mp.rows, d_cf))) return st;
    mp.idx = d_idx;
    mp.d_sq = d_sq;
    mp.cfact = d_cf;
    mp.pos = pos;
    mp.occ = occ;
    mp.bdw = bdw;
    if ((st = ensure(c, c->rec, sizeof(AtomRec) * std::max(ns, 1)))) return st;
    PrepArgs pa = base_prep(mp.g, 0);
    pa.src = pos;
    pa.src_ld = 0;
    pa.idx = mp.idx;
    pa.occ_src = occ;
    pa.bdw_src = bdw;
    pa.n = ns;
    if ((st = stage_flush(c))) return st;
    HIPCHK(launch_prep(pa, ptr<AtomRec>(c->rec), c->st));
    c->rec_hash = false;
    return 0;
}

// F (complex, device m_f) and I (device dsi) over the grid.
int model_forward(dc_ctx *c, const dc_model_desc *m, ModelPlan &mp) {
    int st;
    const GemmGeom &gg = mp.pl.gg;
    SliceSet ss;
    int off = 0;
    add_segments(ss, mp.segs, slice_len(c, kchunk_for(mp.pl, mp.segs, mp.pl.scheme)), off);
    if (ss.beg.empty()) ss.beg.push_back(0);
    const int nslice = (int)ss.type.size();
    ss.lot = {0, nslice};
    int *d_beg, *d_lot, *d_type;
    if ((st = stage(c, c->slice_beg, ss.beg.data(), ss.beg.size(), d_beg))) return st;
    if ((st = stage(c, c->lot_slice, ss.lot.data(), ss.lot.size(), d_lot))) return st;
    if ((st = stage(c, c->slice_type, ss.type.data(), ss.type.size(), d_type))) return st;
    if ((st = stage_flush(c))) return st;
    if ((st = ensure(c, c->partial, sizeof(float2) * gg.P * std::max(nslice, 1)))) return st;
    if ((st = ensure(c, c->m_f, sizeof(double) * 2 * mp.g.P))) return st;
    if ((st = ensure(c, c->dsi, sizeof(double) * mp.g.P))) return st;
    hipEvent_t e0, e1;
    if ((st = mark(c, e0))) return st;
    if ((st = run_gemm(c, mp.pl, ss.beg, d_beg, ptr<float2>(c->partial), mp.any_b ? mp.d_sq : nullptr))) return st;
    ReduceArgs ra{};
    ra.g = mp.g;
    ra.partial = ptr<float2>(c->partial);
    ra.slice0 = 0;
    ra.lot_slice = d_lot;
    ra.slice_type = d_type;
    ra.nlots = nslice > 0 ? 1 : 0;
    ra.lform = 1;
    ra.cfact = mp.cfact;
    ra.ncfact = mp.rows;
    ra.ntype = m->nscat;
    ra.dsi = ptr<double>(c->dsi);
    ra.csf = ptr<double>(c->m_f);
    ra.fresh = 1;
    if (nslice > 0) {
        HIPCHK(launch_reduce_lots(ra, c->st));
    } else {
        HIPCHK(hipMemsetAsync(c->m_f.p, 0, sizeof(double) * 2 * mp.g.P, c->st));
        HIPCHK(hipMemsetAsync(c->dsi.p, 0, sizeof(double) * mp.g.P, c->st));
    }
    if ((st = mark(c, e1))) return st;
    span(c, e0, e1, &c->stats.forward_ms);
    c->stats.pairs += (double)mp.nsorted * (double)mp.g.P;
    c->stats.slices += nslice;
    return 0;
}

// Gradient (5, natoms) on the device (grad) from F (m_f) and G (m_gi).
int model_adjoint(dc_ctx *c, const dc_model_desc *m, ModelPlan &mp, double *grad) {
    int st;
    if (!mp.separable)
        return set_err(c, DC_ERR_ARG, DC_ER_LIB, "model gradient: needs vi(:,1) metric-orthogonal to vi(:,2), vi(:,3)");
    const GemmGeom &gg = mp.pl.gg;
    const int nq = (int)mp.segs.size();
    std::vector<int> qtype(std::max(nq, 1), 0);
    for (int t = 0; t < nq; ++t) qtype[t] = mp.segs[t].first;
    // atom tiles inside one type
    const int na = adjoint_tile_atoms();
    std::vector<int> tiles;
    std::vector<int2> ranges(std::max(nq, 1), make_int2(0, 0));
    int a0 = 0;
    for (int t = 0; t < nq; ++t) {
        const int n = mp.segs[t].second;
        ranges[t] = make_int2(a0, a0 + n);
        for (int b = 0; b < n; b += na) {
            tiles.insert(tiles.end(), {a0 + b, a0 + std::min(n, b + na), t, 0});
        }
        a0 += n;
    }
    const int ntiles = (int)tiles.size() / 4;

    hipEvent_t e0, e1;
    if ((st = mark(c, e0))) return st;
    int *d_qt, *d_tiles;
    int2 *d_ranges;
    if ((st = stage(c, c->m_qt, qtype.data(), qtype.size(), d_qt))) return st;
    if ((st = stage(c, c->m_tiles, tiles.data(), tiles.size(), d_tiles))) return st;
    if ((st = stage(c, c->m_rng, ranges.data(), ranges.size(), d_ranges))) return st;
    if ((st = stage_flush(c))) return st;
    if ((st = ensure(c, c->m_q, sizeof(float2) * gg.P * std::max(nq, 1)))) return st;
    if ((st = ensure(c, c->m_ref, sizeof(float) * ranges.size()))) return st;
    if (ntiles == 0) HIPCHK(launch_adj_begin(AdjArgs{}, 0, grad, 5 * m->natoms, c->st));
    if (ntiles > 0) {
        QArgs qa{};
        qa.g = mp.g;
        qa.R = gg.R;
        qa.C = gg.C;
        qa.C0 = gg.C0;
        qa.plane = gg.P;
        qa.f = ptr<double>(c->m_f);
        qa.gi = ptr<double>(c->m_gi);
        qa.cfact = mp.cfact;
        qa.ncfact = mp.rows;
        qa.qtype = d_qt;
        qa.nq = nq;
        qa.q = ptr<float2>(c->m_q);
        HIPCHK(launch_model_q(qa, c->st));

        AdjArgs aa{};
        aa.rec = ptr<AtomRec>(c->rec);
        aa.tiles = reinterpret_cast<const int4 *>(d_tiles);
        aa.q = ptr<float2>(c->m_q);
        aa.sq = mp.d_sq;
        aa.planes_per_sq = std::max(nq, 1);
        aa.R = gg.R;
        aa.C = gg.C;
        aa.C0 = gg.C0;
        aa.f1 = mp.g.f[1];
        aa.plane = gg.P;
        aa.natoms = mp.nsorted;
        aa.rc = 0.5f * (float)(mp.g.f[0] - 1);
        aa.jc = 0.5f * (float)(mp.g.f[1] - 1);
        aa.mc = 0.5f * (float)(mp.g.f[2] - 1);
        aa.fold = !mp.any_b || (mirrored_sides(gg, mp.sq.data()) & FOLD_ROWS);
        aa.damped = mp.any_b;
        adjoint_plan(aa, ntiles, c->prec != DC_PREC_FP32, c->adj_walk);
        c->stats.adjoint_walk = aa.walk;
        if ((st = ensure(c, c->m_part, sizeof(double) * 6 * (size_t)aa.nset * std::max(mp.nsorted, 1)))) return st;
        aa.part = ptr<double>(c->m_part);
        aa.ranges = d_ranges;
        aa.ref = ptr<float>(c->m_ref);
        HIPCHK(launch_adj_begin(aa, nq, grad, 5 * m->natoms, c->st));
        const std::vector<AdjSpan> spans = adjoint_spans(aa, tiles.data(), ntiles);
        long long most = 0;
        for (const AdjSpan &s : spans) most = std::max<long long>(most, s.nplanes);
        if ((st = ensure(c, c->m_qs, sizeof(uint4) * (size_t)(aa.plane_words * most)))) return st;
        for (const AdjSpan &s : spans) HIPCHK(launch_adjoint(aa, s, ptr<uint4>(c->m_qs), c->st));

        AdjFinishArgs fa{};
        fa.part = ptr<double>(c->m_part);
        fa.nset = aa.nset;
        fa.natoms = mp.nsorted;
        fa.idx = mp.idx;
        fa.occ = mp.occ;
        for (int k = 0; k < 3; ++k)
            fa.hc[k] = m->eck[k] + (double)aa.rc * m->vi[k] + (double)aa.jc * m->vi[3 + k] + (double)aa.mc * m->vi[6 + k];
        for (int k = 0; k < 9; ++k) fa.v[k] = m->vi[k];
        fa.grad = grad;
        HIPCHK(launch_adjoint_finish(fa, c->st));
    }
    if ((st = mark(c, e1))) return st;
    span(c, e0, e1, &c->stats.adjoint_ms);
    return 0;
}

int model_begin(dc_ctx *c, const dc_model_desc *m, ModelPlan &mp, bool dev = false) {
    c->err.clear();
    c->err_typ = DC_ER_NONE;
    int st;
    if ((st = check_model(c, m))) return st;
    if (cancelled(c)) return set_err(c, DC_ERR_CANCEL, DC_ER_COMM, "cancelled");
    HIPCHK(hipSetDevice(c->device));
    stats_begin(c);
    HIPCHK(hipEventRecord(c->ev[0], c->st));
    if ((st = stage_begin(c))) return st;
    if ((st = plan_model(c, m, mp, dev))) return st;
    return upload_model(c, m, mp, dev);
}

int model_end(dc_ctx *c) {
    HIPCHK(hipEventRecord(c->ev[1], c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    c->arena_busy = false;
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    c->stats.total_ms = ms;
    return resolve_spans(c);
}

}  // namespace

extern "C" {

int dc_model_intensity(dc_ctx *c, const dc_model_desc *m, double *icalc, double *fcalc) {
    if (!c) return DC_ERR_ARG;
    ModelPlan mp;
    int st;
    if ((st = model_begin(c, m, mp))) return st;
    if ((st = model_forward(c, m, mp))) return st;
    if (icalc) HIPCHK(hipMemcpyAsync(icalc, c->dsi.p, sizeof(double) * mp.g.P, hipMemcpyDeviceToHost, c->st));
    if (fcalc) HIPCHK(hipMemcpyAsync(fcalc, c->m_f.p, sizeof(double) * 2 * mp.g.P, hipMemcpyDeviceToHost, c->st));
    return model_end(c);
}

int dc_model_vjp(dc_ctx *c, const dc_model_desc *m, const double *fcalc, const double *gi, double *grad) {
    if (!c) return DC_ERR_ARG;
    if (!fcalc || !gi || !grad) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "dc_model_vjp: null pointer");
    ModelPlan mp;
    int st;
    if ((st = model_begin(c, m, mp))) return st;
    if ((st = upload(c, c->m_f, fcalc, 2 * (size_t)mp.g.P))) return st;
    if ((st = upload(c, c->m_gi, gi, (size_t)mp.g.P))) return st;
    if ((st = ensure(c, c->m_grad, sizeof(double) * 5 * std::max<int64_t>(m->natoms, 1)))) return st;
    if ((st = model_adjoint(c, m, mp, ptr<double>(c->m_grad)))) return st;
    HIPCHK(hipMemcpyAsync(grad, c->m_grad.p, sizeof(double) * 5 * m->natoms, hipMemcpyDeviceToHost, c->st));
    return model_end(c);
}

int dc_model_jvp(dc_ctx *c, const dc_model_desc *m, const double *fcalc, int ndir, const double *dparam,
                 double *di, double *df) {
    if (!c) return DC_ERR_ARG;
    if (!fcalc || !dparam || !di || ndir < 0) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "dc_model_jvp: null pointer or bad ndir");
    ModelPlan mp;
    int st;
    if ((st = model_begin(c, m, mp))) return st;
    const GemmGeom &gg = mp.pl.gg;
    const long long P = mp.g.P;
    const int ns = mp.nsorted;
    if ((st = upload(c, c->m_f, fcalc, 2 * (size_t)P))) return st;
    // [ndir][P] dI, then dF: pinned memory that the kernel writes, or device
    const size_t obytes = sizeof(double) * (size_t)P * std::max(ndir, 1) * (df ? 3 : 1);
    const bool pinned = obytes <= HOST_OUT_BYTES;
    if ((st = pinned ? pin_ensure(c, c->h_out, obytes) : ensure(c, c->m_di, obytes))) return st;
    double *out = pinned ? reinterpret_cast<double *>(c->h_out.p) : ptr<double>(c->m_di);
    // directions per batch so that the slice planes fit the budget
    std::vector<std::pair<int, int>> all;
    for (int k = 0; k < 5 * std::min(ndir, 64); ++k) all.insert(all.end(), mp.segs.begin(), mp.segs.end());
    const int kchunk = slice_len(c, kchunk_for(mp.pl, all, mp.pl.scheme));
    long long slices_per_dir = 0;
    for (auto &sg : mp.segs) slices_per_dir += 5 * ((sg.second + kchunk - 1) / kchunk);
    const double dir_bytes = (double)std::max<long long>(slices_per_dir, 1) * gg.P * sizeof(float2);
    const int per = std::max(1, std::min(ndir, (int)(JVP_PARTIAL_BUDGET / dir_bytes)));
    HIPCHK(hipEventRecord(c->ev[4], c->st));
    for (int d0 = 0; d0 < ndir; d0 += per) {
        if (cancelled(c)) return set_err(c, DC_ERR_CANCEL, DC_ER_COMM, "cancelled");
        const int nd = std::min(per, ndir - d0);
        SliceSet ss;
        std::vector<int> dsl;
        int off = 0;
        for (int g5 = 0; g5 < 5 * nd; ++g5) {
            dsl.push_back((int)ss.type.size());
            add_segments(ss, mp.segs, kchunk, off);
        }
        dsl.push_back((int)ss.type.size());
        if (ss.beg.empty()) ss.beg.push_back(0);
        const int nslice = (int)ss.type.size();
        const long long nrec = 5LL * nd * ns;
        double *d_par;
        int *d_dsl, *d_beg, *d_type;
        if ((st = stage(c, c->m_jw, dparam + 5 * (size_t)m->natoms * d0, 5 * (size_t)m->natoms * nd, d_par))) return st;
        if ((st = stage(c, c->m_dsl, dsl.data(), dsl.size(), d_dsl))) return st;
        if ((st = stage(c, c->slice_beg, ss.beg.data(), ss.beg.size(), d_beg))) return st;
        if ((st = stage(c, c->slice_type, ss.type.data(), ss.type.size(), d_type))) return st;
        if ((st = stage_flush(c))) return st;
        if ((st = ensure(c, c->rec, sizeof(AtomRec) * (size_t)std::max<long long>(nrec, 1)))) return st;
        if ((st = ensure(c, c->partial, sizeof(float2) * gg.P * std::max(nslice, 1)))) return st;
        PrepArgs pa = base_prep(mp.g, 0);
        pa.src = mp.pos;
        pa.src_ld = 0;
        pa.idx = mp.idx;
        pa.occ_src = mp.occ;
        pa.bdw_src = mp.bdw;
        pa.dpar = d_par;
        pa.dn = std::max(ns, 1);
        pa.dnat = m->natoms;
        pa.n = nrec;
        if (pa.n > 0) HIPCHK(launch_prep(pa, ptr<AtomRec>(c->rec), c->st));
        c->rec_hash = false;
        if ((st = run_gemm(c, mp.pl, ss.beg, d_beg, ptr<float2>(c->partial), mp.any_b ? mp.d_sq : nullptr))) return st;
        JvpArgs ja{};
        ja.g = mp.g;
        ja.partial = ptr<float2>(c->partial);
        ja.dslice = d_dsl;
        ja.slice_type = d_type;
        ja.cfact = mp.cfact;
        ja.ncfact = mp.rows;
        ja.f = ptr<double>(c->m_f);
        ja.ndir = nd;
        ja.di = out + (size_t)d0 * P;
        ja.df = df ? out + (size_t)ndir * P + 2 * (size_t)d0 * P : nullptr;
        HIPCHK(launch_jvp_reduce(ja, c->st));
        c->stats.pairs += (double)nrec * (double)P;
        c->stats.slices += nslice;
    }
    HIPCHK(hipEventRecord(c->ev[5], c->st));
    if (ndir > 0 && !pinned) {
        HIPCHK(hipMemcpyAsync(di, out, sizeof(double) * (size_t)P * ndir, hipMemcpyDeviceToHost, c->st));
        if (df)
            HIPCHK(hipMemcpyAsync(df, out + (size_t)ndir * P, sizeof(double) * 2 * (size_t)P * ndir, hipMemcpyDeviceToHost, c->st));
    }
    if ((st = model_end(c))) return st;
    if (pinned) {
        std::memcpy(di, out, sizeof(double) * (size_t)P * ndir);
        if (df) std::memcpy(df, out + (size_t)ndir * P, sizeof(double) * 2 * (size_t)P * ndir);
    }
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, c->ev[4], c->ev[5]));
    c->stats.forward_ms = ms;
    return DC_OK;
}

// dev: the per-atom arrays of m, target, weight, icalc and grad are device
// arrays, read and written in place.
static int model_chi2(dc_ctx *c, const dc_model_desc *m, const double *target, const double *weight, double *chi2,
                      double *icalc, double *grad, bool dev) {
    if (!c) return DC_ERR_ARG;
    if (!target || !chi2) return set_err(c, DC_ERR_ARG, DC_ER_LIB, "dc_model_chi2: null pointer");
    ModelPlan mp;
    int st;
    if ((st = model_begin(c, m, mp, dev))) return st;
    if ((st = model_forward(c, m, mp))) return st;
    const long long P = mp.g.P;
    if ((st = ensure(c, c->m_gi, sizeof(double) * P))) return st;
    const double *d_t = target, *d_w = weight;
    if (!dev) {
        if ((st = ensure(c, c->w, sizeof(double) * 2 * P))) return st;
        double *t = ptr<double>(c->w);
        HIPCHK(hipMemcpyAsync(t, target, sizeof(double) * P, hipMemcpyHostToDevice, c->st));
        if (weight) HIPCHK(hipMemcpyAsync(t + P, weight, sizeof(double) * P, hipMemcpyHostToDevice, c->st));
        d_t = t;
        d_w = weight ? t + P : nullptr;
    }
    // the blocks' sums come back through pinned memory
    if ((st = pin_ensure(c, c->h_out, sizeof(double) * CHI2_BLOCKS))) return st;
    double *sums = reinterpret_cast<double *>(c->h_out.p);
    HIPCHK(launch_chi2_resid(ptr<double>(c->dsi), d_t, d_w, P, ptr<double>(c->m_gi), sums, CHI2_BLOCKS, c->st));
    if (icalc)
        HIPCHK(hipMemcpyAsync(icalc, c->dsi.p, sizeof(double) * P, dev ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, c->st));
    if (grad) {
        double *d_grad = grad;
        if (!dev) {
            if ((st = ensure(c, c->m_grad, sizeof(double) * 5 * std::max<int64_t>(m->natoms, 1)))) return st;
            d_grad = ptr<double>(c->m_grad);
        }
        if ((st = model_adjoint(c, m, mp, d_grad))) return st;
        if (!dev) HIPCHK(hipMemcpyAsync(grad, d_grad, sizeof(double) * 5 * m->natoms, hipMemcpyDeviceToHost, c->st));
    }
    if ((st = model_end(c))) return st;
    double s = 0.0;
    for (int k = 0; k < CHI2_BLOCKS; ++k) s += sums[k];
    *chi2 = s;
    return DC_OK;
}

int dc_model_chi2(dc_ctx *c, const dc_model_desc *m, const double *target, const double *weight, double *chi2,
                  double *icalc, double *grad) {
    return model_chi2(c, m, target, weight, chi2, icalc, grad, false);
}

int dc_model_chi2_dev(dc_ctx *c, const dc_model_desc *m, const double *target, const double *weight, double *chi2,
                      double *icalc, double *grad) {
    return model_chi2(c, m, target, weight, chi2, icalc, grad, true);
}

}  // extern "C"
