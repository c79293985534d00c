// Host side of the C ABI (include/aimdhf.h): plan state, device buffers,
// launch sequencing. Compiled with hipcc together with the kernels.

#include "../../include/aimdhf.h"
#include "aimdhf_internal.h"
#include "jk_digest.h"
#include "scf_small.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <vector>

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

struct HipError {
    int code;
};

#define HIPCHECK(x)                                                                  \
    do {                                                                             \
        hipError_t e_ = (x);                                                         \
        if (e_ != hipSuccess) {                                                      \
            g_err = std::string(#x) + ": " + hipGetErrorString(e_);                  \
            throw HipError{e_ == hipErrorOutOfMemory ? AIMDHF_E_NOMEM : AIMDHF_E_HIP}; \
        }                                                                            \
    } while (0)

// Device buffer that grows on demand and is freed with the plan.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    // grows with 1/8 slack: per-geometry sizes drift along a trajectory, and each
    // reallocation (hipFree synchronises the device) would stall the pipeline
    void ensure(size_t n) {
        if (n <= bytes) return;
        if (p) HIPCHECK(hipFree(p));
        p = nullptr;
        bytes = 0;
        const size_t want = std::max<size_t>(n + n / 8, 256);
        HIPCHECK(hipMalloc(&p, want));
        bytes = want;
    }
    void release() {
        if (p) hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    template <class T>
    T* as() const { return (T*)p; }
};

template <class T>
void upload(DevBuf& b, const std::vector<T>& v) {
    b.ensure(sizeof(T) * std::max<size_t>(v.size(), 1));
    if (!v.empty()) HIPCHECK(hipMemcpy(b.p, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice));
}

int ncart(int l) { return (l + 1) * (l + 2) / 2; }
int nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
constexpr int NQCLASS = 21;
constexpr int REC_HDR = 8;
// single molecules up to nset nao^2 of this digest all classes in one or two launches:
// measured per build against 21 launches, (1, 19 AOs) 30 : 174 us, (1, 114) 93 : 187,
// (2, 100) 128 : 169, (1, 152) 175 : 219; past it the per-class kernels' own thread counts
// and two densities at once win
constexpr int SMALL_JK = 200 * 200;

// Boys grid table F_n(k/10), n < 43 (aimd/qc/boys.py:57-75): series for the
// highest order, then the downward recursion.
std::vector<double> boys_table() {
    const int NG = 402, NR = 43, top = NR - 1;
    std::vector<double> tab((size_t)NG * NR);
    std::vector<double> col(NR);
    for (int k = 0; k < NG; ++k) {
        double x = k * 0.1;
        double term = 1.0 / (2 * top + 1), total = term;
        for (int m = 1; m < 400; ++m) {
            term = term * (2.0 * x) / (double)(2 * top + 2 * m + 1);
            total += term;
        }
        double ex = std::exp(-x);
        col[top] = ex * total;
        for (int n = top - 1; n >= 0; --n) col[n] = (2.0 * x * col[n + 1] + ex) / (double)(2 * n + 1);
        for (int n = 0; n < NR; ++n) tab[(size_t)k * NR + n] = col[n];
    }
    return tab;
}

// Optional per-launch timing with HIP events on the caller's stream.
// Kinds as listed at aimdhf_profile_enable in aimdhf.h.
struct Profiler {
    static constexpr int NKIND = 119;
    bool on = false;
    struct Rec {
        int kind;
        hipEvent_t a, b;
    };
    std::vector<hipEvent_t> pool;
    std::vector<Rec> recs;
    double ms[NKIND] = {0};
    long long n[NKIND] = {0};
    hipEvent_t get() {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e;
        HIPCHECK(hipEventCreate(&e));
        return e;
    }
    template <class F>
    void time(int kind, hipStream_t st, F&& launch) {
        if (!on) {
            launch();
            return;
        }
        Rec r{kind, get(), get()};
        HIPCHECK(hipEventRecord(r.a, st));
        launch();
        HIPCHECK(hipEventRecord(r.b, st));
        recs.push_back(r);
    }
    void collect() {
        for (Rec& r : recs) {
            HIPCHECK(hipEventSynchronize(r.b));
            float t = 0.0f;
            HIPCHECK(hipEventElapsedTime(&t, r.a, r.b));
            ms[r.kind] += t;
            n[r.kind] += 1;
            pool.push_back(r.a);
            pool.push_back(r.b);
        }
        recs.clear();
    }
    // host wall-clock phase (milliseconds since t0), recorded when enabled
    using clock = std::chrono::steady_clock;
    void host(int kind, clock::time_point t0) {
        if (!on) return;
        ms[kind] += std::chrono::duration<double, std::milli>(clock::now() - t0).count();
        n[kind] += 1;
    }
    void reset() {
        collect();
        for (int i = 0; i < NKIND; ++i) { ms[i] = 0.0; n[i] = 0; }
    }
    ~Profiler() {
        for (Rec& r : recs) { (void)hipEventDestroy(r.a); (void)hipEventDestroy(r.b); }
        for (hipEvent_t e : pool) (void)hipEventDestroy(e);
    }
};

// Fan-out of independent launches over the caller's stream and NAUX extra
// streams (default priority, created on first use): fork() makes the extra
// streams wait for the caller's work so far, on(i) picks a stream round-robin,
// join() makes the caller's stream wait for everything launched on them.
struct Fan {
    static constexpr int NAUX = 3;
    hipStream_t aux[NAUX] = {};
    hipEvent_t fork_ev = nullptr, join_ev[NAUX] = {};
    hipStream_t base = nullptr;
    bool serial = false;        // every launch on the caller's stream
    void init() {
        if (fork_ev) return;
        for (int i = 0; i < NAUX; ++i) {
            HIPCHECK(hipStreamCreateWithFlags(&aux[i], hipStreamNonBlocking));
            HIPCHECK(hipEventCreateWithFlags(&join_ev[i], hipEventDisableTiming));
        }
        HIPCHECK(hipEventCreateWithFlags(&fork_ev, hipEventDisableTiming));
    }
    // whether st records a graph, into which the auxiliary streams are not drawn
    static bool capturing(hipStream_t st) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        HIPCHECK(hipStreamIsCapturing(st, &status));
        return status != hipStreamCaptureStatusNone;
    }
    void fork(hipStream_t st) {
        base = st;
        if (serial) return;
        init();
        HIPCHECK(hipEventRecord(fork_ev, st));
        for (int i = 0; i < NAUX; ++i) HIPCHECK(hipStreamWaitEvent(aux[i], fork_ev, 0));
    }
    hipStream_t on(int i) const { return serial || i % (NAUX + 1) == 0 ? base : aux[i % (NAUX + 1) - 1]; }
    void join() {
        if (serial) return;
        for (int i = 0; i < NAUX; ++i) {
            HIPCHECK(hipEventRecord(join_ev[i], aux[i]));
            HIPCHECK(hipStreamWaitEvent(base, join_ev[i], 0));
        }
    }
    ~Fan() {
        for (int i = 0; i < NAUX; ++i) {
            if (aux[i]) (void)hipStreamDestroy(aux[i]);
            if (join_ev[i]) (void)hipEventDestroy(join_ev[i]);
        }
        if (fork_ev) (void)hipEventDestroy(fork_ev);
    }
};

// The streams of the six one-electron pair classes: all the caller's, or the heaviest
// classes (d d, d p, d s) apart on the fan's, since each is a chain of a few hundred
// microseconds in small molecules whose classes do not fill the card
struct PairStreams {
    hipStream_t on[6];
    explicit PairStreams(hipStream_t st) { std::fill(on, on + 6, st); }
    explicit PairStreams(const Fan& fan) {
        for (int c = 0; c < 6; ++c) on[c] = fan.on(5 - c);
    }
};

}  // namespace

struct aimdhf_plan {
    Profiler prof;
    Fan fan;
    int natm = 0, nshell = 0, nao = 0, npair = 0, nblock = 0, nbpair = 0, lmax = 0;
    std::vector<int> shell_atom, shell_l, shell_prim, shell_ao, shell_block;
    std::vector<double> prim_exp, prim_coef, charges, pos;
    std::vector<int> pair_a, pair_b, pair_cls, rec_size, cls_pairs, cls_pair_off, ncls;
    std::vector<long long> rec_off;
    std::vector<int> bp_off, bp_list;
    long long rec_total = 0;
    bool have_geometry = false;
    double threshold = 0.0;
    std::vector<long long> qcount;   // per class
    std::vector<long long> q64count; // per class, quartets with q_P q_Q >= the FP32 switch (listed first)
    long long qtotal = 0;

    DevBuf d_shell_atom, d_shell_l, d_shell_prim, d_shell_ao, d_prim_exp, d_prim_coef, d_pos;
    DevBuf d_pair_a, d_pair_b, d_pair_cls, d_rec_size, d_rec_off, d_cls_pairs, d_cls_pair_off, d_ncls;
    DevBuf d_bp_off, d_bp_list, d_boys;
    DevBuf d_recs, d_npp, d_qshell, d_qblock, d_qscr, d_counts, d_offsets, d_list;
    DevBuf d_fx, d_dsym, d_charges, d_glist, d_gfx, d_gden, d_scratch;
    std::vector<long long> gcount;
    // integral store: mode (0 auto, 1 direct, 2 store), byte limit (0: half the free device memory)
    int jk_mode = 0;
    long long store_limit = 0;
    bool stored = false;
    long long store_bytes = 0;
    // ranked pairs (jk_digest.h): component base of every pair class, the quartet list's
    // runs, and the byte offset of every class's FP64 and FP32 blocks in the store
    long long koff[7] = {0}, npao = 0, runbase[NQCLASS + 1] = {0};
    int list_parts = 1;
    int nheavy[6] = {0};            // leading ranks of each class with ERI_HEAVY primitive pairs or more
    long long h64count[NQCLASS] = {0}, h32count[NQCLASS] = {0};
    long long list_off[NQCLASS + 1] = {0}, base64[NQCLASS] = {0}, base32[NQCLASS] = {0};
    size_t store_need = 0;
    int lds_limit = 65536;
    DevBuf d_oab, d_rank_rep, d_rep_shell, d_seg, d_rq, d_gcell, d_lcnt, d_loff, d_lsum, d_lbra, d_lket;
    DevBuf d_dket, d_kacc, d_jacc, d_dcell, d_geo;
    aimdhf::DigestArgs last_dig[NQCLASS];
    DevBuf d_gkeep, d_gsel, d_nsel, d_gblk;
    // precision: 0 FP64 everywhere; 1 mixed (FP32 below the switches)
    int precision = 0;
    double jk_switch = 0.0, grad_switch = 0.0;
    DevBuf d_store;
    // least quartets a workgroup of the J/K digestion takes from a long run
    int unit_items = 1024;
    DevBuf d_gdmax;                 // per shell pair density maxima for the gradient screening
    long long* h_pin = nullptr;     // pinned host words for the totals and the error flag
    // batched plans: independent molecules (replicas) sharing one plan; shells and
    // atoms grouped by replica, pairs and quartets only within a replica, matrices
    // in the padded layout (replica r's ld x ld block at r ld^2)
    bool batched = false;
    int nrep = 1, bld = 0;
    int batch_jk_lanes = 64;        // batched J/K digestion: four threads per lane of this and workgroup
    std::vector<int> rep_shell, rep_atom, rep_nao, shell_rep, shell_first, shell_pair0, pair_lo;
    long long tens_total = 0;       // elements of one dense n_r^4 tensor per replica, none of which exists (aimdhf_batch_layout)
    DevBuf d_shell_rep, d_shell_first, d_shell_pair0, d_pair_lo, d_rep_atom, d_rep_nao;
    // elements of one stack of matrices (nao^2, or nrep ld^2 for a batch)
    size_t mat_elems() const { return batched ? (size_t)nrep * bld * bld : (size_t)nao * nao; }
    // device address and size of the fixed scratch array of the allocation-free
    // entry point on this plan's device (resolved at plan creation)
    void* noalloc_ptr = nullptr;
    size_t noalloc_bytes = 0;
    // runtime-l path (a shell with l = 3 or 4): every shell pair i >= j in index
    // order; the energy quartets in d_list / qtotal, the last gradient list in
    // d_glist / gen_gq; bounds per shell pair in d_qshell, per block pair in d_qblock
    bool have_last_store = false;   // last_dig holds a build at the current geometry
    bool generic = false;
    std::vector<int> gpair_i, gpair_j, gpair_bp, gen_npp;
    std::vector<double> gen_qb;
    long long gen_gq = 0;
    DevBuf d_gpair_i, d_gpair_j;

    aimdhf::GenArgs gen_args() const {
        aimdhf::GenArgs g{};
        g.nao = nao;
        g.natm = natm;
        g.nset = 1;
        g.shell_atom = d_shell_atom.as<int>();
        g.shell_l = d_shell_l.as<int>();
        g.shell_prim = d_shell_prim.as<int>();
        g.shell_ao = d_shell_ao.as<int>();
        g.prim_exp = d_prim_exp.as<double>();
        g.prim_coef = d_prim_coef.as<double>();
        g.pos = d_pos.as<double>();
        g.charges = d_charges.as<double>();
        g.boys = d_boys.as<double>();
        g.pair_i = d_gpair_i.as<int>();
        g.pair_j = d_gpair_j.as<int>();
        g.q = d_qshell.as<double>();
        return g;
    }

    // unique shell quartets (P >= Q) whose block-pair bounds give q_P q_Q >= thr, the
    // heaviest first, into dst; returns their number
    long long gen_build_list(double thr, DevBuf& dst) {
        std::vector<int> ord(npair);
        for (int i = 0; i < npair; ++i) ord[i] = i;
        std::stable_sort(ord.begin(), ord.end(),
                         [&](int a, int b) { return gen_qb[gpair_bp[a]] > gen_qb[gpair_bp[b]]; });
        std::vector<int2> out;
        for (int x = 0; x < npair; ++x) {
            const double qa = gen_qb[gpair_bp[ord[x]]];
            for (int y = 0; y < npair; ++y) {
                if (!(qa * gen_qb[gpair_bp[ord[y]]] >= thr)) break;
                const int P = ord[x], Q = ord[y];
                if (P >= Q) out.push_back(make_int2(P, Q));
            }
        }
        auto cost = [&](const int2& q) {
            const int a = gpair_i[q.x], b = gpair_j[q.x], c = gpair_i[q.y], d = gpair_j[q.y];
            const long long np = (long long)gen_npp[q.x] * gen_npp[q.y];
            return np * ncart(shell_l[a]) * ncart(shell_l[b]) * ncart(shell_l[c]) * ncart(shell_l[d]);
        };
        std::stable_sort(out.begin(), out.end(), [&](const int2& a, const int2& b) { return cost(a) > cost(b); });
        upload(dst, out);
        return (long long)out.size();
    }

    ~aimdhf_plan() {
        for (DevBuf* b : {&d_shell_atom, &d_shell_l, &d_shell_prim, &d_shell_ao, &d_prim_exp, &d_prim_coef,
                          &d_pos, &d_pair_a, &d_pair_b, &d_pair_cls, &d_rec_size, &d_rec_off, &d_cls_pairs,
                          &d_cls_pair_off, &d_ncls, &d_bp_off, &d_bp_list, &d_boys, &d_recs, &d_npp,
                          &d_qshell, &d_qblock, &d_qscr, &d_counts, &d_offsets, &d_list, &d_fx, &d_dsym,
                          &d_charges, &d_glist, &d_gfx, &d_gden, &d_scratch, &d_store, &d_oab, &d_rank_rep, &d_rep_shell,
                          &d_seg, &d_rq, &d_gcell, &d_lcnt, &d_loff, &d_lsum, &d_lbra, &d_lket, &d_dket, &d_kacc,
                          &d_jacc, &d_dcell, &d_geo, &d_gkeep, &d_gsel, &d_nsel, &d_gblk,
                          &d_gdmax, &d_shell_rep, &d_shell_first,
                          &d_shell_pair0, &d_pair_lo, &d_rep_atom, &d_rep_nao,
                          &d_gpair_i, &d_gpair_j})
            b->release();
        if (h_pin) (void)hipHostFree(h_pin);
    }

    aimdhf::PairArgs pair_args() const {
        aimdhf::PairArgs g;
        g.npair = npair;
        g.nbpair = nbpair;
        g.pair_a = d_pair_a.as<int>();
        g.pair_b = d_pair_b.as<int>();
        g.pair_cls = d_pair_cls.as<int>();
        g.shell_l = d_shell_l.as<int>();
        g.shell_atom = d_shell_atom.as<int>();
        g.shell_prim = d_shell_prim.as<int>();
        g.prim_exp = d_prim_exp.as<double>();
        g.prim_coef = d_prim_coef.as<double>();
        g.pos = d_pos.as<double>();
        g.rec_off = d_rec_off.as<long long>();
        g.rec_size = d_rec_size.as<int>();
        g.recs = d_recs.as<double>();
        g.npp = d_npp.as<int>();
        g.cls_pairs = d_cls_pairs.as<int>();
        g.cls_pair_off = d_cls_pair_off.as<int>();
        g.ncls_pairs = d_ncls.as<int>();
        g.qshell = d_qshell.as<double>();
        g.qblock = d_qblock.as<double>();
        g.qscr = d_qscr.as<double>();
        g.bp_off = d_bp_off.as<int>();
        g.bp_list = d_bp_list.as<int>();
        g.boys = d_boys.as<double>();
        g.pair_lo = batched ? d_pair_lo.as<int>() : nullptr;
        return g;
    }

    // List of unique shell quartets with q_P q_Q >= thr into buf, binned by class and cost;
    // counts[k] receives the per-class sizes. Synchronises the stream.
    void build_list(double thr, DevBuf& buf, std::vector<long long>& counts, hipStream_t st) {
        aimdhf::PairArgs g = pair_args();
        const int nb = aimdhf::NCOSTBIN, nv = NQCLASS * nb;
        d_counts.ensure(sizeof(int) * (size_t)npair * nv);
        d_offsets.ensure(sizeof(long long) * ((size_t)npair * nv + 2 * nv));
        long long* offs = d_offsets.as<long long>();
        long long* totals = offs + (size_t)npair * nv;
        long long* base = totals + nv;
        aimdhf::launch_count_quartets(g, thr, d_counts.as<int>(), offs, totals, base, st);
        HIPCHECK(hipGetLastError());
        std::vector<long long> tot(nv);
        HIPCHECK(hipMemcpyAsync(tot.data(), totals, sizeof(long long) * nv, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        counts.assign(NQCLASS, 0);
        long long total = 0;
        for (int k = 0; k < NQCLASS; ++k)
            for (int b = 0; b < nb; ++b) counts[k] += tot[k * nb + b];
        for (long long c : counts) total += c;
        buf.ensure(sizeof(int2) * std::max<long long>(total, 1));
        aimdhf::launch_fill_quartets(g, thr, offs, base, buf.as<int2>(), st);
        HIPCHECK(hipGetLastError());
    }

    int matrix_ld() const { return batched ? bld : nao; }

    // Screened quartets of the current geometry (quartet_list.hip): rank-ordered
    // screening values, runs of kets per bra and class, totals to the host.
    // Synchronises the stream.
    void build_quartets(double thr, double sw, hipStream_t st) {
        if (!h_pin) HIPCHECK(hipHostMalloc((void**)&h_pin, sizeof(long long) * 128 + sizeof(aimdhf::DigestGeo) * NQCLASS));
        aimdhf::GeoArgs g;
        g.nshell = nshell;
        g.npair = npair;
        g.shell_l = d_shell_l.as<int>();
        g.shell_rep = batched ? d_shell_rep.as<int>() : nullptr;
        g.shell_first = batched ? d_shell_first.as<int>() : nullptr;
        g.shell_pair0 = batched ? d_shell_pair0.as<int>() : nullptr;
        g.rep_shell = batched ? d_rep_shell.as<int>() : nullptr;
        g.cls_pairs = d_cls_pairs.as<int>();
        g.qscr = d_qscr.as<double>();
        g.rq = d_rq.as<double>();
        g.gcell = d_gcell.as<unsigned long long>();
        g.nrep = nrep;
        aimdhf::launch_geo_bounds(g, st);
        list_parts = sw > 0.0 ? 2 : 1;
        long long runs = 0;
        for (int k = 0; k < NQCLASS; ++k) {
            runbase[k] = runs;
            runs += (long long)list_parts * ncls[bra_class(k)];
        }
        runbase[NQCLASS] = runs;
        const long long cells = runs * aimdhf::LIST_WAVES;
        d_lcnt.ensure(sizeof(long long) * cells);
        d_loff.ensure(sizeof(long long) * (cells + 1));
        d_lsum.ensure(sizeof(long long) * (aimdhf::list_scan_blocks(cells) + 128));
        long long* picked = d_lsum.as<long long>() + aimdhf::list_scan_blocks(cells);
        aimdhf::QListArgs la;
        la.npair = npair;
        la.nrep = nrep;
        la.nparts = list_parts;
        la.thr = thr;
        la.sw = sw;
        for (int c = 0; c < 7; ++c) la.cls_off[c] = cls_pair_off[c];
        for (int k = 0; k < NQCLASS; ++k) la.runbase[k] = runbase[k];
        la.seg = d_seg.as<int>();
        la.rank_rep = batched ? d_rank_rep.as<int>() : nullptr;
        la.rq = d_rq.as<double>();
        la.cnt = d_lcnt.as<long long>();
        la.off = d_loff.as<long long>();
        la.lbra = la.lket = nullptr;
        aimdhf::launch_qlist_count(la, st);
        aimdhf::launch_list_scan(la.cnt, d_loff.as<long long>(), cells, d_lsum.as<long long>(), st);
        aimdhf::PickArgs pk;
        pk.n = 0;
        for (int k = 0; k < NQCLASS; ++k) {
            pk.at[pk.n++] = runbase[k] * aimdhf::LIST_WAVES;
            pk.at[pk.n++] = (runbase[k] + ncls[bra_class(k)]) * aimdhf::LIST_WAVES;
        }
        pk.at[pk.n++] = cells;
        // where each part's contracted bras end
        for (int k = 0; k < NQCLASS; ++k)
            for (int part = 0; part < list_parts; ++part)
                pk.at[pk.n++] = (runbase[k] + (long long)part * ncls[bra_class(k)] + nheavy[bra_class(k)]) *
                                aimdhf::LIST_WAVES;
        aimdhf::launch_pick(pk, d_loff.as<long long>(), picked, st);
        HIPCHECK(hipGetLastError());
        HIPCHECK(hipMemcpyAsync(h_pin, picked, sizeof(long long) * pk.n, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        qcount.assign(NQCLASS, 0);
        q64count.assign(NQCLASS, 0);
        for (int k = 0; k < NQCLASS; ++k) {
            list_off[k] = h_pin[2 * k];
            q64count[k] = h_pin[2 * k + 1] - h_pin[2 * k];
            qcount[k] = h_pin[2 * k + 2] - h_pin[2 * k];
        }
        qtotal = list_off[NQCLASS] = h_pin[2 * NQCLASS];
        for (int k = 0; k < NQCLASS; ++k) {
            const long long* h = h_pin + 2 * NQCLASS + 1 + list_parts * k;
            h64count[k] = h[0] - list_off[k];
            h32count[k] = list_parts == 2 ? h[1] - list_off[k] - q64count[k] : 0;
        }
        d_lbra.ensure(sizeof(int) * std::max<long long>(qtotal, 1));
        d_lket.ensure(sizeof(int) * std::max<long long>(qtotal, 1));
        la.lbra = d_lbra.as<int>();
        la.lket = d_lket.as<int>();
        if (qtotal) aimdhf::launch_qlist_fill(la, st);
        HIPCHECK(hipGetLastError());
        // the store's layout: per class its FP64 blocks, then its FP32 blocks, in tiles of 64 quartets
        size_t b = 0;
        for (int k = 0; k < NQCLASS; ++k) {
            const size_t blk = (size_t)aimdhf::store_block(k);
            base64[k] = (long long)b;
            b += sizeof(double) * ((q64count[k] + 63) / 64 * 64) * blk;
            base32[k] = (long long)b;
            b += sizeof(float) * ((qcount[k] - q64count[k] + 63) / 64 * 64) * blk;
        }
        store_need = b;
    }

    static int bra_class(int k) {
        int hi = 0;
        while ((hi + 1) * (hi + 2) / 2 <= k) ++hi;
        return hi;
    }
    static int ket_class(int k) { return k - bra_class(k) * (bra_class(k) + 1) / 2; }

    // Evaluate the screened quartets into the store.
    void build_store(hipStream_t st) {
        d_store.ensure(std::max<size_t>(store_need, 1));
        fan.fork(st);
        for (int k = 0, i = 0; k < NQCLASS; ++k) {
            if (!qcount[k]) continue;
            const aimdhf::EriArgs ea = eri_args(k, list_off[k]);
            hipStream_t s2 = fan.on(i++);
            prof.time(47, s2, [&] { aimdhf::launch_eri(k, ea, q64count[k], h64count[k], qcount[k] - q64count[k], h32count[k], s2); });
        }
        fan.join();
        HIPCHECK(hipGetLastError());
        // the digestion's view of the store (the stream was synchronised when the list was
        // built: no earlier copy from this pinned block is pending)
        aimdhf::DigestGeo* geo = (aimdhf::DigestGeo*)(h_pin + 128);
        for (int k = 0; k < NQCLASS; ++k) {
            geo[k].t64 = list_off[k];
            geo[k].t32 = list_off[k] + q64count[k];
            geo[k].lo64 = geo[k].t64;
            geo[k].hi64 = geo[k].t32;
            geo[k].lo32 = geo[k].t32;
            geo[k].hi32 = list_off[k] + qcount[k];
            geo[k].off = d_loff.as<long long>() + runbase[k] * aimdhf::LIST_WAVES;
            geo[k].lket = d_lket.as<int>();
            geo[k].s64 = (const double*)(d_store.as<char>() + base64[k]);
            geo[k].s32 = (const float*)(d_store.as<char>() + base32[k]);
        }
        d_geo.ensure(sizeof(aimdhf::DigestGeo) * NQCLASS);
        HIPCHECK(hipMemcpyAsync(d_geo.p, geo, sizeof(aimdhf::DigestGeo) * NQCLASS, hipMemcpyHostToDevice, st));
        store_bytes = (long long)store_need + 8 * qtotal;
        ensure_digest(1);
    }

    // Direct mode: the list cut into pieces whose integrals fit a bounded buffer; a J/K build
    // evaluates and digests piece by piece. Cuts lie between the runs of a class (a lane sums its
    // share of a whole run in FP64 before it is rounded), and a piece is evaluated from the start of
    // the tile that its first run begins in (up to 63 quartets again), so neither a quartet's
    // arithmetic nor a sum depends on where the cuts lie: J and K do not depend on the buffer's size.
    struct Piece {
        long long base[NQCLASS], lo[NQCLASS], hi[NQCLASS];     // evaluated from base, digested from lo
        size_t at[NQCLASS];
    };
    std::vector<Piece> pieces;
    void build_direct(hipStream_t st) {
        size_t fr = 0, tot = 0;
        HIPCHECK(hipMemGetInfo(&fr, &tot));
        size_t cap = std::min<size_t>((size_t)1 << 30, std::max<size_t>(fr / 8 + d_store.bytes, (size_t)1 << 20));
        if (store_limit > 0) cap = std::min<size_t>(cap, std::max<size_t>((size_t)store_limit, (size_t)1 << 26));
        // first quartet of every run, where the list does not fit as a whole
        std::vector<long long> starts;
        if (store_need > cap) {
            starts.resize(runbase[NQCLASS]);
            aimdhf::launch_run_starts(d_loff.as<long long>(), runbase[NQCLASS], d_lcnt.as<long long>(), st);
            HIPCHECK(hipGetLastError());
            HIPCHECK(hipMemcpyAsync(starts.data(), d_lcnt.p, sizeof(long long) * starts.size(), hipMemcpyDeviceToHost, st));
            HIPCHECK(hipStreamSynchronize(st));
        }
        pieces.clear();
        Piece cur{};
        size_t used = 0, most = 1;
        auto close = [&] {
            if (used > 0) pieces.push_back(cur);
            cur = Piece{};
            used = 0;
        };
        for (int k = 0; k < NQCLASS; ++k) {
            const size_t tile = sizeof(double) * 64 * (size_t)aimdhf::store_block(k);
            const long long end = list_off[k] + qcount[k];
            const auto r0 = starts.begin() + (starts.empty() ? 0 : runbase[k]);
            const auto r1 = starts.begin() + (starts.empty() ? 0 : runbase[k + 1]);
            for (long long pos = list_off[k]; pos < end;) {
                const long long base = pos - (pos - list_off[k]) % 64;
                const long long fit = base + (long long)((cap - std::min(used, cap)) / tile) * 64;
                long long hi = end;
                if (fit < end) {        // the last run boundary that fits
                    const auto r = std::upper_bound(r0, r1, fit);
                    hi = r == r0 ? pos : *(r - 1);
                }
                if (hi <= pos) {
                    if (used > 0) {
                        close();
                        continue;
                    }
                    const auto r = std::upper_bound(r0, r1, pos);   // a run longer than the buffer enlarges it
                    hi = r == r1 ? end : *r;
                }
                cur.base[k] = base;
                cur.lo[k] = pos;
                cur.hi[k] = hi;
                cur.at[k] = used;
                used += (size_t)((hi - base + 63) / 64) * tile;
                most = std::max(most, used);
                pos = hi;
                if (pos < end) close();         // one range of a class per piece
            }
        }
        close();
        d_store.ensure(most);
        std::vector<aimdhf::DigestGeo> geo(std::max<size_t>(pieces.size(), 1) * NQCLASS);
        for (size_t c = 0; c < pieces.size(); ++c)
            for (int k = 0; k < NQCLASS; ++k) {
                aimdhf::DigestGeo& g = geo[c * NQCLASS + k];
                g.t64 = pieces[c].base[k];
                g.lo64 = pieces[c].lo[k];
                g.hi64 = g.t32 = g.lo32 = g.hi32 = pieces[c].hi[k];
                g.off = d_loff.as<long long>() + runbase[k] * aimdhf::LIST_WAVES;
                g.lket = d_lket.as<int>();
                g.s64 = (const double*)(d_store.as<char>() + pieces[c].at[k]);
                g.s32 = nullptr;
            }
        upload(d_geo, geo);             // the stream was synchronised when the list was built
        ensure_digest(1);
    }

    aimdhf::EriArgs eri_args(int k, long long lo) const {
        aimdhf::EriArgs ea;
        ea.recs = d_recs.as<double>();
        ea.rec_off = d_rec_off.as<long long>();
        ea.npp = d_npp.as<int>();
        ea.cls_pairs = d_cls_pairs.as<int>();
        ea.boys = d_boys.as<double>();
        ea.lbra = d_lbra.as<int>() + lo;
        ea.lket = d_lket.as<int>() + lo;
        ea.out64 = (double*)(d_store.as<char>() + base64[k]);
        ea.out32 = (float*)(d_store.as<char>() + base32[k]);
        return ea;
    }

    // copies of the global J/K accumulators: one per XCD where the matrices are few
    int digest_copies() const { return batched ? 1 : 8; }

    // one launch for all classes where the runs are short (see jk_digest_all.hip)
    bool digest_in_one(int nset) const {
        return (batched || (long long)nset * nao * nao <= SMALL_JK) && aimdhf::digest_all_fits(matrix_ld(), lds_limit);
    }

    void ensure_digest(int nset) {
        const size_t mats = mat_elems() * nset, c = digest_copies();
        d_dsym.ensure(sizeof(double) * mats);
        d_dket.ensure(sizeof(double) * std::max<long long>(npao * nset, 1));
        d_kacc.ensure(sizeof(long long) * mats * c);
        d_jacc.ensure(sizeof(long long) * std::max<long long>(npao * nset, 1) * c);
        d_dcell.ensure(sizeof(long long) * aimdhf::JK_CELLS * nrep * nset);
    }

    aimdhf::PrepArgs prep_args(int nset, const double* dens, double* J, double* K) const {
        aimdhf::PrepArgs a;
        a.ld = matrix_ld();
        a.nset = nset;
        a.nrep = nrep;
        a.ncopy = digest_copies();
        a.npair = npair;
        for (int c = 0; c < 7; ++c) {
            a.cls_off[c] = cls_pair_off[c];
            a.koff[c] = koff[c];
        }
        a.npao = npao;
        a.kstride = (long long)(mat_elems() * nset);
        a.oab = d_oab.as<unsigned>();
        a.rank_rep = batched ? d_rank_rep.as<int>() : nullptr;
        a.rep_nao = batched ? d_rep_nao.as<int>() : nullptr;
        a.dens = dens;
        a.dsym = d_dsym.as<double>();
        a.dket = d_dket.as<double>();
        a.kacc = d_kacc.as<unsigned long long>();
        a.jacc = d_jacc.as<unsigned long long>();
        a.dcell = d_dcell.as<unsigned long long>();
        a.gcell = d_gcell.as<unsigned long long>();
        a.J = J;
        a.K = K;
        a.rq = d_rq.as<double>();
        return a;
    }

    // class k, or every class (k < 0) for launch_digest_all
    aimdhf::DigestArgs digest_args(int k, int nset, bool delta, double dthr) const {
        aimdhf::DigestArgs a;
        a.geo = d_geo.as<aimdhf::DigestGeo>();
        const int nk = k < 0 ? 0 : ncls[ket_class(k)];
        a.ld = matrix_ld();
        a.nset = nset;
        a.ncopy = digest_copies();
        a.lds_limit = lds_limit;
        a.nparts = list_parts;
        a.unit = unit_items;
        a.nchunk = batched ? 1 : (int)std::min<long long>(16, std::max<long long>(1, nk / (8LL * unit_items)));
        a.oab = d_oab.as<unsigned>();
        a.rank_rep = batched ? d_rank_rep.as<int>() : nullptr;
        a.dsym = d_dsym.as<double>();
        a.dket = d_dket.as<double>();
        a.npao = npao;
        for (int c = 0; c < 7; ++c) {
            a.cls_off[c] = cls_pair_off[c];
            a.koff[c] = koff[c];
        }
        a.kacc = d_kacc.as<unsigned long long>();
        a.jacc = d_jacc.as<unsigned long long>();
        a.kstride = (long long)(mat_elems() * nset);
        a.dcell = d_dcell.as<unsigned long long>();
        a.gcell = d_gcell.as<unsigned long long>();
        a.rep_nao = batched ? d_rep_nao.as<int>() : nullptr;
        a.delta = delta ? 1 : 0;
        a.dthr = dthr;
        a.rq = d_rq.as<double>();
        return a;
    }

    aimdhf::OneElArgs oneel_args() const {
        aimdhf::OneElArgs g;
        g.npair = npair;
        g.nao = nao;
        g.natm = natm;
        for (int c = 0; c < 6; ++c) {
            g.ncls_host[c] = ncls[c];
            g.cls_off_host[c] = cls_pair_off[c];
        }
        g.cls_pairs = d_cls_pairs.as<int>();
        g.pair_a = d_pair_a.as<int>();
        g.pair_b = d_pair_b.as<int>();
        g.shell_atom = d_shell_atom.as<int>();
        g.shell_l = d_shell_l.as<int>();
        g.shell_prim = d_shell_prim.as<int>();
        g.shell_ao = d_shell_ao.as<int>();
        g.prim_exp = d_prim_exp.as<double>();
        g.prim_coef = d_prim_coef.as<double>();
        g.pos = d_pos.as<double>();
        g.charges = d_charges.as<double>();
        g.boys = d_boys.as<double>();
        g.parts = 3;
        g.ld = batched ? bld : nao;
        g.mstride = (long long)mat_elems();
        g.shell_rep = batched ? d_shell_rep.as<int>() : nullptr;
        g.rep_atom = batched ? d_rep_atom.as<int>() : nullptr;
        return g;
    }

};

static int pair_class(int la, int lb) { return la * (la + 1) / 2 + lb; }

extern "C" {

int aimdhf_last_error(char* buf, size_t len) {
    if (buf && len) {
        std::strncpy(buf, g_err.c_str(), len - 1);
        buf[len - 1] = 0;
    }
    return AIMDHF_OK;
}

int aimdhf_lmax(void) { return aimdhf::GEN_LMAX; }

}  // extern "C"

// Plan of one molecule (nrep = 0) or of nrep replicas (shells and atoms grouped
// by replica: rep_shell / rep_atom hold nrep + 1 offsets)
static int create_plan(int natm, int nshell, const int64_t* shell_atom, const int64_t* shell_l,
                       const int64_t* shell_prim, const int64_t* shell_block, const double* prim_exp,
                       const double* prim_coef, const double* charges, int nrep, const int64_t* rep_atom,
                       const int64_t* rep_shell, aimdhf_plan** out) {
    if (!out) return fail(AIMDHF_E_ARG, "out is NULL");
    *out = nullptr;
    if (natm <= 0 || nshell <= 0) return fail(AIMDHF_E_ARG, "natm and nshell must be positive");
    if (!shell_atom || !shell_l || !shell_prim || !shell_block || !prim_exp || !prim_coef || !charges)
        return fail(AIMDHF_E_ARG, "NULL basis array");
    if (nrep > 0) {
        if (!rep_atom || !rep_shell) return fail(AIMDHF_E_ARG, "NULL replica offsets");
        if (rep_atom[0] != 0 || rep_shell[0] != 0 || rep_atom[nrep] != natm || rep_shell[nrep] != nshell)
            return fail(AIMDHF_E_ARG, "replica offsets must run from 0 to natm and nshell");
        for (int r = 0; r < nrep; ++r)
            if (rep_atom[r + 1] <= rep_atom[r] || rep_shell[r + 1] <= rep_shell[r])
                return fail(AIMDHF_E_ARG, "every replica needs at least one atom and one shell");
        for (int r = 0; r < nrep; ++r)
            for (int64_t sh = rep_shell[r]; sh < rep_shell[r + 1]; ++sh)
                if (shell_atom[sh] < rep_atom[r] || shell_atom[sh] >= rep_atom[r + 1])
                    return fail(AIMDHF_E_ARG, "a shell sits on an atom of another replica");
    }
    aimdhf_plan* p = new (std::nothrow) aimdhf_plan();
    if (!p) return fail(AIMDHF_E_NOMEM, "host allocation failed");
    try {
        p->natm = natm;
        p->nshell = nshell;
        p->batched = nrep > 0;
        p->nrep = nrep > 0 ? nrep : 1;
        // replica of every shell and the first shell of its replica (one replica: 0)
        p->shell_rep.assign(nshell, 0);
        p->shell_first.assign(nshell, 0);
        p->rep_shell.assign(p->nrep + 1, 0);
        p->rep_atom.assign(p->nrep + 1, 0);
        p->rep_shell[p->nrep] = nshell;
        p->rep_atom[p->nrep] = natm;
        if (p->batched)
            for (int r = 0; r < nrep; ++r) {
                p->rep_shell[r] = (int)rep_shell[r];
                p->rep_atom[r] = (int)rep_atom[r];
                for (int64_t sh = rep_shell[r]; sh < rep_shell[r + 1]; ++sh) {
                    p->shell_rep[sh] = r;
                    p->shell_first[sh] = (int)rep_shell[r];
                }
            }
        int nprim = (int)shell_prim[nshell];
        p->shell_atom.resize(nshell);
        p->shell_l.resize(nshell);
        p->shell_prim.resize(nshell + 1);
        p->shell_block.resize(nshell);
        p->shell_ao.resize(nshell + 1);
        p->shell_ao[0] = 0;
        for (int s = 0; s < nshell; ++s) {
            if (shell_l[s] < 0 || shell_l[s] > aimdhf::GEN_LMAX || (nrep > 0 && shell_l[s] > 2)) {
                delete p;
                return fail(AIMDHF_E_UNSUPPORTED,
                            "angular momentum l = " + std::to_string(shell_l[s]) + " is not supported" +
                                (nrep > 0 ? std::string(" in batched plans (l <= 2)")
                                          : " (l <= " + std::to_string(aimdhf::GEN_LMAX) + ")"));
            }
            if (shell_atom[s] < 0 || shell_atom[s] >= natm || shell_prim[s + 1] <= shell_prim[s]) {
                delete p;
                return fail(AIMDHF_E_ARG, "inconsistent shell arrays");
            }
            p->shell_atom[s] = (int)shell_atom[s];
            p->shell_l[s] = (int)shell_l[s];
            p->shell_prim[s] = (int)shell_prim[s];
            p->shell_block[s] = (int)shell_block[s];
            p->shell_ao[s + 1] = p->shell_ao[s] + ncart(p->shell_l[s]);
            p->lmax = std::max(p->lmax, p->shell_l[s]);
        }
        p->shell_prim[nshell] = nprim;
        p->nao = p->shell_ao[nshell];
        if (p->lmax > 2) {
            // runtime-l kernels for every integral: shell pairs, bounds, no pair records
            p->generic = true;
            p->nblock = p->shell_block[nshell - 1] + 1;
            p->nbpair = p->nblock * (p->nblock + 1) / 2;
            p->prim_exp.assign(prim_exp, prim_exp + nprim);
            p->prim_coef.assign(prim_coef, prim_coef + nprim);
            p->charges.assign(charges, charges + natm);
            p->npair = nshell * (nshell + 1) / 2;
            for (int i = 0; i < nshell; ++i)
                for (int j = 0; j <= i; ++j) {
                    p->gpair_i.push_back(i);
                    p->gpair_j.push_back(j);
                    const int b1 = p->shell_block[i], b2 = p->shell_block[j];
                    p->gpair_bp.push_back(b1 * (b1 + 1) / 2 + b2);
                }
            p->qcount.assign(NQCLASS, 0);
            p->gcount.assign(NQCLASS, 0);
            upload(p->d_shell_atom, p->shell_atom);
            upload(p->d_shell_l, p->shell_l);
            upload(p->d_shell_prim, p->shell_prim);
            upload(p->d_shell_ao, p->shell_ao);
            upload(p->d_prim_exp, p->prim_exp);
            upload(p->d_prim_coef, p->prim_coef);
            upload(p->d_charges, p->charges);
            upload(p->d_boys, boys_table());
            upload(p->d_gpair_i, p->gpair_i);
            upload(p->d_gpair_j, p->gpair_j);
            p->d_scratch.ensure(sizeof(double) * 1024);
            p->d_pos.ensure(sizeof(double) * 3 * natm);
            p->d_qshell.ensure(sizeof(double) * p->npair);
            p->d_qblock.ensure(sizeof(double) * p->nbpair);
            *out = p;
            return AIMDHF_OK;
        }
        if (p->batched) {
            // AO offsets within each replica; replica sizes, padded dimension, tensors
            p->rep_nao.assign(p->nrep, 0);
            for (int r = 0; r < p->nrep; ++r) {
                const int a0 = p->shell_ao[p->rep_shell[r]];
                p->rep_nao[r] = p->shell_ao[p->rep_shell[r + 1]] - a0;
                p->bld = std::max(p->bld, p->rep_nao[r]);
            }
            std::vector<int> local(nshell + 1);
            for (int sh = 0; sh < nshell; ++sh) local[sh] = p->shell_ao[sh] - p->shell_ao[p->shell_first[sh]];
            local[nshell] = 0;
            p->shell_ao = local;
            for (int r = 0; r < p->nrep; ++r) {
                const long long n = p->rep_nao[r];
                p->tens_total += n * n * n * n;
            }
        }
        p->nblock = p->shell_block[nshell - 1] + 1;
        p->prim_exp.assign(prim_exp, prim_exp + nprim);
        p->prim_coef.assign(prim_coef, prim_coef + nprim);
        p->charges.assign(charges, charges + natm);
        // shell pairs (s1 >= s2) in the reference's pair order, oriented l_A >= l_B; in a
        // batch only the pairs within a replica, replica by replica
        p->npair = 0;
        for (int r = 0; r < p->nrep; ++r) {
            const int ns = p->rep_shell[r + 1] - p->rep_shell[r];
            p->npair += ns * (ns + 1) / 2;
        }
        p->pair_a.resize(p->npair);
        p->pair_b.resize(p->npair);
        p->pair_cls.resize(p->npair);
        p->rec_size.resize(p->npair);
        p->rec_off.resize(p->npair + 1);
        long long off = 0;
        int P = 0;
        std::vector<std::vector<int>> bylcls(6);
        // block pairs within each replica, replica by replica (one molecule: i(i+1)/2+j)
        std::vector<int> rep_b0(p->nrep), rep_bp0(p->nrep + 1, 0), rep_p0(p->nrep + 1, 0);
        for (int r = 0; r < p->nrep; ++r) {
            rep_b0[r] = p->shell_block[p->rep_shell[r]];
            const int nb = p->shell_block[p->rep_shell[r + 1] - 1] - rep_b0[r] + 1;
            rep_bp0[r + 1] = rep_bp0[r] + nb * (nb + 1) / 2;
            const int ns = p->rep_shell[r + 1] - p->rep_shell[r];
            rep_p0[r + 1] = rep_p0[r] + ns * (ns + 1) / 2;
        }
        p->nbpair = rep_bp0[p->nrep];
        std::vector<std::vector<int>> bpl(p->nbpair);
        p->shell_pair0.assign(nshell, 0);
        p->pair_lo.assign(p->npair, 0);
        for (int s1 = 0; s1 < nshell; ++s1) p->shell_pair0[s1] = rep_p0[p->shell_rep[s1]];
        for (int s1 = 0; s1 < nshell; ++s1)
            for (int s2 = p->shell_first[s1]; s2 <= s1; ++s2, ++P) {
                p->pair_lo[P] = p->shell_pair0[s1];
                int a = s1, b = s2;
                if (p->shell_l[s2] > p->shell_l[s1]) std::swap(a, b);
                int la = p->shell_l[a], lb = p->shell_l[b];
                p->pair_a[P] = a;
                p->pair_b[P] = b;
                p->pair_cls[P] = pair_class(la, lb);
                int rs = REC_HDR + nherm(la + lb) * ncart(la) * ncart(lb);
                p->rec_size[P] = rs;
                p->rec_off[P] = off;
                off += (long long)rs * (shell_prim[s1 + 1] - shell_prim[s1]) * (shell_prim[s2 + 1] - shell_prim[s2]);
                bylcls[p->pair_cls[P]].push_back(P);
                const int r = p->shell_rep[s1];
                int b1 = p->shell_block[s1] - rep_b0[r], b2 = p->shell_block[s2] - rep_b0[r];
                bpl[rep_bp0[r] + b1 * (b1 + 1) / 2 + b2].push_back(P);
            }
        p->rec_off[p->npair] = off;
        p->rec_total = off;
        // rank order of the pairs (jk_digest.h): per class, replica by replica, the most
        // contracted first, then along the diagonals of the pair triangle
        {
            std::vector<int> first(p->npair), second(p->npair);
            for (int r = 0, Q = 0; r < p->nrep; ++r)
                for (int s1 = p->rep_shell[r]; s1 < p->rep_shell[r + 1]; ++s1)
                    for (int s2 = p->rep_shell[r]; s2 <= s1; ++s2, ++Q) {
                        first[Q] = s1;
                        second[Q] = s2;
                    }
            auto nprim_of = [&](int sh) { return (int)(shell_prim[sh + 1] - shell_prim[sh]); };
            for (auto& v : bylcls)
                std::stable_sort(v.begin(), v.end(), [&](int x, int y) {
                    const int rx = p->shell_rep[first[x]], ry = p->shell_rep[first[y]];
                    if (rx != ry) return rx < ry;
                    const int cx = nprim_of(first[x]) * nprim_of(second[x]), cy = nprim_of(first[y]) * nprim_of(second[y]);
                    if (cx != cy) return cx > cy;
                    const int dx = p->pair_a[x] - p->pair_b[x], dy = p->pair_a[y] - p->pair_b[y];
                    return dx != dy ? dx < dy : first[x] < first[y];
                });
            // in a batch the contracted pairs of a class come replica by replica: all of them
            // count as contracted where any is
            for (int c = 0; c < 6; ++c) {
                int n = 0;
                for (int x : bylcls[c]) n += nprim_of(first[x]) * nprim_of(second[x]) >= aimdhf::ERI_HEAVY;
                p->nheavy[c] = p->batched && n > 0 ? (int)bylcls[c].size() : n;
            }
        }
        p->cls_pair_off.assign(7, 0);
        p->ncls.assign(6, 0);
        for (int c = 0; c < 6; ++c) {
            p->cls_pair_off[c + 1] = p->cls_pair_off[c] + (int)bylcls[c].size();
            p->ncls[c] = (int)bylcls[c].size();
            p->cls_pairs.insert(p->cls_pairs.end(), bylcls[c].begin(), bylcls[c].end());
        }
        // AO offsets and replica of every rank, rank range of every (class, replica), and
        // the base of every class's components
        std::vector<unsigned> oab(p->npair);
        std::vector<int> rank_rep(p->npair), seg(6 * p->nrep + 1, p->npair);
        for (int r = p->npair - 1; r >= 0; --r) {
            const int Q = p->cls_pairs[r], a = p->pair_a[Q], b = p->pair_b[Q];
            oab[r] = aimdhf::oab_pack(p->shell_ao[a], p->shell_ao[b]);
            rank_rep[r] = p->shell_rep[a];
            seg[p->pair_cls[Q] * p->nrep + rank_rep[r]] = r;
        }
        // segments without pairs start where the next one does
        for (int i = 6 * p->nrep - 1; i >= 0; --i) {
            const int c = i / p->nrep;
            const bool any = seg[i] < p->npair && p->pair_cls[p->cls_pairs[seg[i]]] == c &&
                             rank_rep[seg[i]] == i % p->nrep;
            if (!any) seg[i] = seg[i + 1];
        }
        p->koff[0] = 0;
        for (int c = 0; c < 6; ++c) {
            const int la = c == 0 ? 0 : c <= 2 ? 1 : 2, lb = c - la * (la + 1) / 2;
            p->koff[c + 1] = p->koff[c] + (long long)p->ncls[c] * ncart(la) * ncart(lb);
        }
        p->npao = p->koff[6];
        upload(p->d_oab, oab);
        upload(p->d_seg, seg);
        if (p->batched) {
            upload(p->d_rank_rep, rank_rep);
            upload(p->d_rep_shell, p->rep_shell);
        }
        p->d_rq.ensure(sizeof(double) * p->npair);
        p->d_gcell.ensure(sizeof(long long) * 3 * p->nrep);
        {
            int dev = 0, lim = 0;
            HIPCHECK(hipGetDevice(&dev));
            HIPCHECK(hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
            p->lds_limit = std::max(lim, 65536);
        }
        p->bp_off.assign(p->nbpair + 1, 0);
        for (int i = 0; i < p->nbpair; ++i) {
            p->bp_off[i + 1] = p->bp_off[i] + (int)bpl[i].size();
            p->bp_list.insert(p->bp_list.end(), bpl[i].begin(), bpl[i].end());
        }
        // device copies
        upload(p->d_shell_atom, p->shell_atom);
        upload(p->d_shell_l, p->shell_l);
        upload(p->d_shell_prim, p->shell_prim);
        upload(p->d_shell_ao, p->shell_ao);
        upload(p->d_prim_exp, p->prim_exp);
        upload(p->d_prim_coef, p->prim_coef);
        upload(p->d_pair_a, p->pair_a);
        upload(p->d_pair_b, p->pair_b);
        upload(p->d_pair_cls, p->pair_cls);
        upload(p->d_rec_size, p->rec_size);
        upload(p->d_rec_off, p->rec_off);
        upload(p->d_cls_pairs, p->cls_pairs);
        upload(p->d_cls_pair_off, p->cls_pair_off);
        upload(p->d_ncls, p->ncls);
        upload(p->d_bp_off, p->bp_off);
        upload(p->d_bp_list, p->bp_list);
        upload(p->d_boys, boys_table());
        upload(p->d_charges, p->charges);
        if (p->batched) {
            upload(p->d_shell_rep, p->shell_rep);
            upload(p->d_shell_first, p->shell_first);
            upload(p->d_shell_pair0, p->shell_pair0);
            upload(p->d_pair_lo, p->pair_lo);
            upload(p->d_rep_atom, p->rep_atom);
            upload(p->d_rep_nao, p->rep_nao);
        }
        p->d_scratch.ensure(sizeof(double) * 1024);
        p->d_pos.ensure(sizeof(double) * 3 * natm);
        p->d_recs.ensure(sizeof(double) * std::max<long long>(off, 1));
        p->d_npp.ensure(sizeof(int) * p->npair);
        p->d_qshell.ensure(sizeof(double) * p->npair);
        p->d_qscr.ensure(sizeof(double) * p->npair);
        p->d_qblock.ensure(sizeof(double) * p->nbpair);
        p->qcount.assign(NQCLASS, 0);
        p->noalloc_ptr = aimdhf::noalloc_scratch(&p->noalloc_bytes);
        if (!p->noalloc_ptr) {
            delete p;
            return fail(AIMDHF_E_HIP, "hipGetSymbolAddress of the fixed scratch array failed");
        }
    } catch (const HipError& e) {
        delete p;
        return e.code;
    } catch (const std::bad_alloc&) {
        delete p;
        return fail(AIMDHF_E_NOMEM, "host allocation failed");
    }
    *out = p;
    return AIMDHF_OK;
}

// ------------------------------------------------------------ runtime-l path
static int set_geometry_generic(aimdhf_plan* p, const double* positions, double thr, hipStream_t st) {
    try {
        p->pos.assign(positions, positions + 3 * p->natm);
        HIPCHECK(hipMemcpyAsync(p->d_pos.p, positions, sizeof(double) * 3 * p->natm, hipMemcpyHostToDevice, st));
        aimdhf::GenArgs g = p->gen_args();
        p->prof.time(42, st, [&] { aimdhf::launch_gen_schwarz(g, p->npair, st); });
        HIPCHECK(hipGetLastError());
        std::vector<double> qs(p->npair);
        HIPCHECK(hipMemcpyAsync(qs.data(), p->d_qshell.p, sizeof(double) * p->npair, hipMemcpyDeviceToHost, st));
        HIPCHECK(hipStreamSynchronize(st));
        auto t0 = Profiler::clock::now();
        // block-pair bounds: the largest shell-pair bound of the block pair
        p->gen_qb.assign(p->nbpair, 0.0);
        for (int P = 0; P < p->npair; ++P) p->gen_qb[p->gpair_bp[P]] = std::max(p->gen_qb[p->gpair_bp[P]], qs[P]);
        upload(p->d_qblock, p->gen_qb);
        // kept primitive pairs (mu |AB|^2 <= 50) per shell pair
        p->gen_npp.assign(p->npair, 0);
        for (int P = 0; P < p->npair; ++P) {
            const int a = p->gpair_i[P], b = p->gpair_j[P];
            double r2 = 0.0;
            for (int d = 0; d < 3; ++d) {
                const double x = p->pos[3 * p->shell_atom[a] + d] - p->pos[3 * p->shell_atom[b] + d];
                r2 += x * x;
            }
            int n = 0;
            for (int i = p->shell_prim[a]; i < p->shell_prim[a + 1]; ++i)
                for (int j = p->shell_prim[b]; j < p->shell_prim[b + 1]; ++j) {
                    const double x = p->prim_exp[i], y = p->prim_exp[j];
                    if (x * y / (x + y) * r2 <= 50.0) ++n;
                }
            p->gen_npp[P] = n;
        }
        p->qtotal = p->gen_build_list(thr, p->d_list);
        p->threshold = thr;
        p->stored = false;
        p->store_bytes = 0;
        p->prof.host(85, t0);
        p->have_geometry = true;
    } catch (const HipError& e) {
        p->have_geometry = false;
        return e.code;
    }
    return AIMDHF_OK;
}

static int jk_generic(aimdhf_plan* p, int nset, const double* dens, double* J, double* K, hipStream_t st) {
    try {
        const size_t nn = (size_t)p->nao * p->nao;
        p->d_dsym.ensure(sizeof(double) * nset * nn);
        p->d_fx.ensure(sizeof(long long) * 4 * nset * nn);
        aimdhf::launch_symmetrize(dens, nset, p->nao, p->d_dsym.as<double>(), st);
        aimdhf::launch_zero64(p->d_fx.as<long long>(), 4 * nset * nn, st);
        aimdhf::GenArgs g = p->gen_args();
        g.nset = nset;
        g.dens = p->d_dsym.as<double>();
        g.fx = p->d_fx.as<long long>();
        g.quartets = p->d_list.as<int2>();
        g.nq = p->qtotal;
        p->prof.time(95, st, [&] { aimdhf::launch_gen_jk(g, st); });
        aimdhf::launch_jk_finalize(p->d_fx.as<long long>(), nset, p->nao, J, K, st);
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

// one-electron gradient terms `parts` (1 kinetic, 2 nuclear attraction, 4 overlap) into grad
static void grad_one_generic(aimdhf_plan* p, const double* D, const double* W, int parts, double* grad, hipStream_t st) {
    const size_t nn = (size_t)p->nao * p->nao;
    p->d_gden.ensure(sizeof(double) * 2 * nn);
    double* Ds = p->d_gden.as<double>();
    double* Ws = Ds + nn;
    aimdhf::launch_symmetrize(D, 1, p->nao, Ds, st);
    aimdhf::launch_symmetrize(W, 1, p->nao, Ws, st);
    p->d_gfx.ensure(sizeof(long long) * 6 * p->natm);
    aimdhf::launch_zero64(p->d_gfx.as<long long>(), 6 * p->natm, st);
    aimdhf::GenArgs g = p->gen_args();
    g.D = Ds;
    g.W = Ws;
    g.parts = parts;
    g.fx = p->d_gfx.as<long long>();
    p->prof.time(44, st, [&] { aimdhf::launch_gen_grad1(g, p->npair, st); });
    aimdhf::launch_fx_to_double(p->d_gfx.as<long long>(), 3 * p->natm, grad, st);
    HIPCHECK(hipGetLastError());
}

static int grad_two_generic(aimdhf_plan* p, const double* Dc, int nx, const double* Dx, double kfac, double thr,
                            double* grad, hipStream_t st) {
    try {
        const size_t nn = (size_t)p->nao * p->nao;
        p->d_gden.ensure(sizeof(double) * (1 + nx) * nn);
        double* dc = p->d_gden.as<double>();
        double* dx = dc + nn;
        aimdhf::launch_symmetrize(Dc, 1, p->nao, dc, st);
        aimdhf::launch_symmetrize(Dx, nx, p->nao, dx, st);
        // quartets with q_P q_Q max|Gamma| >= thr for the largest possible |Gamma| element
        const double mc = aimdhf::device_absmax(dc, nn, p->d_scratch.as<double>(), st);
        const double mx = aimdhf::device_absmax(dx, nx * nn, p->d_scratch.as<double>(), st);
        if (mc < 0.0 || mx < 0.0) return fail(AIMDHF_E_HIP, "max reduction failed");
        const double gbound = 4.0 * (mc * mc + std::fabs(kfac) * nx * mx * mx);
        auto t0 = Profiler::clock::now();
        p->gen_gq = p->gen_build_list(gbound > 0.0 ? thr / gbound : 0.0, p->d_glist);
        p->prof.host(88, t0);
        p->d_gfx.ensure(sizeof(long long) * 6 * p->natm);
        aimdhf::launch_zero64(p->d_gfx.as<long long>(), 6 * p->natm, st);
        aimdhf::GenArgs g = p->gen_args();
        g.dc = dc;
        g.dx = dx;
        g.nx = nx;
        g.kfac = kfac;
        g.fx = p->d_gfx.as<long long>();
        g.quartets = p->d_glist.as<int2>();
        g.nq = p->gen_gq;
        p->prof.time(96, st, [&] { aimdhf::launch_gen_grad2(g, st); });
        aimdhf::launch_fx_to_double(p->d_gfx.as<long long>(), 3 * p->natm, grad, st);
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

extern "C" {

int aimdhf_plan_create(int natm, int nshell, const int64_t* shell_atom, const int64_t* shell_l,
                       const int64_t* shell_prim, const int64_t* shell_block, const double* prim_exp,
                       const double* prim_coef, const double* charges, aimdhf_plan** out) {
    return create_plan(natm, nshell, shell_atom, shell_l, shell_prim, shell_block, prim_exp, prim_coef, charges, 0,
                       nullptr, nullptr, out);
}

int aimdhf_batch_create(int nrep, const int64_t* rep_atom, const int64_t* rep_shell, int natm, int nshell,
                        const int64_t* shell_atom, const int64_t* shell_l, const int64_t* shell_prim,
                        const int64_t* shell_block, const double* prim_exp, const double* prim_coef,
                        const double* charges, aimdhf_plan** out) {
    if (nrep <= 0) return fail(AIMDHF_E_ARG, "a batch needs at least one replica");
    return create_plan(natm, nshell, shell_atom, shell_l, shell_prim, shell_block, prim_exp, prim_coef, charges, nrep,
                       rep_atom, rep_shell, out);
}

int aimdhf_batch_layout(aimdhf_plan* p, int* nrep, int* ld, int64_t* tensor_bytes) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (nrep) *nrep = p->batched ? p->nrep : 0;
    if (ld) *ld = p->batched ? p->bld : p->nao;
    if (tensor_bytes) *tensor_bytes = p->batched ? 8 * p->tens_total : 0;
    return AIMDHF_OK;
}

int aimdhf_plan_destroy(aimdhf_plan* plan) {
    delete plan;
    return AIMDHF_OK;
}

int aimdhf_set_geometry(aimdhf_plan* p, const double* positions, double thr, void* stream) {
    if (!p || !positions) return fail(AIMDHF_E_ARG, "NULL plan or positions");
    for (int i = 0; i < 3 * p->natm; ++i)
        if (!std::isfinite(positions[i])) return fail(AIMDHF_E_ARG, "atomic positions must be finite (got NaN or inf)");
    if (!(thr >= 0.0)) return fail(AIMDHF_E_ARG, "schwarz threshold must be >= 0");
    hipStream_t st = (hipStream_t)stream;
    p->have_last_store = false;     // the store's buffers may move
    if (p->generic) return set_geometry_generic(p, positions, thr, st);
    // 16-bit offsets of the quartet list (J, K, the density and its copies of a larger
    // matrix, 34 GB each, would not fit)
    if (p->matrix_ld() > aimdhf::MAX_LD)
        return fail(AIMDHF_E_UNSUPPORTED, "matrices of more than " + std::to_string(aimdhf::MAX_LD) + " AOs");
    try {
        p->pos.assign(positions, positions + 3 * p->natm);
        HIPCHECK(hipMemcpyAsync(p->d_pos.p, positions, sizeof(double) * 3 * p->natm, hipMemcpyHostToDevice, st));
        aimdhf::PairArgs g = p->pair_args();
        p->prof.time(42, st, [&] {
            aimdhf::launch_build_pairs(g, st);
            aimdhf::launch_schwarz(g, p->ncls.data(), st);
        });
        HIPCHECK(hipGetLastError());
        auto t0 = Profiler::clock::now();
        // direct mode evaluates in FP64 throughout
        const double sw = p->precision == 1 && p->jk_switch > thr ? p->jk_switch : 0.0;
        p->build_quartets(thr, p->jk_mode == 1 && !p->batched ? 0.0 : sw, st);
        p->threshold = thr;
        p->prof.host(85, t0);
        p->stored = false;
        p->store_bytes = 0;
        if (p->batched) {
            auto t1 = Profiler::clock::now();
            p->build_store(st);
            p->prof.host(87, t1);
            p->have_geometry = true;
            return AIMDHF_OK;
        }
        bool store = false;
        if (p->jk_mode != 1) {
            long long limit = p->store_limit;
            if (limit <= 0) {
                size_t fr = 0, tot = 0;
                HIPCHECK(hipMemGetInfo(&fr, &tot));
                limit = (long long)(fr / 2);
            }
            store = p->jk_mode == 2 || (long long)p->store_need <= limit;
        }
        if (!store) {
            t0 = Profiler::clock::now();
            if (p->list_parts == 2) p->build_quartets(thr, 0.0, st);
            p->build_direct(st);
            p->prof.host(86, t0);
        } else {
            auto t1 = Profiler::clock::now();
            p->build_store(st);
            p->prof.host(87, t1);
            p->stored = true;
        }
        p->have_geometry = true;
    } catch (const HipError& e) {
        p->have_geometry = false;
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_schwarz_bounds(aimdhf_plan* p, double* out, int64_t cap) {
    if (!p || !out) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    if (cap < p->nbpair) return fail(AIMDHF_E_ARG, "output too small");
    try {
        HIPCHECK(hipMemcpy(out, p->d_qblock.p, sizeof(double) * p->nbpair, hipMemcpyDeviceToHost));
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_quartet_count(aimdhf_plan* p, int64_t* count) {
    if (!p || !count) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    *count = p->qtotal;
    return AIMDHF_OK;
}

int aimdhf_quartets(aimdhf_plan* p, int64_t* out, int64_t cap, int64_t* count) {
    if (!p || !count) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    *count = p->qtotal;
    if (!out || cap <= 0) return AIMDHF_OK;
    try {
        long long n = std::min<long long>(cap, p->qtotal);
        std::vector<int2> tmp(n);
        if (p->generic) {
            if (n) HIPCHECK(hipMemcpy(tmp.data(), p->d_list.p, sizeof(int2) * n, hipMemcpyDeviceToHost));
        } else if (n) {
            std::vector<int> b(n), k(n);
            HIPCHECK(hipMemcpy(b.data(), p->d_lbra.p, sizeof(int) * n, hipMemcpyDeviceToHost));
            HIPCHECK(hipMemcpy(k.data(), p->d_lket.p, sizeof(int) * n, hipMemcpyDeviceToHost));
            for (long long i = 0; i < n; ++i) tmp[i] = make_int2(p->cls_pairs[b[i]], p->cls_pairs[k[i]]);
        }
        for (long long i = 0; i < n; ++i) {
            int a = tmp[i].x, b = tmp[i].y;
            out[2 * i] = std::max(a, b);
            out[2 * i + 1] = std::min(a, b);
        }
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_grad_quartets(aimdhf_plan* p, int64_t* out, int64_t cap, int64_t* count) {
    if (!p || !count) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    try {
        if (p->generic) {
            std::vector<int2> lst(p->gen_gq);
            if (p->gen_gq)
                HIPCHECK(hipMemcpy(lst.data(), p->d_glist.p, sizeof(int2) * p->gen_gq, hipMemcpyDeviceToHost));
            for (long long i = 0; out && i < std::min<long long>(cap, p->gen_gq); ++i) {
                out[2 * i] = lst[i].x;
                out[2 * i + 1] = lst[i].y;
            }
            *count = p->gen_gq;
            return AIMDHF_OK;
        }
        long long tot = 0;
        for (long long c : p->gcount) tot += c;
        std::vector<int2> lst(tot);
        std::vector<unsigned char> keep(tot);
        if (tot) {
            HIPCHECK(hipMemcpy(lst.data(), p->d_glist.p, sizeof(int2) * tot, hipMemcpyDeviceToHost));
            HIPCHECK(hipMemcpy(keep.data(), p->d_gkeep.p, tot, hipMemcpyDeviceToHost));
        }
        long long n = 0;
        for (long long i = 0; i < tot; ++i) {
            if (!keep[i]) continue;
            if (out && n < cap) {
                out[2 * n] = std::max(lst[i].x, lst[i].y);
                out[2 * n + 1] = std::min(lst[i].x, lst[i].y);
            }
            ++n;
        }
        *count = n;
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

// J and K from the integral store (one molecule, or every replica of a batch);
// delta: dens is a density difference and quartets below dthr may be skipped
static int jk_from_store(aimdhf_plan* p, int nset, const double* dens, double* J, double* K, bool delta, double dthr,
                         hipStream_t st) {
    try {
        p->have_last_store = false;     // a failed allocation below leaves the last build's arguments stale
        p->ensure_digest(nset);
        const aimdhf::PrepArgs pa = p->prep_args(nset, dens, J, K);
        p->prof.time(45, st, [&] { aimdhf::launch_jk_prep(pa, st); });
        // the classes add to the same accumulators in any order
        const int threads = p->batched ? 4 * p->batch_jk_lanes : 256;
        if (p->digest_in_one(nset)) {
            const aimdhf::DigestArgs da = p->digest_args(-1, nset, delta, dthr);
            for (int k = 0; k < NQCLASS; ++k) p->last_dig[k] = p->digest_args(k, nset, delta, dthr);
            p->prof.time(94, st, [&] { aimdhf::launch_digest_all(da, threads, st); });
        } else {
            // spread over the fan's streams; a batch's launches and those that a graph records stay
            // on the caller's stream (the graph outlives calls and must not depend on the plan's
            // streams), and a batch's cover every class, as its graph is replayed at other geometries
            const bool one = p->batched || Fan::capturing(st);
            if (!one) p->fan.fork(st);
            int i = 0;
            for (int k = NQCLASS - 1; k >= 0; --k) {
                if (!p->qcount[k] && !p->batched) continue;
                p->last_dig[k] = p->digest_args(k, nset, delta, dthr);
                hipStream_t s2 = one ? st : p->fan.on(i++);
                p->prof.time(98 + k, s2, [&] { aimdhf::launch_digest(k, p->last_dig[k], threads, s2); });
            }
            if (!one) p->fan.join();
        }
        p->have_last_store = true;
        p->prof.time(93, st, [&] { aimdhf::launch_jk_finish(pa, st); });
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_jk_delta(aimdhf_plan* p, int nset, const double* ddens, double* dJ, double* dK, double threshold,
                    void* stream) {
    if (!p || !ddens || !dJ || !dK) return fail(AIMDHF_E_ARG, "NULL argument");
    if (nset < 1 || nset > 2) return fail(AIMDHF_E_ARG, "nset must be 1 or 2");
    if (!(threshold >= 0.0) || !std::isfinite(threshold)) return fail(AIMDHF_E_ARG, "threshold must be finite and >= 0");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    if (p->batched || !p->stored) return aimdhf_jk(p, nset, ddens, dJ, dK, stream);
    return jk_from_store(p, nset, ddens, dJ, dK, true, threshold, (hipStream_t)stream);
}

// J and K with the integrals evaluated piece by piece (direct mode)
static int jk_direct(aimdhf_plan* p, int nset, const double* dens, double* J, double* K, hipStream_t st) {
    try {
        p->ensure_digest(nset);
        const aimdhf::PrepArgs pa = p->prep_args(nset, dens, J, K);
        p->prof.time(45, st, [&] { aimdhf::launch_jk_prep(pa, st); });
        const bool one = Fan::capturing(st);    // a graph records the caller's stream alone
        for (size_t c = 0; c < p->pieces.size(); ++c) {
            const aimdhf_plan::Piece& pc = p->pieces[c];
            // a class is digested on the stream that evaluates it; the pieces share the buffer
            if (!one) p->fan.fork(st);
            int i = 0;
            for (int k = NQCLASS - 1; k >= 0; --k) {
                if (pc.hi[k] <= pc.lo[k]) continue;
                const long long n = pc.hi[k] - pc.base[k];
                hipStream_t s2 = one ? st : p->fan.on(i++);
                aimdhf::EriArgs ea = p->eri_args(k, pc.base[k]);
                ea.out64 = (double*)(p->d_store.as<char>() + pc.at[k]);
                const long long h = p->list_off[k] + p->h64count[k] - pc.base[k];
                p->prof.time(46, s2, [&] { aimdhf::launch_eri(k, ea, n, std::min(std::max(h, 0LL), n), 0, 0, s2); });
                aimdhf::DigestArgs da = p->digest_args(k, nset, false, 0.0);
                da.geo += c * NQCLASS;
                p->prof.time(98 + k, s2, [&] { aimdhf::launch_digest(k, da, 256, s2); });
            }
            if (!one) p->fan.join();
        }
        p->prof.time(93, st, [&] { aimdhf::launch_jk_finish(pa, st); });
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_jk(aimdhf_plan* p, int nset, const double* dens, double* J, double* K, void* stream) {
    if (!p || !dens || !J || !K) return fail(AIMDHF_E_ARG, "NULL argument");
    if (nset < 1 || nset > 2) return fail(AIMDHF_E_ARG, "nset must be 1 or 2");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    hipStream_t st = (hipStream_t)stream;
    if (p->generic) return jk_generic(p, nset, dens, J, K, st);
    if (p->batched || p->stored) return jk_from_store(p, nset, dens, J, K, false, 0.0, st);
    return jk_direct(p, nset, dens, J, K, st);
}

int aimdhf_one_electron(aimdhf_plan* p, double* S, double* T, double* V, double* M, void* stream) {
    if (!p || !S || !T || !V || !M) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    hipStream_t st = (hipStream_t)stream;
    try {
        if (p->batched) {
            // padded layout: only the replicas' own blocks are written
            const size_t n = p->mat_elems();
            aimdhf::launch_zero_d(S, n, st);
            aimdhf::launch_zero_d(T, n, st);
            aimdhf::launch_zero_d(V, n, st);
            aimdhf::launch_zero_d(M, 3 * n, st);
        }
        if (p->generic) {
            aimdhf::GenArgs g = p->gen_args();
            g.S = S;
            g.T = T;
            g.V = V;
            g.M = M;
            p->prof.time(43, st, [&] { aimdhf::launch_gen_oneel(g, p->npair, st); });
        } else {
            p->prof.time(43, st, [&] {
                const bool one = Fan::capturing(st);
                if (!one) p->fan.fork(st);
                aimdhf::launch_oneel(p->oneel_args(), S, T, M, V, (one ? PairStreams(st) : PairStreams(p->fan)).on);
                if (!one) p->fan.join();
            });
        }
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_grad_one(aimdhf_plan* p, const double* D, const double* W, double* grad, void* stream) {
    if (!p || !D || !W || !grad) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    hipStream_t st = (hipStream_t)stream;
    try {
        if (p->generic) {
            grad_one_generic(p, D, W, 7, grad, st);
            return AIMDHF_OK;
        }
        const size_t nn = p->mat_elems();
        const int nmat = p->batched ? p->nrep : 1, ld = p->batched ? p->bld : p->nao;
        p->d_gden.ensure(sizeof(double) * 2 * nn);
        double* Ds = p->d_gden.as<double>();
        double* Wn = Ds + nn;
        aimdhf::launch_symmetrize(D, nmat, ld, Ds, st);
        aimdhf::launch_symmetrize(W, nmat, ld, Wn, st);
        aimdhf::launch_negate(Wn, nn, Wn, st);
        p->d_gfx.ensure(sizeof(long long) * 6 * p->natm);
        aimdhf::launch_zero64(p->d_gfx.as<long long>(), 6 * p->natm, st);
        p->prof.time(44, st, [&] {
            const bool one = Fan::capturing(st);
            if (!one) p->fan.fork(st);
            aimdhf::launch_grad_one(p->oneel_args(), Ds, Wn, p->d_gfx.as<long long>(),
                                    (one ? PairStreams(st) : PairStreams(p->fan)).on);
            if (!one) p->fan.join();
        });
        aimdhf::launch_fx_to_double(p->d_gfx.as<long long>(), 3 * p->natm, grad, st);
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_grad_one_noalloc(aimdhf_plan* p, const double* D, const double* W, double* grad, void* stream) {
    if (!p || !D || !W || !grad) return fail(AIMDHF_E_ARG, "NULL argument");
    if (p->batched) return fail(AIMDHF_E_UNSUPPORTED, "aimdhf_grad_one_noalloc takes single-molecule plans");
    if (p->generic) return fail(AIMDHF_E_UNSUPPORTED, "aimdhf_grad_one_noalloc takes bases with l <= 2");
    const size_t nn = (size_t)p->nao * p->nao;
    const size_t mats = (sizeof(double) * 2 * nn + 255) & ~(size_t)255;
    const size_t need = mats + sizeof(long long) * 6 * (size_t)p->natm;
    if (!p->noalloc_ptr || need > p->noalloc_bytes)
        return fail(AIMDHF_E_ARG, "aimdhf_grad_one_noalloc: nao = " + std::to_string(p->nao) + ", natm = " +
                                      std::to_string(p->natm) + " need " + std::to_string(need) +
                                      " bytes of scratch, more than its fixed " + std::to_string(p->noalloc_bytes) +
                                      " (16 nao^2 + 48 natm bytes must fit; use aimdhf_grad_one)");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    hipStream_t st = (hipStream_t)stream;
    char* base = (char*)p->noalloc_ptr;
    double* Ds = (double*)base;
    double* Wn = Ds + nn;
    long long* fx = (long long*)(base + mats);
    aimdhf::launch_symmetrize(D, 1, p->nao, Ds, st);
    aimdhf::launch_symmetrize(W, 1, p->nao, Wn, st);
    aimdhf::launch_negate(Wn, nn, Wn, st);
    aimdhf::launch_zero64(fx, 6 * (size_t)p->natm, st);     // a fill kernel: the array keeps the last call's sums
    aimdhf::launch_grad_one(p->oneel_args(), Ds, Wn, fx, PairStreams(st).on);
    aimdhf::launch_fx_to_double(fx, 3 * p->natm, grad, st);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("grad_one_noalloc: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_grad_one_terms(aimdhf_plan* p, const double* D, const double* W, double* g_kin, double* g_nuc,
                          double* g_ovl, void* stream) {
    if (!p || !D || !W || !g_kin || !g_nuc || !g_ovl) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    hipStream_t st = (hipStream_t)stream;
    try {
        if (p->generic) {
            grad_one_generic(p, D, W, 1, g_kin, st);
            grad_one_generic(p, D, W, 2, g_nuc, st);
            grad_one_generic(p, D, W, 4, g_ovl, st);
            return AIMDHF_OK;
        }
        const size_t nn = p->mat_elems();
        const int nmat = p->batched ? p->nrep : 1, ld = p->batched ? p->bld : p->nao;
        p->d_gden.ensure(sizeof(double) * 3 * nn);
        double* Ds = p->d_gden.as<double>();
        double* Wn = Ds + nn;
        double* Z = Wn + nn;
        aimdhf::launch_symmetrize(D, nmat, ld, Ds, st);
        aimdhf::launch_symmetrize(W, nmat, ld, Wn, st);
        aimdhf::launch_negate(Wn, nn, Wn, st);
        aimdhf::launch_zero_d(Z, nn, st);
        p->d_gfx.ensure(sizeof(long long) * 18 * p->natm);
        long long* fx = p->d_gfx.as<long long>();
        aimdhf::launch_zero64(fx, 18 * p->natm, st);
        aimdhf::OneElArgs g = p->oneel_args();
        // kinetic: overlap/kinetic part with W = 0; nuclear attraction alone; overlap:
        // overlap/kinetic part with D = 0 (the -W S term)
        g.parts = 1;
        aimdhf::launch_grad_one(g, Ds, Z, fx, PairStreams(st).on);
        aimdhf::launch_grad_one(g, Z, Wn, fx + 12 * p->natm, PairStreams(st).on);
        g.parts = 2;
        aimdhf::launch_grad_one(g, Ds, Z, fx + 6 * p->natm, PairStreams(st).on);
        aimdhf::launch_fx_to_double(fx, 3 * p->natm, g_kin, st);
        aimdhf::launch_fx_to_double(fx + 6 * p->natm, 3 * p->natm, g_nuc, st);
        aimdhf::launch_fx_to_double(fx + 12 * p->natm, 3 * p->natm, g_ovl, st);
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_grad_two(aimdhf_plan* p, const double* Dc, int nx, const double* Dx, double kfac, double thr,
                    double* grad, void* stream) {
    if (!p || !Dc || !Dx || !grad) return fail(AIMDHF_E_ARG, "NULL argument");
    if (nx < 1 || nx > 2) return fail(AIMDHF_E_ARG, "nx must be 1 (RHF) or 2 (UHF)");
    if (!(thr >= 0.0)) return fail(AIMDHF_E_ARG, "gradient screening threshold must be >= 0");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    hipStream_t st = (hipStream_t)stream;
    if (p->generic) return grad_two_generic(p, Dc, nx, Dx, kfac, thr, grad, st);
    try {
        const size_t nn = p->mat_elems();
        const int nmat = p->batched ? p->nrep : 1, ld = p->batched ? p->bld : p->nao;
        p->d_gden.ensure(sizeof(double) * (1 + nx) * nn);
        double* dc = p->d_gden.as<double>();
        double* dx = dc + nn;
        aimdhf::launch_symmetrize(Dc, nmat, ld, dc, st);
        aimdhf::launch_symmetrize(Dx, nmat * nx, ld, dx, st);
        // candidate quartets: q_P q_Q >= thr / max|Gamma| over every possible element
        double mc = aimdhf::device_absmax(dc, nn, p->d_scratch.as<double>(), st);
        double mx = aimdhf::device_absmax(dx, nx * nn, p->d_scratch.as<double>(), st);
        if (mc < 0.0 || mx < 0.0) return fail(AIMDHF_E_HIP, "max reduction failed");
        double gbound = 4.0 * (mc * mc + std::fabs(kfac) * nx * mx * mx);
        double lthr = gbound > 0.0 ? thr / gbound : 0.0;
        auto t0 = Profiler::clock::now();
        p->build_list(lthr, p->d_glist, p->gcount, st);
        p->prof.host(88, t0);
        p->d_gfx.ensure(sizeof(long long) * 6 * p->natm);
        aimdhf::launch_zero64(p->d_gfx.as<long long>(), 6 * p->natm, st);
        aimdhf::GradArgs a;
        a.nao = p->nao;
        a.natm = p->natm;
        a.nx = nx;
        a.kfac = kfac;
        a.thr = thr;
        a.pair_a = p->d_pair_a.as<int>();
        a.pair_b = p->d_pair_b.as<int>();
        a.shell_ao = p->d_shell_ao.as<int>();
        a.shell_atom = p->d_shell_atom.as<int>();
        a.npp = p->d_npp.as<int>();
        a.rec_off = p->d_rec_off.as<long long>();
        a.recs = p->d_recs.as<double>();
        a.boys = p->d_boys.as<double>();
        a.pos = p->d_pos.as<double>();
        a.qscr = p->d_qscr.as<double>();
        a.dc = dc;
        a.dx = dx;
        a.npair = p->npair;
        a.ld = ld;
        a.shell_rep = p->batched ? p->d_shell_rep.as<int>() : nullptr;
        a.shell_first = p->batched ? p->d_shell_first.as<int>() : nullptr;
        a.shell_pair0 = p->batched ? p->d_shell_pair0.as<int>() : nullptr;
        p->d_gdmax.ensure(sizeof(double) * (1 + nx) * std::max(p->npair, 1));
        a.dmc = p->d_gdmax.as<double>();
        a.dmx = a.dmc + p->npair;
        aimdhf::launch_pair_dmax(a, p->d_shell_l.as<int>(), p->d_gdmax.as<double>(), p->d_gdmax.as<double>() + p->npair,
                                 st);
        a.out = p->d_gfx.as<long long>();
        long long gtot = 0;
        for (int k = 0; k < NQCLASS; ++k) gtot += p->gcount[k];
        p->d_gkeep.ensure(std::max<long long>(gtot, 1));
        p->d_gsel.ensure(sizeof(int) * 2 * std::max<long long>(gtot, 1));
        p->d_nsel.ensure(sizeof(int) * 2 * NQCLASS);
        p->d_gblk.ensure(sizeof(int) * 4 * (gtot / 256 + 2 * NQCLASS));
        a.fp32_switch = p->precision == 1 ? p->grad_switch : 0.0;
        long long off = 0;
        p->fan.fork(st);
        for (int k = 0, i = 0; k < NQCLASS; ++k) {
            const int2* lst = p->d_glist.as<int2>() + off;
            hipStream_t s2 = p->gcount[k] > 0 ? p->fan.on(i++) : st;
            a.keep = p->d_gkeep.as<unsigned char>() + off;
            a.sel64 = p->d_gsel.as<int>() + off;
            a.sel32 = p->d_gsel.as<int>() + gtot + off;
            a.nsel = p->d_nsel.as<int>() + 2 * k;
            a.bcnt = p->d_gblk.as<int>() + 4 * (off / 256 + k);
            a.boff = a.bcnt + 2 * ((p->gcount[k] + 255) / 256);
            if (p->gcount[k] > 0) {
                p->prof.time(64 + k, s2, [&] { aimdhf::launch_grad_keep(k, a, lst, p->gcount[k], s2); });
                p->prof.time(21 + k, s2, [&] { aimdhf::launch_grad_one_class(k, a, lst, p->gcount[k], s2); });
            }
            off += p->gcount[k];
        }
        p->fan.join();
        aimdhf::launch_fx_to_double(p->d_gfx.as<long long>(), 3 * p->natm, grad, st);
        HIPCHECK(hipGetLastError());
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_set_jk_mode(aimdhf_plan* p, int mode, int64_t max_store_bytes) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (mode < 0 || mode > 2) return fail(AIMDHF_E_ARG, "jk mode must be 0 (auto), 1 (direct) or 2 (store)");
    if (max_store_bytes < 0) return fail(AIMDHF_E_ARG, "max_store_bytes must be >= 0");
    p->jk_mode = mode;
    p->store_limit = max_store_bytes;
    return AIMDHF_OK;
}

int aimdhf_tc2_step(int n, const double* X, const double* X2, double* Xout, double nocc, double freeze, void* stream) {
    if (n <= 0 || !X || !X2 || !Xout) return fail(AIMDHF_E_ARG, "bad tc2 arguments");
    aimdhf::launch_tc2_step(n, X, X2, Xout, nocc, freeze, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("tc2 step: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_tc2_sums(int n, const double* X, double* sums, void* stream) {
    if (n <= 0 || n > 16384 || !X || !sums) return fail(AIMDHF_E_ARG, "bad tc2 arguments");
    aimdhf::launch_tc2_sums(n, X, sums, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("tc2 sums: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_tc2_fused(int n, const double* X, double* Xout, const double* sums, double* sums_out, double nocc,
                     double freeze, void* stream) {
    if (n <= 0 || n > 16384 || !X || !Xout || X == Xout || !sums || !sums_out || sums == sums_out)
        return fail(AIMDHF_E_ARG, "bad tc2 arguments");
    aimdhf::launch_tc2_fused(n, X, Xout, sums, sums_out, nocc, freeze, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("tc2 fused: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_batch_set_jk_lanes(aimdhf_plan* p, int lanes) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (!p->batched) return fail(AIMDHF_E_STATE, "not a batched plan");
    if (lanes != 16 && lanes != 32 && lanes != 64) return fail(AIMDHF_E_ARG, "lanes must be 16, 32 or 64");
    p->batch_jk_lanes = lanes;
    return AIMDHF_OK;
}

int aimdhf_batch_purify(int nmat, int ld, const double* F, const double* nocc, double* P, int steps, double tol,
                        double* err, void* stream) {
    if (nmat < 0 || ld <= 0 || ld > 64 || steps < 0 || !(tol >= 0.0)) return fail(AIMDHF_E_ARG, "bad purify arguments");
    if (nmat == 0) return AIMDHF_OK;
    if (!F || !nocc || !P || !err) return fail(AIMDHF_E_ARG, "NULL argument");
    aimdhf::launch_batch_purify(nmat, ld, F, nocc, P, steps, tol, err, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("batch purify: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_small_fock(int nrep, int nspin, int ld, const double* H, const double* S, const double* X, const double* D,
                      const double* J, const double* K, double* F, double* Fo, double* E, int64_t rep_stride,
                      int64_t slot_stride, const int64_t* slot, double* energy, double* err, void* stream) {
    if (nrep < 0 || nspin < 1 || nspin > 2 || ld <= 0 || ld > 64) return fail(AIMDHF_E_ARG, "bad small_fock arguments");
    if (nrep == 0) return AIMDHF_OK;
    if (!H || !S || !X || !D || !J || !K || !F || !Fo || !E || !energy || !err) return fail(AIMDHF_E_ARG, "NULL argument");
    aimdhf::SmallFock a{nspin, ld, 2.0 / nspin, H, S, X, D, J, K, F, Fo, E, rep_stride, slot_stride,
                        (const long long*)slot, energy, err};
    aimdhf::launch_small_fock(a, nrep, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("small fock: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_small_diis(int nrep, int nspin, int ld, int m, const int64_t* slot, const int64_t* count, const double* E,
                      const double* Fo, double* G, const int32_t* rep_nao, double pad, double* Fx, void* stream) {
    if (nrep < 0 || nspin < 1 || nspin > 2 || ld <= 0 || ld > 64 || m < 1 || m > 12)
        return fail(AIMDHF_E_ARG, "bad small_diis arguments");
    if (nrep == 0) return AIMDHF_OK;
    if (!slot || !count || !E || !Fo || !G || !Fx) return fail(AIMDHF_E_ARG, "NULL argument");
    aimdhf::SmallDiis a{nspin, ld, m, (const long long*)slot, (const long long*)count, E, Fo, G, rep_nao, pad, Fx};
    aimdhf::launch_small_diis(a, nrep, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("small diis: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_small_density(int nrep, int nspin, int ld, const double* X, const double* P, double* D, uint8_t* frozen,
                         const double* energy, const double* err, double* e_prev, double conv_e, double conv_g,
                         int64_t* slot, int64_t* count, int m, void* stream) {
    if (nrep < 0 || nspin < 1 || nspin > 2 || ld <= 0 || ld > 64) return fail(AIMDHF_E_ARG, "bad small_density arguments");
    if (nrep == 0) return AIMDHF_OK;
    if (!X || !P || !D || (frozen && (!energy || !err || !e_prev)) || (slot && (!count || m < 1)))
        return fail(AIMDHF_E_ARG, "NULL argument");
    aimdhf::SmallDensity a{nspin, ld, X, P, D, frozen, energy, err, e_prev, conv_e, conv_g, (long long*)slot,
                           (long long*)count, m};
    aimdhf::launch_small_density(a, nrep, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("small density: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_small_inv_sqrt(int nmat, int ld, const double* S, double* X, int iters, double tol, double* out, void* stream) {
    if (nmat < 0 || ld <= 0 || ld > 64 || iters < 1 || !(tol >= 0.0)) return fail(AIMDHF_E_ARG, "bad small_inv_sqrt arguments");
    if (nmat == 0) return AIMDHF_OK;
    if (!S || !X || !out) return fail(AIMDHF_E_ARG, "NULL argument");
    aimdhf::launch_small_inv_sqrt(nmat, ld, S, X, iters, tol, out, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("small inv_sqrt: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_batch_diis_solve(int nrep, int m, const double* G, const double* r, double* c, void* stream) {
    if (nrep < 0 || m <= 0 || m > 12) return fail(AIMDHF_E_ARG, "bad DIIS solve arguments (1 <= m <= 12)");
    if (nrep == 0) return AIMDHF_OK;
    if (!G || !r || !c) return fail(AIMDHF_E_ARG, "NULL argument");
    aimdhf::launch_batch_diis_solve(nrep, m, G, r, c, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("batch DIIS solve: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_tc2_init(int n, const double* F, double* X0, void* stream) {
    if (n <= 0 || !F || !X0) return fail(AIMDHF_E_ARG, "bad tc2 arguments");
    aimdhf::launch_tc2_init(n, F, X0, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("tc2 init: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_tc2_error(int n, const double* X, double* err, void* stream) {
    if (n <= 0 || !X || !err) return fail(AIMDHF_E_ARG, "bad tc2 arguments");
    aimdhf::launch_tc2_error(n, X, err, (hipStream_t)stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(AIMDHF_E_HIP, std::string("tc2 error: ") + hipGetErrorString(e));
    return AIMDHF_OK;
}

int aimdhf_set_streams(aimdhf_plan* p, int concurrent) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    p->fan.serial = concurrent == 0;
    return AIMDHF_OK;
}

int aimdhf_set_precision(aimdhf_plan* p, int mode, double jk_switch, double grad_switch, double delta_switch) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (mode < 0 || mode > 1) return fail(AIMDHF_E_ARG, "precision mode must be 0 (fp64) or 1 (mixed)");
    if (!(jk_switch >= 0.0) || !(grad_switch >= 0.0) || !(delta_switch >= 0.0))
        return fail(AIMDHF_E_ARG, "switch thresholds must be >= 0");
    p->precision = mode;
    p->jk_switch = jk_switch;
    p->grad_switch = grad_switch;
    return AIMDHF_OK;
}

int aimdhf_set_store_units(aimdhf_plan* p, int items) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (items < 64 || items > (1 << 16)) return fail(AIMDHF_E_ARG, "store work units take 64 .. 65536 lane items");
    p->unit_items = items;
    return AIMDHF_OK;
}

int aimdhf_jk_info(aimdhf_plan* p, int* stored, int64_t* store_bytes, int64_t* k_entries, int64_t* j_entries,
                   int64_t* gather_bytes) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    if (stored) *stored = p->stored ? 1 : 0;
    if (gather_bytes) *gather_bytes = p->stored ? (int64_t)p->store_need : 0;
    if (store_bytes) *store_bytes = p->store_bytes;
    if (k_entries) *k_entries = p->stored ? p->qtotal : 0;
    if (j_entries) *j_entries = 0;
    return AIMDHF_OK;
}

int aimdhf_jk_type_info(aimdhf_plan* p, int64_t* k_bytes, int64_t* k_entries, int64_t* j_bytes, int64_t* j_entries,
                        int64_t* unique_bytes) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    for (int k = 0; unique_bytes && k < NQCLASS; ++k)
        unique_bytes[k] = p->stored ? aimdhf::store_block(k) * (8 * p->q64count[k] + 4 * (p->qcount[k] - p->q64count[k])) : 0;
    for (int t = 0; t < 9; ++t) {
        if (k_bytes) k_bytes[t] = 0;
        if (k_entries) k_entries[t] = 0;
    }
    for (int c = 0; c < 6; ++c) {
        if (j_bytes) j_bytes[c] = 0;
        if (j_entries) j_entries[c] = 0;
    }
    return AIMDHF_OK;
}

int aimdhf_profile_enable(aimdhf_plan* p, int on) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    try {
        p->prof.collect();
    } catch (const HipError& e) {
        return e.code;
    }
    p->prof.on = on != 0;
    return AIMDHF_OK;
}

int aimdhf_profile_replay(aimdhf_plan* p, int kind, int reps, void* stream, double* avg_ms) {
    if (!p || !avg_ms) return fail(AIMDHF_E_ARG, "NULL argument");
    if (reps < 1) return fail(AIMDHF_E_ARG, "reps must be >= 1");
    const int k = kind - 98;
    if (k < 0 || k >= NQCLASS) return fail(AIMDHF_E_UNSUPPORTED, "replay covers the store-mode digestion kinds 98..118");
    if (!p->have_geometry || !p->stored || !p->have_last_store || !p->qcount[k])
        return fail(AIMDHF_E_STATE, "replay needs a store-mode J/K build at the current geometry");
    hipStream_t st = (hipStream_t)stream;
    hipEvent_t a = nullptr, b = nullptr;
    try {
        HIPCHECK(hipEventCreate(&a));
        HIPCHECK(hipEventCreate(&b));
        // the digestion adds to accumulators that every build clears: replays leave J and K alone
        HIPCHECK(hipEventRecord(a, st));
        for (int r = 0; r < reps; ++r) aimdhf::launch_digest(k, p->last_dig[k], 256, st);
        HIPCHECK(hipEventRecord(b, st));
        HIPCHECK(hipEventSynchronize(b));
        float ms = 0.0f;
        HIPCHECK(hipEventElapsedTime(&ms, a, b));
        *avg_ms = ms / reps;
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
    } catch (const HipError& e) {
        if (a) (void)hipEventDestroy(a);
        if (b) (void)hipEventDestroy(b);
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_profile_read(aimdhf_plan* p, double* ms, int64_t* launches, int nkind, int reset) {
    if (!p || !ms || !launches) return fail(AIMDHF_E_ARG, "NULL argument");
    try {
        p->prof.collect();
        for (int i = 0; i < nkind && i < Profiler::NKIND; ++i) {
            ms[i] = p->prof.ms[i];
            launches[i] = p->prof.n[i];
        }
        if (reset) p->prof.reset();
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

int aimdhf_class_counts(aimdhf_plan* p, int64_t* energy_counts, int64_t* gradient_counts) {
    if (!p) return fail(AIMDHF_E_ARG, "NULL plan");
    for (int k = 0; k < NQCLASS; ++k) {
        if (energy_counts) energy_counts[k] = k < (int)p->qcount.size() ? p->qcount[k] : 0;
        if (gradient_counts) gradient_counts[k] = k < (int)p->gcount.size() ? p->gcount[k] : 0;
    }
    return AIMDHF_OK;
}

int aimdhf_pair_npp(aimdhf_plan* p, int32_t* npp_host, int64_t cap) {
    if (!p || !npp_host) return fail(AIMDHF_E_ARG, "NULL argument");
    if (!p->have_geometry) return fail(AIMDHF_E_STATE, "no geometry set");
    if (cap < p->npair) return fail(AIMDHF_E_ARG, "output too small");
    if (p->generic) {
        for (int P = 0; P < p->npair; ++P) npp_host[P] = p->gen_npp[P];
        return AIMDHF_OK;
    }
    try {
        HIPCHECK(hipMemcpy(npp_host, p->d_npp.p, sizeof(int) * p->npair, hipMemcpyDeviceToHost));
    } catch (const HipError& e) {
        return e.code;
    }
    return AIMDHF_OK;
}

}  // extern "C"
