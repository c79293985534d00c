// J and K from the integral store: the digestion of one bra pair's run of kets of a
// quartet class. Every stored integral is read once per build.
//
// One workgroup digests (part of) the run of one bra pair (I, J): all kets (K, L)
// of the class. Everything K receives from such a run lies in the rows of I and
// J, so those rows of K are held in LDS as 64-bit integers next to the same rows
// of the density, and flushed once. A lane holds one ket (or one ket and one
// component of K for the heavy kets) and walks its columns kl:
//   K_ik += (ij|kl) D_jl   K_il += (ij|kl) D_jk   K_jk += (ij|kl) D_il   K_jl += (ij|kl) D_ik
//   J_ij += 2 (ij|kl) D_kl                        J_kl += 2 (ij|kl) D_ij
// halved for I = J, K = L and equal pairs; K = A + A^T afterwards. Lane sums are
// FP64; what leaves a lane is rounded to 64-bit fixed point (jk_digest.h), so the
// integer sums, and J and K, do not depend on the order of arrival. Kets are
// ranked along the diagonals of the pair triangle, so the 64 lanes of a
// wavefront name different K and different L: their LDS additions rarely meet.
// The J of the kets goes to global accumulators in rank order (coalesced); both
// kinds of global accumulators are kept in copies, one per XCD's workgroups.

#pragma once
#include "jk_digest.h"
#include "md_core.h"

namespace aimdhf {
using namespace md;

namespace {
constexpr int pc_hi(int qc) { int h = 0; while ((h + 1) * (h + 2) / 2 <= qc) ++h; return h; }
constexpr int pc_lo(int qc) { return qc - pc_hi(qc) * (pc_hi(qc) + 1) / 2; }
constexpr int la_of(int pc) { return pc == 0 ? 0 : pc <= 2 ? 1 : 2; }
constexpr int lb_of(int pc) { return pc - la_of(pc) * (la_of(pc) + 1) / 2; }
constexpr int JSLOT = 16;       // LDS words per component of the bra's J

// shapes of quartet class QC
template <int QC>
struct Dig {
    static constexpr int CB = pc_hi(QC), CK = pc_lo(QC);
    static constexpr int NA = NC(la_of(CB)), NB = NC(lb_of(CB)), NCc = NC(la_of(CK)), ND = NC(lb_of(CK));
    static constexpr int NAB = NA * NB, NCD = NCc * ND, BLK = NAB * NCD, NR = NA + NB;
    // lanes per ket: one per component of K where the column sums of a whole ket
    // would not fit the registers
    static constexpr int SP = CK >= 4 ? NCc : 1;
    // words of a column of the bra's rows in LDS (Rows)
    static constexpr int colw(int nset) { return 2 * NR * nset + 1; }
    // bytes of LDS ahead of the columns: the bra's density block and J sums
    static constexpr int head(int nset) { return nset * NAB * (JSLOT + 1); }
};

__device__ __forceinline__ void add64(unsigned long long* p, unsigned long long v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void add64_dev(unsigned long long* p, unsigned long long v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// per AO column: for each set the NR rows of K (integers), then the NR rows of the
// density; an odd number of words per column, so neighbouring columns start in
// different banks, and one address per column serves every row
extern __shared__ unsigned long long dig_lds[];
// LDSROWS: the K and D rows of the bra in LDS; otherwise (matrices too large for
// that) D is read from memory and K added to the global accumulators directly
template <int QC, int NSET, bool LDSROWS>
struct Rows {
    static constexpr int NA = Dig<QC>::NA, NR = Dig<QC>::NR, W = Dig<QC>::colw(NSET), C0 = Dig<QC>::head(NSET);
    int ld;
    const double* D[NSET];          // dsym of each set
    unsigned long long* Kg[NSET];
    double sk[NSET];
    int oI, oJ;
    __device__ __forceinline__ int row(int r) const { return r < NA ? oI + r : oJ + (r - NA); }
    __device__ __forceinline__ double d(int s, int r, int c) const {
        if constexpr (LDSROWS)
            return __longlong_as_double((long long)dig_lds[C0 + c * W + (2 * s + 1) * NR + r]);
        return D[s][(size_t)row(r) * ld + c] * sk[s];
    }
    __device__ __forceinline__ void add(int s, int r, int c, double x) const {
        const unsigned long long v = jk_fixed(x);
        if constexpr (LDSROWS) add64(&dig_lds[C0 + c * W + 2 * s * NR + r], v);
        else add64_dev(&Kg[s][(size_t)row(r) * ld + c], v);
    }
};

// quartets [t0, t1) of one precision part (tb: the part's first list index)
template <int QC, typename Real, int NSET, bool LDSROWS>
__device__ __forceinline__ void digest_part(const DigestArgs& a, const Rows<QC, NSET, LDSROWS>& R,
                                            const Real* __restrict__ blocks,
                                            const int* __restrict__ lket, long long tb, long long t0, long long t1,
                                            int rank, double wbra, const double* sj, const double* dij,
                                            const int copy, const int set0, const double qb,
                                            double (&jacc)[NSET][Dig<QC>::NAB]) {
    using S = Dig<QC>;
    constexpr int CB = S::CB, CK = S::CK, NA = S::NA, NB = S::NB, NCc = S::NCc, ND = S::ND, NAB = S::NAB, BLK = S::BLK,
                  NR = S::NR, SP = S::SP;
    const int ket0 = a.cls_off[CK], nk = a.cls_off[CK + 1] - ket0;
    const long long kket = a.koff[CK];
    const int n = (int)(t1 - t0), nit = n * SP;
    auto ket_at = [&](int it) { return lket[t0 + (SP > 1 ? it % n : it)]; };
    // the ket and its AO offsets run one item ahead, so that an item's loads and
    // LDS addresses do not wait for them
    int kr_next = 0;
    unsigned o_next = 0;
    if ((int)threadIdx.x < nit) {
        kr_next = ket_at(threadIdx.x);
        o_next = a.oab[kr_next];
    }
    for (int it = threadIdx.x; it < nit; it += blockDim.x) {
        const int c0 = SP > 1 ? it / n : 0;
        const int tt = SP > 1 ? it - c0 * n : it;
        const int kr = kr_next;
        const unsigned o = o_next;
        const int it2 = it + blockDim.x;
        if (it2 < nit) {
            kr_next = ket_at(it2);
            o_next = a.oab[kr_next];
        }
        // a density difference below the threshold for all 64 kets of the wavefront
        if (a.delta && !__any(!(qb * a.rq[kr] < a.dthr))) continue;
        const int oK = oab_first(o), oL = oab_second(o);
        double w = oab_same(o) ? 0.5 * wbra : wbra;
        if (CB == CK && kr == rank) w *= 0.5;
        const long long t = t0 + tt - tb;
        const Real* __restrict__ p = blocks + (t >> 6) * (64 * BLK) + (t & 63);
        const size_t je = (size_t)(kr - ket0);
        double kl[NSET][SP > 1 ? 1 : ND][NR];
        if constexpr (SP == 1) {
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int l = 0; l < ND; ++l)
#pragma unroll
                    for (int r = 0; r < NR; ++r) kl[s][l][r] = 0.0;
        }
#pragma unroll 1
        for (int c = c0; c < (SP > 1 ? c0 + 1 : NCc); ++c) {
            double kk[NSET][NR];
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int r = 0; r < NR; ++r) kk[s][r] = 0.0;
#pragma unroll
            for (int l = 0; l < ND; ++l) {
                const int cd = c * ND + l;
                double v[NAB];
#pragma unroll
                for (int i = 0; i < NAB; ++i) v[i] = double(__builtin_nontemporal_load(p + (cd * NAB + i) * 64));
#pragma unroll
                for (int s = 0; s < NSET; ++s) {
                    const double dkl = a.dket[(set0 + s) * a.npao + kket + (long long)cd * nk + je] * (2.0 * w * sj[s]);
                    double jkl = 0.0;
#pragma unroll
                    for (int i = 0; i < NAB; ++i) {
                        jacc[s][i] += v[i] * dkl;
                        jkl += v[i] * dij[s * NAB + i];
                    }
                    add64_dev(a.jacc + ((size_t)copy * a.nset + set0 + s) * a.npao + kket + (long long)cd * nk + je,
                              jk_fixed(jkl * (2.0 * w)));
                    double dk[NR], dl[NR];
#pragma unroll
                    for (int r = 0; r < NR; ++r) {
                        dk[r] = R.d(s, r, oK + c);
                        dl[r] = R.d(s, r, oL + l);
                    }
                    double x[NR];
#pragma unroll
                    for (int r = 0; r < NR; ++r) x[r] = 0.0;
#pragma unroll
                    for (int i = 0; i < NA; ++i)
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
                            const double e = v[i * NB + j];
                            kk[s][i] += e * dl[NA + j];
                            kk[s][NA + j] += e * dl[i];
                            x[i] += e * dk[NA + j];
                            x[NA + j] += e * dk[i];
                        }
#pragma unroll
                    for (int r = 0; r < NR; ++r) {
                        if constexpr (SP > 1) R.add(s, r, oL + l, x[r] * w);
                        else kl[s][l][r] += x[r];
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int r = 0; r < NR; ++r) R.add(s, r, oK + c, kk[s][r] * w);
        }
        if constexpr (SP == 1) {
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int l = 0; l < ND; ++l)
#pragma unroll
                    for (int r = 0; r < NR; ++r) R.add(s, r, oL + l, kl[s][l][r] * w);
        }
    }
}

// the run of bra bi of its class (piece `chunk`, precision part `part`) for densities
// set0 .. set0 + NSET - 1
template <int QC, int NSET, bool LDSROWS>
__device__ __forceinline__ void digest_run(const DigestArgs& a, int bi, int part, int chunk, int set0, int copy) {
    using S = Dig<QC>;
    constexpr int CB = S::CB, NAB = S::NAB, NR = S::NR, W = S::colw(NSET), C0 = S::head(NSET);
    double* sD = (double*)dig_lds;
    unsigned long long* sJ = dig_lds + NSET * NAB;
    const int bra0 = a.cls_off[CB], nb = a.cls_off[CB + 1] - bra0;
    const long long kbra = a.koff[CB];
    const long long run = (long long)part * nb + bi;
    const DigestGeo g = a.geo[QC];
    long long t0 = g.off[run * LIST_WAVES], t1 = g.off[(run + 1) * LIST_WAVES];
    const long long lo = part ? g.lo32 : g.lo64, hi = part ? g.hi32 : g.hi64;
    if (t0 < lo) t0 = lo;
    if (t1 > hi) t1 = hi;
    if (a.nchunk > 1) {
        long long per = (t1 - t0 + a.nchunk - 1) / a.nchunk;
        if (per < a.unit) per = a.unit;
        const long long b = t0 + chunk * per;
        if (b + per < t1) t1 = b + per;
        t0 = b;
    }
    if (t0 >= t1) return;
    const int rank = bra0 + bi;
    const int rep = a.rank_rep ? a.rank_rep[rank] : 0;
    const size_t ld2 = (size_t)a.ld * a.ld;
    const int nao = a.rep_nao ? a.rep_nao[rep] : a.ld;
    const unsigned o = a.oab[rank];
    double sj[NSET], dm = 0.0;
    Rows<QC, NSET, LDSROWS> R;
    R.ld = a.ld;
    R.oI = oab_first(o);
    R.oJ = oab_second(o);
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
        const size_t mat = (size_t)rep * a.nset + set0 + s;
        const unsigned long long* dc = a.dcell + JK_CELLS * mat;
        const unsigned long long* gc = a.gcell + 3 * rep;
        R.D[s] = a.dsym + mat * ld2;
        R.Kg[s] = a.kacc + (size_t)copy * a.kstride + mat * ld2;
        R.sk[s] = jk_scale(jk_bound_k(gc, dc));
        sj[s] = jk_scale(jk_bound_j(gc, dc, nao));
        dm = fmax(dm, __longlong_as_double((long long)dc[2]));
    }
    double qb = 0.0;
    if (a.delta) {
        qb = a.rq[rank] * dm;
        // no ket of the class can reach the threshold (q_Q <= the replica's largest)
        if (qb * __longlong_as_double((long long)a.gcell[3 * rep]) < a.dthr) return;
    }
    if constexpr (LDSROWS) {
        for (int c = threadIdx.x; c < a.ld; c += blockDim.x)
#pragma unroll
            for (int x = 0; x < NSET; ++x)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    unsigned long long* w = dig_lds + C0 + c * W + 2 * x * NR + r;
                    w[0] = 0ull;
                    w[NR] = (unsigned long long)__double_as_longlong(R.D[x][(size_t)R.row(r) * a.ld + c] * R.sk[x]);
                }
    }
    for (int i = threadIdx.x; i < NSET * NAB * JSLOT; i += blockDim.x) sJ[i] = 0ull;
    for (int i = threadIdx.x; i < NSET * NAB; i += blockDim.x) {
        const int s = i / NAB, ab = i % NAB;
        sD[i] = a.dket[(set0 + s) * a.npao + kbra + (long long)ab * nb + bi] * (s ? sj[NSET - 1] : sj[0]);
    }
    __syncthreads();
    const double wbra = oab_same(o) ? 0.5 : 1.0;
    double jacc[NSET][NAB];
#pragma unroll
    for (int s = 0; s < NSET; ++s)
#pragma unroll
        for (int i = 0; i < NAB; ++i) jacc[s][i] = 0.0;
    if (part == 0)
        digest_part<QC, double, NSET, LDSROWS>(a, R, g.s64, g.lket, g.t64, t0, t1, rank, wbra, sj, sD, copy, set0, qb, jacc);
    else
        digest_part<QC, float, NSET, LDSROWS>(a, R, g.s32, g.lket, g.t32, t0, t1, rank, wbra, sj, sD, copy, set0, qb, jacc);
#pragma unroll
    for (int s = 0; s < NSET; ++s)
#pragma unroll
        for (int i = 0; i < NAB; ++i)
            add64(&sJ[(s * NAB + i) * JSLOT + (threadIdx.x & (JSLOT - 1))], jk_fixed(jacc[s][i]));
    __syncthreads();
    for (int i = threadIdx.x; i < NSET * NAB; i += blockDim.x) {
        const int s = i / NAB, ab = i % NAB;
        unsigned long long v = 0;
        for (int k = 0; k < JSLOT; ++k) v += sJ[i * JSLOT + k];
        if (v) add64_dev(a.jacc + ((size_t)copy * a.nset + set0 + s) * a.npao + kbra + (long long)ab * nb + bi, v);
    }
    if constexpr (LDSROWS) {
        for (int c = threadIdx.x; c < a.ld; c += blockDim.x)
#pragma unroll
            for (int x = 0; x < NSET; ++x)
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const unsigned long long v = dig_lds[C0 + c * W + 2 * x * NR + r];
                    if (v) add64_dev(&R.Kg[x][(size_t)R.row(r) * a.ld + c], v);
                }
    }
}

}  // namespace
}  // namespace aimdhf
