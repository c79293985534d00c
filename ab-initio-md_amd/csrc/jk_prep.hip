// Around the J/K digestion of one build: symmetrised densities, densities by
// ranked pair component, the magnitudes that set the fixed-point exponents and
// the cleared accumulators before it (one launch), J and K from the
// accumulators after it (one launch).

#include "aimdhf_internal.h"
#include "jk_digest.h"

namespace aimdhf {

namespace {

__device__ __forceinline__ int nc_of(int c) {   // Cartesian components of a pair class' second shell
    return c == 0 || c == 1 || c == 3 ? 1 : c == 5 ? 6 : 3;
}

// rank and component of pair-component index e (component-major within a class)
struct PairComp {
    int cls, rank, comp, stride;
};
__device__ __forceinline__ PairComp pair_comp(const PrepArgs& a, long long e) {
    PairComp p;
    p.cls = 0;
    while (p.cls < 5 && e >= a.koff[p.cls + 1]) ++p.cls;
    p.stride = a.cls_off[p.cls + 1] - a.cls_off[p.cls];
    const long long r = e - a.koff[p.cls];
    p.comp = (int)(r / p.stride);
    p.rank = a.cls_off[p.cls] + (int)(r % p.stride);
    return p;
}

// blocks [0, nrow): four rows of one density each (a wavefront per row); then the
// pair components; then clearing, grid-stride
__global__ __launch_bounds__(256) void k_jk_prep(PrepArgs a, int nrow, int npc) {
    const int b = blockIdx.x;
    const size_t ld = a.ld, ld2 = ld * ld;
    if (b < nrow) {
        const int t = b * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
        if (t >= a.nrep * a.nset * a.ld) return;
        const int mat = t / a.ld, r = t % a.ld;
        const double* D = a.dens + mat * ld2;
        double s1 = 0.0, s2 = 0.0, mx = 0.0;
        for (int c = lane; c < a.ld; c += 64) {
            const double v = 0.5 * (D[r * ld + c] + D[c * ld + r]);
            a.dsym[mat * ld2 + r * ld + c] = v;
            s1 += fabs(v);
            s2 += v * v;
            mx = v != v ? fabs(v) : fmax(mx, fabs(v));
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            s1 += __shfl_xor(s1, o, 64);
            s2 += __shfl_xor(s2, o, 64);
            mx = fmax(mx, __shfl_xor(mx, o, 64));
        }
        if (lane == 0) {
            // max of the bit patterns of non-negative doubles: order-independent, and a
            // NaN (cleared sign) is larger than every number
            unsigned long long* c = a.dcell + JK_CELLS * mat;
            atomicMax(c, (unsigned long long)__double_as_longlong(fabs(s1)));
            atomicMax(c + 1, (unsigned long long)__double_as_longlong(fabs(s2)));
            atomicMax(c + 2, (unsigned long long)__double_as_longlong(mx));
        }
        return;
    }
    if (b < nrow + npc) {
        const long long e = (long long)(b - nrow) * 256 + threadIdx.x;
        const bool in = e < a.npao;
        const PairComp p = pair_comp(a, in ? e : a.npao - 1);
        const unsigned o = a.oab[p.rank];
        const int nb = nc_of(p.cls);
        const size_t m = oab_first(o) + p.comp / nb, n = oab_second(o) + p.comp % nb;
        const int rep = a.rank_rep ? a.rank_rep[p.rank] : 0;
        const bool one = __all(rep == __shfl(rep, 0, 64));
        for (int s = 0; s < a.nset; ++s) {
            const size_t mat = (size_t)rep * a.nset + s;
            const double* D = a.dens + mat * ld2;
            const double d = 0.5 * (D[m * ld + n] + D[n * ld + m]);
            if (in) a.dket[s * a.npao + e] = d;
            // sum of q |D| over AO pairs in both orders, in integers (order-independent)
            unsigned long long x = 0;
            if (in) x = (unsigned long long)ceil(fmin(fabs(d) * a.rq[p.rank] * (oab_same(o) ? 1.0 : 2.0), 1e10) * 16777216.0);
            unsigned long long* cell = a.dcell + JK_CELLS * mat + 3;
            if (one) {
#pragma unroll
                for (int h = 32; h >= 1; h >>= 1) x += __shfl_xor(x, h, 64);
                if ((threadIdx.x & 63) == 0) atomicAdd(cell, x);
            } else if (x)
                atomicAdd(cell, x);
        }
        return;
    }
    const size_t nk = (size_t)a.ncopy * a.kstride, nj = (size_t)a.ncopy * a.nset * a.npao;
    const size_t step = (size_t)(gridDim.x - nrow - npc) * 256;
    for (size_t i = (size_t)(b - nrow - npc) * 256 + threadIdx.x; i < nk + nj; i += step)
        (i < nk ? a.kacc[i] : a.jacc[i - nk]) = 0ull;
}

__device__ __forceinline__ double from_fixed(unsigned long long v, double inv) { return (double)(long long)v * inv; }

// K = A + A^T (threads over matrix elements), then J (threads over pair components)
__global__ __launch_bounds__(256) void k_jk_finish(PrepArgs a, int nkb) {
    const size_t ld = a.ld, ld2 = ld * ld;
    const double nan = __longlong_as_double(0x7ff8000000000000ll);
    if ((int)blockIdx.x < nkb) {
        const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
        if (i >= (size_t)a.kstride) return;
        const size_t mat = i / ld2, r = i % ld2, m = r / ld, n = r % ld;
        const size_t rep = mat / a.nset, ji = mat * ld2 + n * ld + m;
        const int nao = a.rep_nao ? a.rep_nao[rep] : a.ld;
        if ((int)m >= nao || (int)n >= nao) {
            a.K[i] = 0.0;
            a.J[i] = 0.0;
            return;
        }
        unsigned long long v = 0;
        for (int c = 0; c < a.ncopy; ++c) v += a.kacc[c * a.kstride + i] + a.kacc[c * a.kstride + ji];
        const double bound = jk_bound_k(a.gcell + 3 * rep, a.dcell + JK_CELLS * mat);
        a.K[i] = isfinite(bound) ? from_fixed(v, ldexp(1.0, -jk_exponent(bound))) : nan;
        return;
    }
    const long long e = (long long)(blockIdx.x - nkb) * 256 + threadIdx.x;
    if (e >= a.npao) return;
    const PairComp p = pair_comp(a, e);
    const unsigned o = a.oab[p.rank];
    const int nb = nc_of(p.cls);
    const int i = p.comp / nb, j = p.comp % nb;
    const bool same = oab_same(o);
    const size_t m = oab_first(o) + i, n = oab_second(o) + j;
    const size_t rep = a.rank_rep ? a.rank_rep[p.rank] : 0;
    const long long et = same ? e + (long long)((j * nb + i) - p.comp) * p.stride : e;
    for (int s = 0; s < a.nset; ++s) {
        unsigned long long v = 0;
        for (int c = 0; c < a.ncopy; ++c) {
            const unsigned long long* acc = a.jacc + ((size_t)c * a.nset + s) * a.npao;
            v += acc[e];
            if (same) v += acc[et];
        }
        const size_t mat = rep * a.nset + s;
        const double bound = jk_bound_j(a.gcell + 3 * rep, a.dcell + JK_CELLS * mat, a.rep_nao ? a.rep_nao[rep] : a.ld);
        const double x = isfinite(bound) ? from_fixed(v, ldexp(1.0, -jk_exponent(bound))) : nan;
        double* J = a.J + mat * ld2;
        J[m * ld + n] = x;
        J[n * ld + m] = x;
    }
}

__global__ void k_clear_cells(unsigned long long* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

__global__ void k_zero_d(double* p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

}  // namespace

void launch_zero_d(double* p, size_t n, hipStream_t st) {
    if (n) k_zero_d<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(p, n);
}

void launch_jk_prep(const PrepArgs& a, hipStream_t st) {
    const int ncell = JK_CELLS * a.nrep * a.nset;
    k_clear_cells<<<dim3((ncell + 255) / 256), dim3(256), 0, st>>>(a.dcell, ncell);
    const int nrow = (a.nrep * a.nset * a.ld + 3) / 4, npc = (int)((a.npao + 255) / 256);
    const long long words = (long long)a.ncopy * (a.kstride + a.nset * a.npao);
    const long long nz = (words + 1023) / 1024;
    k_jk_prep<<<dim3((unsigned)(nrow + npc + (nz > 2048 ? 2048 : nz))), dim3(256), 0, st>>>(a, nrow, npc);
}

void launch_jk_finish(const PrepArgs& a, hipStream_t st) {
    const int nkb = (int)((a.kstride + 255) / 256), njb = (int)((a.npao + 255) / 256);
    k_jk_finish<<<dim3((unsigned)(nkb + njb)), dim3(256), 0, st>>>(a, nkb);
}

}  // namespace aimdhf
