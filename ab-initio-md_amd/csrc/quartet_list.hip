// Screened quartet list: for every bra pair the kets of each lighter or equal
// pair class with q_P q_Q >= thr (the test of aimd/qc/integrals.py:902), in
// rank order, split in mixed precision into the part held in FP64 (q_P q_Q >=
// sw) and the rest. One workgroup per bra, each of its wavefronts a contiguous
// quarter of every ket segment, so the ordered fill needs no synchronisation:
// ballots and one running offset per wavefront and part.

#include "jk_digest.h"

namespace aimdhf {

namespace {

__device__ __forceinline__ int class_of_rank(const int* cls_off, int r) {
    int c = 0;
#pragma unroll
    for (int i = 1; i < 6; ++i) c += r >= cls_off[i];
    return c;
}

// f(k, lo, hi, cell): this wavefront's quarter of the kets of class k
template <class F>
__device__ __forceinline__ void for_segments(const QListArgs& a, int rank, int w, F&& f) {
    const int cb = class_of_rank(a.cls_off, rank);
    const int rep = a.rank_rep ? a.rank_rep[rank] : 0;
    for (int ck = 0; ck <= cb; ++ck) {
        const int s0 = a.seg[ck * a.nrep + rep], hi = a.seg[ck * a.nrep + rep + 1];
        const int lo = ck == cb ? rank : s0;
        const int per = (hi - lo + LIST_WAVES - 1) / LIST_WAVES;
        const int b0 = lo + w * per, b1 = b0 + per < hi ? b0 + per : hi;
        const int k = cb * (cb + 1) / 2 + ck;
        const long long run = a.runbase[k] + (rank - a.cls_off[cb]);
        f(b0, b1, run, (long long)(a.cls_off[cb + 1] - a.cls_off[cb]));
    }
}

__device__ __forceinline__ void qlist_count(const QListArgs& a, int rank) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double qb = a.rq[rank];
    for_segments(a, rank, w, [&](int b0, int b1, long long run, long long nb) {
        long long c0 = 0, c1 = 0;
        for (int i = b0; i < b1; i += 256) {
            double q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = i + 64 * u + lane;
                q[u] = j < b1 ? qb * a.rq[j] : -1.0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool in = i + 64 * u + lane < b1 && !(q[u] < a.thr);
                const unsigned long long m = __ballot(in);
                if (a.nparts == 2) {
                    const unsigned long long m1 = __ballot(in && q[u] < a.sw);
                    c1 += __popcll(m1);
                    c0 += __popcll(m & ~m1);
                } else
                    c0 += __popcll(m);
            }
        }
        if (lane == 0) {
            a.cnt[run * LIST_WAVES + w] = c0;
            if (a.nparts == 2) a.cnt[(run + nb) * LIST_WAVES + w] = c1;
        }
    });
}

__device__ __forceinline__ void qlist_fill(const QListArgs& a, int rank) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double qb = a.rq[rank];
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    for_segments(a, rank, w, [&](int b0, int b1, long long run, long long nb) {
        if (b0 >= b1) return;
        long long o0 = a.off[run * LIST_WAVES + w];
        long long o1 = a.nparts == 2 ? a.off[(run + nb) * LIST_WAVES + w] : 0;
        for (int i = b0; i < b1; i += 256) {
            double q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = i + 64 * u + lane;
                q[u] = j < b1 ? qb * a.rq[j] : -1.0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = i + 64 * u + lane;
                const bool in = j < b1 && !(q[u] < a.thr);
                const bool lo = in && a.nparts == 2 && q[u] < a.sw;
                const unsigned long long m = __ballot(in), m1 = __ballot(lo), m0 = m & ~m1;
                if (in) {
                    const long long at = lo ? o1 + __popcll(m1 & below) : o0 + __popcll(m0 & below);
                    a.lbra[at] = rank;
                    a.lket[at] = j;
                }
                o0 += __popcll(m0);
                o1 += __popcll(m1);
            }
        }
    });
}

__global__ __launch_bounds__(64 * LIST_WAVES) void k_qlist_count(QListArgs a) {
    for (int rank = blockIdx.x; rank < a.npair; rank += gridDim.x) qlist_count(a, rank);
}

__global__ __launch_bounds__(64 * LIST_WAVES) void k_qlist_fill(QListArgs a) {
    for (int rank = blockIdx.x; rank < a.npair; rank += gridDim.x) qlist_fill(a, rank);
}

// three-pass exclusive scan: block scans, a scan of the block totals, the add
constexpr int SCAN_T = 1024, SCAN_V = 4, SCAN_B = SCAN_T * SCAN_V;

__device__ long long block_scan(long long v, long long* wsum, long long& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    long long x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const long long t = __shfl_up(x, o, 64);
        if (lane >= o) x += t;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
        long long s = lane < SCAN_T / 64 ? wsum[lane] : 0;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const long long t = __shfl_up(s, o, 64);
            if (lane >= o) s += t;
        }
        if (lane < SCAN_T / 64) wsum[lane] = s;
    }
    __syncthreads();
    total = wsum[SCAN_T / 64 - 1];
    const long long before = w ? wsum[w - 1] : 0;
    __syncthreads();
    return before + x - v;
}

__global__ __launch_bounds__(SCAN_T) void k_scan_block(const long long* in, long long* out, long long n, long long* bsum) {
    __shared__ long long wsum[SCAN_T / 64];
    const long long i0 = (long long)blockIdx.x * SCAN_B + threadIdx.x * SCAN_V;
    long long v[SCAN_V], s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_V; ++k) {
        v[k] = i0 + k < n ? in[i0 + k] : 0;
        s += v[k];
    }
    long long total;
    long long p = block_scan(s, wsum, total);
#pragma unroll
    for (int k = 0; k < SCAN_V; ++k) {
        if (i0 + k < n) out[i0 + k] = p;
        p += v[k];
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

// exclusive scan of the block totals in place (one workgroup, SCAN_B at a time)
__global__ __launch_bounds__(SCAN_T) void k_scan_sums(long long* bsum, long long nb, long long* out, long long n) {
    __shared__ long long wsum[SCAN_T / 64];
    long long carry = 0;
    for (long long base = 0; base < nb; base += SCAN_B) {
        const long long i0 = base + threadIdx.x * SCAN_V;
        long long v[SCAN_V], s = 0;
#pragma unroll
        for (int k = 0; k < SCAN_V; ++k) {
            v[k] = i0 + k < nb ? bsum[i0 + k] : 0;
            s += v[k];
        }
        long long total;
        long long p = carry + block_scan(s, wsum, total);
#pragma unroll
        for (int k = 0; k < SCAN_V; ++k) {
            if (i0 + k < nb) bsum[i0 + k] = p;
            p += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) out[n] = carry;
}

__global__ __launch_bounds__(256) void k_scan_add(long long* out, long long n, const long long* bsum) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] += bsum[i / SCAN_B];
}

__global__ void k_pick(PickArgs a, const long long* off, long long* out) {
    if ((int)threadIdx.x < a.n) out[threadIdx.x] = off[a.at[threadIdx.x]];
}

__global__ __launch_bounds__(256) void k_run_starts(const long long* off, long long nrun, long long* out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < nrun) out[i] = off[i * LIST_WAVES];
}

// Screening values by rank, and per replica what bounds J and K: the largest q,
// the largest sum of q^2 over a row of AO pairs and the sum over all of them
// (in 2^20 fixed point, rounded up: an integer sum does not depend on the
// order). One wavefront per shell for the rows; max of the bit patterns.
__global__ __launch_bounds__(256) void k_geo_bounds(GeoArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.npair) a.rq[i] = a.qscr[a.cls_pairs[i]];
    const int x = i >> 6, lane = threadIdx.x & 63;
    if (x >= a.nshell) return;
    const int rep = a.shell_rep ? a.shell_rep[x] : 0;
    const int s0 = a.shell_rep ? a.rep_shell[rep] : 0, s1 = a.shell_rep ? a.rep_shell[rep + 1] : a.nshell;
    const int base = a.shell_rep ? a.shell_pair0[x] : 0;
    double m = 0.0, s = 0.0;
    for (int y = s0 + lane; y < s1; y += 64) {
        const int u = x - s0, v = y - s0;
        const double q = a.qscr[base + (u > v ? u * (u + 1) / 2 + v : v * (v + 1) / 2 + u)];
        const int l = a.shell_l[y];
        m = fmax(m, q);
        s += q * q * ((l + 1) * (l + 2) / 2);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        m = fmax(m, __shfl_xor(m, o, 64));
        s += __shfl_xor(s, o, 64);
    }
    if (lane == 0) {
        unsigned long long* g = a.gcell + 3 * rep;
        const int l = a.shell_l[x];
        atomicMax(g, (unsigned long long)__double_as_longlong(m));
        atomicMax(g + 1, (unsigned long long)__double_as_longlong(s));
        atomicAdd(g + 2, (unsigned long long)ceil(fmin(s * ((l + 1) * (l + 2) / 2), 1e12) * 1048576.0));
    }
}

__global__ void k_zero_cells(unsigned long long* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

}  // namespace

// a grid of 2^32 work-items or more (16.8 million pairs) wraps without an error: workgroups
// take every GRID_MAX-th pair from there on
constexpr int GRID_MAX = 1 << 21;

void launch_qlist_count(const QListArgs& a, hipStream_t st) {
    if (a.npair > 0) k_qlist_count<<<dim3(a.npair < GRID_MAX ? a.npair : GRID_MAX), dim3(64 * LIST_WAVES), 0, st>>>(a);
}

void launch_qlist_fill(const QListArgs& a, hipStream_t st) {
    if (a.npair > 0) k_qlist_fill<<<dim3(a.npair < GRID_MAX ? a.npair : GRID_MAX), dim3(64 * LIST_WAVES), 0, st>>>(a);
}

long long list_scan_blocks(long long n) { return (n + SCAN_B - 1) / SCAN_B; }

void launch_list_scan(const long long* in, long long* out, long long n, long long* bsum, hipStream_t st) {
    const long long nb = list_scan_blocks(n);
    if (n > 0) k_scan_block<<<dim3((unsigned)nb), dim3(SCAN_T), 0, st>>>(in, out, n, bsum);
    k_scan_sums<<<dim3(1), dim3(SCAN_T), 0, st>>>(bsum, nb, out, n);
    if (nb > 1) k_scan_add<<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st>>>(out, n, bsum);
}

void launch_pick(const PickArgs& a, const long long* off, long long* out, hipStream_t st) {
    k_pick<<<dim3(1), dim3(128), 0, st>>>(a, off, out);
}

void launch_run_starts(const long long* off, long long nrun, long long* out, hipStream_t st) {
    if (nrun > 0) k_run_starts<<<dim3((unsigned)((nrun + 255) / 256)), dim3(256), 0, st>>>(off, nrun, out);
}

void launch_geo_bounds(const GeoArgs& a, hipStream_t st) {
    k_zero_cells<<<dim3((3 * a.nrep + 255) / 256), dim3(256), 0, st>>>(a.gcell, 3 * a.nrep);
    const int n = a.npair > 64 * a.nshell ? a.npair : 64 * a.nshell;
    k_geo_bounds<<<dim3((n + 255) / 256), dim3(256), 0, st>>>(a);
}

}  // namespace aimdhf
