// SCF algebra. Small matrices (ld <= 64): one workgroup per matrix or replica with
// everything in LDS, products on the FP64 matrix cores: Fock matrices with energies
// and commutators, Pulay extrapolation, densities from projectors, S^(-1/2). For
// batches of replicas and for single small molecules, where each product or
// elementwise pass on its own is a launch of 3-8 us for well under 1 us of work
// (a 12-replica iteration: about 100 launches around the J/K build, one batched Gram
// product alone 275 us; now 88 us Fock matrices, 35 us Pulay step, 23 us densities. A
// step of 12 replicas 14.7 -> 9.9 ms, of 128 29.8 -> 23.6 ms, of one water molecule
// 8.7 -> 4.9 ms, with the purification.) Bound by the serial chain of products and
// passes in one CU.
//
// A matrix sits zero-padded to 64 x 64 in LDS, row stride 65 doubles (the 16 rows of
// one operand load fall in distinct banks); wavefront w of four forms the 16 x 64 row
// block w of a product as 16 x 16 tiles of v_mfma_f64_16x16x4f64. Operand and result
// lanes: A(i, k) from lane i + 16 k, B(k, j) from lane j + 16 k, D(i, j) in register
// i / 4 of lane j + 16 (i % 4). Tiles past ceil(ld / 16) are skipped.

#include "scf_small.h"

namespace aimdhf {

namespace {

constexpr int LD = 64, LS = LD + 1, MAT = LD * LS, NT = 256, NTD = 1024;
typedef double v4d __attribute__((ext_vector_type(4)));

struct Tiles {
    v4d t[4];
};

// acc += row block w of A B (TA: of A^T B, TB: of A B^T); k and columns up to nt tiles
template <bool TA = false, bool TB = false>
__device__ __forceinline__ void mm(const double* A, const double* B, int nt, Tiles& acc) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    if (w >= nt) return;
#pragma unroll 4
    for (int k0 = 0; k0 < 16 * nt; k0 += 4) {
        const double a = TA ? A[(k0 + lk) * LS + 16 * w + li] : A[(16 * w + li) * LS + k0 + lk];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j < nt) {
                const double b = TB ? B[(16 * j + li) * LS + k0 + lk] : B[(k0 + lk) * LS + 16 * j + li];
                acc.t[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc.t[j], 0, 0, 0);
            }
    }
}

// f(row, column, value) for the lane's results of the first nt tiles
template <class F>
__device__ __forceinline__ void each(const Tiles& acc, int nt, F&& f) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    if (w >= nt) return;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (j < nt)
#pragma unroll
            for (int v = 0; v < 4; ++v) f(16 * w + lk + 4 * v, 16 * j + li, acc.t[j][v]);
}

__device__ __forceinline__ void zero(Tiles& acc) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc.t[j] = v4d{0.0, 0.0, 0.0, 0.0};
}

// C = A B (or A^T B); the barriers around it let C be A or B
template <bool TA = false>
__device__ __forceinline__ void product(const double* A, const double* B, double* C, int nt) {
    Tiles acc;
    zero(acc);
    mm<TA>(A, B, nt, acc);
    __syncthreads();
    each(acc, nt, [&](int i, int j, double x) { C[i * LS + j] = x; });
    __syncthreads();
}

// f(r, row, column) for the thread's 16 elements of the padded matrix, in the order of r
template <class F>
__device__ __forceinline__ void own(F&& f) {
#pragma unroll
    for (int r = 0; r < 16; ++r) f(r, 16 * (r >> 2) + ((int)threadIdx.x >> 4), 16 * (r & 3) + ((int)threadIdx.x & 15));
}

// all loads in flight before the first is stored (each stored before the next load:
// 113 against 88 us for k_small_fock of 12 replicas, ld 50)
__device__ __forceinline__ void load(const double* __restrict__ src, int ld, double* dst) {
    double v[16];
    own([&](int r, int i, int j) { v[r] = i < ld && j < ld ? src[i * ld + j] : 0.0; });
    own([&](int r, int i, int j) { dst[i * LS + j] = v[r]; });
}

__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// NaN counts as largest
__device__ __forceinline__ double max_nan(double a, double b) { return a != a || a > b ? a : b; }
__device__ __forceinline__ double block_max(double v, double* red) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = max_nan(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return max_nan(max_nan(red[0], red[1]), max_nan(red[2], red[3]));
}

// One workgroup per replica, spin after spin: F_s = sym(H + g sum J - K_s), the
// electronic energy, Fo = X^T F X and the commutator e = X^T (F D S - S D F) X
__global__ __launch_bounds__(NT) void k_small_fock(SmallFock a) {
    extern __shared__ double lds[];
    __shared__ double red[4];
    double *A = lds, *B = lds + MAT, *C = lds + 2 * MAT;
    const int rep = blockIdx.x, ld = a.ld, n2 = ld * ld, nt = (ld + 15) / 16;
    const double* H = a.H + (size_t)rep * n2;
    const double* S = a.S + (size_t)rep * n2;
    const double* X = a.X + (size_t)rep * n2;
    const long long slot = a.slot ? *a.slot : 0;
    double en = 0.0, em = 0.0;
    for (int s = 0; s < a.nspin; ++s) {
        const size_t m = ((size_t)rep * a.nspin + s) * n2;
        const double* J0 = a.J + (size_t)rep * a.nspin * n2;
        const double* J1 = J0 + (size_t)(a.nspin - 1) * n2;
        const double* K = a.K + m;
        const double* D = a.D + m;
        double* F = a.F + m;
        const double gj = a.nspin == 2 ? a.g : 0.5 * a.g;       // one density: J0 and J1 are the same
        double h[16], d[16], f[16];
        own([&](int r, int i, int j) {
            const int u = i * ld + j;
            const bool in = i < ld && j < ld;
            h[r] = in ? H[u] : 0.0;
            d[r] = in ? D[u] : 0.0;
            f[r] = in ? h[r] + gj * (J0[u] + J1[u]) - K[u] : 0.0;
        });
        own([&](int r, int i, int j) {
            A[i * LS + j] = f[r];
            B[i * LS + j] = d[r];
        });
        __syncthreads();
        own([&](int r, int i, int j) {
            f[r] = 0.5 * (f[r] + A[j * LS + i]);
            en += d[r] * (h[r] + f[r]);
            if (i < ld && j < ld) F[i * ld + j] = f[r];
        });
        __syncthreads();
        own([&](int r, int i, int j) { A[i * LS + j] = f[r]; });
        __syncthreads();
        product(A, B, B, nt);                                   // F D
        load(S, ld, C);
        __syncthreads();
        product(B, C, B, nt);                                   // F D S
        load(X, ld, C);
        own([&](int r, int i, int j) { f[r] = B[i * LS + j] - B[j * LS + i]; });
        __syncthreads();
        own([&](int r, int i, int j) { B[i * LS + j] = f[r]; });
        __syncthreads();
        product(B, C, B, nt);
        double* eo = a.E + rep * a.rep_stride + slot * a.slot_stride + (size_t)s * n2;
        double* fo = a.Fo + rep * a.rep_stride + slot * a.slot_stride + (size_t)s * n2;
        Tiles acc;
        zero(acc);
        mm<true>(C, B, nt, acc);
        each(acc, nt, [&](int i, int j, double x) {
            if (i < ld && j < ld) {
                eo[i * ld + j] = x;
                em = max_nan(fabs(x), em);
            }
        });
        product(A, C, A, nt);                                   // F X
        zero(acc);
        mm<true>(C, A, nt, acc);
        each(acc, nt, [&](int i, int j, double x) {
            if (i < ld && j < ld) fo[i * ld + j] = x;
        });
        __syncthreads();
    }
    const double e = block_sum(en, red), m = block_max(em, red);
    if (threadIdx.x == 0) {
        a.energy[rep] = 0.5 * a.g * e;
        a.err[rep] = m;
    }
}

// One workgroup per replica: the new vector's row of the ring's Gram matrix, the
// Pulay system of the differences to it (Gauss-Jordan with partial pivoting, one thread
// per element; a pivot below 1e-14 of the largest diagonal leaves its unknown 0), and
// the extrapolated Fock matrices, padded orbitals lifted by pad
// Bound by the latency of reading the ring twice from few workgroups: 16 wavefronts
// (12 replicas, ld 50: 35 us; four wavefronts 69 us).
__global__ __launch_bounds__(NTD) void k_small_diis(SmallDiis a) {
    constexpr int MM = 12;
    __shared__ double part[NTD / 64][MM], row[MM], A[MM][MM + 1], c[MM];
    const int rep = blockIdx.x, M = a.m, n = a.nspin * a.ld * a.ld, t = threadIdx.x;
    const int slot = (int)*a.slot, count = (int)*a.count, held = count > slot ? count : slot + 1;
    const double* E = a.E + (size_t)rep * M * n;
    const double* Fr = a.Fo + (size_t)rep * M * n;
    double* G = a.G + (size_t)rep * M * M;
    const double* en = E + (size_t)slot * n;
    double s[MM];
#pragma unroll
    for (int j = 0; j < MM; ++j) s[j] = 0.0;
    for (int e = t; e < n; e += NTD) {
        const double x = en[e];
#pragma unroll
        for (int j = 0; j < MM; ++j)
            if (j < held) s[j] += x * E[(size_t)j * n + e];
    }
#pragma unroll
    for (int j = 0; j < MM; ++j) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) s[j] += __shfl_xor(s[j], o, 64);
        if ((t & 63) == 0) part[t >> 6][j] = s[j];
    }
    __syncthreads();
    if (t < MM) {
        double v = 0.0;
        for (int k = 0; k < NTD / 64; ++k) v += part[k][t];
        row[t] = v;
        if (t < held) G[slot * M + t] = G[t * M + slot] = row[t];
    }
    __syncthreads();
    // held vectors other than the newest are the unknowns; the others' rows are the identity
    const int i = t / (MM + 1), j = t - i * (MM + 1);
    const bool mine = i < MM;
    if (mine) {
        const bool vi = i < held && i != slot, vj = j < held && j != slot;
        const double gaa = row[slot];
        A[i][j] = j == MM ? (vi ? gaa - row[i] : 0.0)
                  : vi && vj ? G[i * M + j] - row[i] - row[j] + gaa : i == j ? 1.0 : 0.0;
    }
    __syncthreads();
    double scale = 0.0;
    for (int k = 0; k < MM; ++k) scale = fmax(scale, fabs(A[k][k]));
    unsigned ok = 0;
    for (int col = 0; col < MM; ++col) {
        int best = col;
        for (int k = col + 1; k < MM; ++k)
            if (fabs(A[k][col]) > fabs(A[best][col])) best = k;
        const double piv = A[best][col];
        const bool good = fabs(piv) > 1e-14 * scale;
        double v = 0.0;
        if (mine) {
            const int src = i == col ? best : i == best ? col : i;  // rows col and best swap
            v = A[src][j];
            if (good && i != col) v -= A[src][col] / piv * A[best][j];
        }
        ok |= (unsigned)good << col;
        __syncthreads();
        if (mine) A[i][j] = v;
        __syncthreads();
    }
    if (t == 0) {
        double x[MM], sum = 0.0, big = 0.0;
        bool fin = true;
#pragma unroll
        for (int k = 0; k < MM; ++k) {
            x[k] = k < held && k != slot && (ok >> k & 1) ? A[k][MM] / A[k][k] : 0.0;
            sum += x[k];
        }
#pragma unroll
        for (int k = 0; k < MM; ++k) {
            if (k == slot) x[k] = 1.0 - sum;
            fin = fin && isfinite(x[k]);
            big = fmax(big, fabs(x[k]));
        }
#pragma unroll
        for (int k = 0; k < MM; ++k) c[k] = fin && big <= 1e4 ? x[k] : k == slot ? 1.0 : 0.0;
    }
    __syncthreads();
    const int nao = a.rep_nao ? a.rep_nao[rep] : a.ld;
    for (int e = t; e < n; e += NTD) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < MM; ++k)
            if (k < held) v += c[k] * Fr[(size_t)k * n + e];
        const int r = e % (a.ld * a.ld), d = r / a.ld;
        if (r - d * a.ld == d && d >= nao) v += a.pad;
        a.Fx[(size_t)rep * n + e] = v;
    }
}

// One workgroup per replica: convergence (|E - E_prev| and the commutator), then
// D = X P X^T of each spin unless the replica is (now) frozen
__global__ __launch_bounds__(NT) void k_small_density(SmallDensity a) {
    extern __shared__ double lds[];
    double *A = lds, *B = lds + MAT;
    __shared__ int frozen;
    const int rep = blockIdx.x, ld = a.ld, n2 = ld * ld, nt = (ld + 15) / 16;
    if (threadIdx.x == 0) {
        int f = 0;
        if (a.frozen) {
            const double e = a.energy[rep];
            f = a.frozen[rep] || (fabs(e - a.e_prev[rep]) < a.conv_e && a.err[rep] < a.conv_g);
            a.frozen[rep] = (unsigned char)f;
            a.e_prev[rep] = e;
        }
        frozen = f;
    }
    __syncthreads();
    if (frozen) return;
    load(a.X + (size_t)rep * n2, ld, A);
    for (int s = 0; s < a.nspin; ++s) {
        const size_t m = ((size_t)rep * a.nspin + s) * n2;
        load(a.P + m, ld, B);
        __syncthreads();
        product(A, B, B, nt);                                   // X P
        Tiles acc;
        zero(acc);
        mm<false, true>(B, A, nt, acc);
        each(acc, nt, [&](int i, int j, double x) {
            if (i < ld && j < ld) a.D[m + i * ld + j] = x;
        });
        __syncthreads();
    }
}

__global__ void k_small_advance(long long* slot, long long* count, int m) {
    *slot = (*slot + 1) % m;
    *count = *count + 1 < m ? *count + 1 : m;
}

// S^(-1/2) by the coupled Newton-Schulz iteration Y0 = S / c, Z0 = 1, T = (3 - Z Y) / 2,
// Y <- Y T, Z <- T Z with c the largest row sum of |S|, until |Z Y - 1| < tol (or iters);
// out[rep] = residual max|X S X - 1|, 1 / largest row sum of |X X| (a lower bound of the
// smallest eigenvalue)
__global__ __launch_bounds__(NT) void k_small_inv_sqrt(int ld, const double* __restrict__ S, double* __restrict__ X,
                                                       int iters, double tol, double* __restrict__ out) {
    extern __shared__ double lds[];
    __shared__ double red[4];
    double *Y = lds, *Z = lds + MAT, *T = lds + 2 * MAT;
    const int rep = blockIdx.x, n2 = ld * ld, nt = (ld + 15) / 16, np = 16 * nt;
    const double* Sm = S + (size_t)rep * n2;
    load(Sm, ld, Y);
    __syncthreads();
    double r = 0.0;
    if ((int)threadIdx.x < ld)
        for (int j = 0; j < ld; ++j) r += fabs(Y[threadIdx.x * LS + j]);
    const double c = block_max(r, red), ic = 1.0 / c;
    for (int e = threadIdx.x; e < np * np; e += NT) {
        const int i = e / np, j = e - i * np;
        const bool pad = i >= ld || j >= ld;
        Y[i * LS + j] = pad ? (i == j ? 1.0 : 0.0) : Y[i * LS + j] * ic;
        Z[i * LS + j] = i == j ? 1.0 : 0.0;
    }
    __syncthreads();
    for (int it = 0; it < iters; ++it) {
        Tiles a, b;
        zero(a);
        mm(Z, Y, nt, a);
        double d = 0.0;
        each(a, nt, [&](int i, int j, double x) {
            const double one = i == j ? 1.0 : 0.0;
            d = max_nan(fabs(x - one), d);
            T[i * LS + j] = 0.5 * (3.0 * one - x);
        });
        d = block_max(d, red);                          // ends with every T written
        __syncthreads();
        zero(a);
        zero(b);
        mm(Y, T, nt, a);
        mm(T, Z, nt, b);
        __syncthreads();
        each(a, nt, [&](int i, int j, double x) { Y[i * LS + j] = x; });
        each(b, nt, [&](int i, int j, double x) { Z[i * LS + j] = x; });
        __syncthreads();
        if (d < tol) break;
    }
    const double f = 1.0 / sqrt(c);
    for (int e = threadIdx.x; e < np * np; e += NT) {
        const int i = e / np, j = e - i * np;
        const double x = i < ld && j < ld ? 0.5 * (Z[i * LS + j] + Z[j * LS + i]) * f : 0.0;
        T[i * LS + j] = x;
        if (i < ld && j < ld) X[(size_t)rep * n2 + i * ld + j] = x;
    }
    __syncthreads();
    load(Sm, ld, Y);
    __syncthreads();
    product(T, Y, Y, nt);                                       // X S
    Tiles a;
    zero(a);
    mm(Y, T, nt, a);
    double d = 0.0;
    each(a, nt, [&](int i, int j, double x) {
        if (i < ld && j < ld) d = max_nan(fabs(x - (i == j ? 1.0 : 0.0)), d);
    });
    d = block_max(d, red);
    product(T, T, Z, nt);                                       // X X = S^-1
    r = 0.0;
    if ((int)threadIdx.x < ld)
        for (int j = 0; j < ld; ++j) r += fabs(Z[threadIdx.x * LS + j]);
    r = block_max(r, red);
    if (threadIdx.x == 0) {
        out[2 * rep] = d;
        out[2 * rep + 1] = 1.0 / r;
    }
}

// ------------------------------------------------- purification step above 64 orbitals
// One purification step of a symmetric n x n X in one launch: Xout = X^2 if tr X > nocc
// else 2 X - X^2, or X where |tr X - sum X_ij^2| < freeze. One workgroup per 16 x 16 tile
// of the upper triangle, written on both sides; its wavefronts take every fourth
// k step of four rows (both operands are rows of X: X is symmetric, so A(i, k) is read as
// X(k, i), 128 consecutive bytes), four partial tiles meet in LDS. tr X and sum X_ij^2 come
// from the tile sums that the step before wrote (sums[0..nt): diagonal, sums[nt..2 nt):
// squares, off-diagonal tiles twice), so no step needs a pass over X of its own.
// Bound by launch and load latency up to a few hundred orbitals (190 workgroups at 304).
// Against a library product and an update kernel: 304 orbitals 12.2 -> 7.3 us a step, 76
// orbitals 10.6 -> 4.8 us, 608 orbitals 29.5 -> 15.3 us.
constexpr int TW = 4;                   // wavefronts of a workgroup

__device__ __forceinline__ void tile_sums(double x, bool diag_elem, bool diag_tile, double* sums, double (*red)[TW]) {
    double t = diag_elem ? x : 0.0, q = x * x * (diag_tile ? 1.0 : 2.0);
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        t += __shfl_xor(t, o, 64);
        q += __shfl_xor(q, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = t;
        red[1][threadIdx.x >> 6] = q;
    }
    __syncthreads();
    if (threadIdx.x < 2)
        sums[threadIdx.x * gridDim.x + blockIdx.x] =
            (red[threadIdx.x][0] + red[threadIdx.x][1]) + (red[threadIdx.x][2] + red[threadIdx.x][3]);
}

// upper-triangle tile of a workgroup: row by row
__device__ __forceinline__ void upper_tile(int q, int nt, int& ti, int& tj) {
    int i = (int)((2 * nt + 1 - sqrt((double)(2 * nt + 1) * (2 * nt + 1) - 8.0 * q)) * 0.5);
    while (i > 0 && i * nt - i * (i - 1) / 2 > q) --i;
    while ((i + 1) * nt - (i + 1) * i / 2 <= q) ++i;
    ti = i;
    tj = i + q - (i * nt - i * (i - 1) / 2);
}

__global__ __launch_bounds__(64 * TW) void k_tc2_sums(int n, int nt, const double* __restrict__ X,
                                                      double* __restrict__ sums) {
    __shared__ double red[2][TW];
    int ti, tj;
    upper_tile(blockIdx.x, nt, ti, tj);
    const int i = 16 * ti + ((int)threadIdx.x >> 4), j = 16 * tj + ((int)threadIdx.x & 15);
    tile_sums(i < n && j < n ? X[(size_t)i * n + j] : 0.0, i == j, ti == tj, sums, red);
}

__global__ __launch_bounds__(64 * TW) void k_tc2_fused(int n, int nt, const double* __restrict__ X,
                                                       double* __restrict__ Xout, const double* __restrict__ sums,
                                                       double* __restrict__ sums_out, double nocc, double freeze) {
    __shared__ double part[TW][256];
    __shared__ double red[2][TW];
    int ti, tj;
    upper_tile(blockIdx.x, nt, ti, tj);
    const int t = threadIdx.x, w = t >> 6, lane = t & 63, li = lane & 15, lk = lane >> 4;
    // traces of X from its tile sums
    double tr = 0.0, sq = 0.0;
    for (int b = t; b < (int)gridDim.x; b += 64 * TW) {
        tr += sums[b];
        sq += sums[gridDim.x + b];
    }
    const int ca = 16 * ti + li, cb = 16 * tj + li;
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    constexpr int U = 8;
    for (int k0 = 4 * w; k0 < n; k0 += 4 * TW * U) {
        double a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + 4 * TW * u + lk;
            a[u] = k < n && ca < n ? X[(size_t)k * n + ca] : 0.0;
            b[u] = k < n && cb < n ? X[(size_t)k * n + cb] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc, 0, 0, 0);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        tr += __shfl_xor(tr, o, 64);
        sq += __shfl_xor(sq, o, 64);
    }
    if (lane == 0) {
        red[0][w] = tr;
        red[1][w] = sq;
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) part[w][(lk + 4 * v) * 16 + li] = acc[v];
    __syncthreads();
    tr = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
    sq = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    const bool hold = freeze > 0.0 && fabs(tr - sq) < freeze, square = tr > nocc;
    const int r = t >> 4, c = t & 15, i = 16 * ti + r, j = 16 * tj + c;
    const double x2 = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    double x = 0.0;
    if (i < n && j < n) {
        const double x0 = X[(size_t)i * n + j];
        x = hold ? x0 : square ? x2 : 2.0 * x0 - x2;
        Xout[(size_t)i * n + j] = x;
    }
    __syncthreads();
    part[0][t] = x;
    tile_sums(x, i == j, ti == tj, sums_out, red);      // its barrier also completes part
    if (ti != tj) {
        const int mi = 16 * tj + r, mj = 16 * ti + c;   // the mirrored tile, row by row
        if (mi < n && mj < n) Xout[(size_t)mi * n + mj] = part[0][c * 16 + r];
    }
}

template <class K>
void big_lds(K k, size_t bytes) {
    (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

}  // namespace

void launch_small_fock(const SmallFock& a, int nrep, hipStream_t st) {
    const size_t lds = sizeof(double) * 3 * MAT;
    big_lds(k_small_fock, lds);
    if (nrep > 0) k_small_fock<<<dim3(nrep), dim3(NT), lds, st>>>(a);
}

void launch_small_diis(const SmallDiis& a, int nrep, hipStream_t st) {
    if (nrep > 0) k_small_diis<<<dim3(nrep), dim3(NTD), 0, st>>>(a);
}

void launch_small_density(const SmallDensity& a, int nrep, hipStream_t st) {
    const size_t lds = sizeof(double) * 2 * MAT;
    big_lds(k_small_density, lds);
    if (nrep > 0) k_small_density<<<dim3(nrep), dim3(NT), lds, st>>>(a);
    if (a.slot) k_small_advance<<<dim3(1), dim3(1), 0, st>>>(a.slot, a.count, a.m);
}

void launch_small_inv_sqrt(int nrep, int ld, const double* S, double* X, int iters, double tol, double* out,
                           hipStream_t st) {
    const size_t lds = sizeof(double) * 3 * MAT;
    big_lds(k_small_inv_sqrt, lds);
    if (nrep > 0) k_small_inv_sqrt<<<dim3(nrep), dim3(NT), lds, st>>>(ld, S, X, iters, tol, out);
}

void launch_tc2_sums(int n, const double* X, double* sums, hipStream_t st) {
    const int nt = (n + 15) / 16;
    if (n > 0) k_tc2_sums<<<dim3(nt * (nt + 1) / 2), dim3(64 * TW), 0, st>>>(n, nt, X, sums);
}

void launch_tc2_fused(int n, const double* X, double* Xout, const double* sums, double* sums_out, double nocc,
                      double freeze, hipStream_t st) {
    const int nt = (n + 15) / 16;
    if (n > 0)
        k_tc2_fused<<<dim3(nt * (nt + 1) / 2), dim3(64 * TW), 0, st>>>(n, nt, X, Xout, sums, sums_out, nocc, freeze);
}

}  // namespace aimdhf
