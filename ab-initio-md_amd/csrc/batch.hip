// Batched plans: many independent small molecules (replicas) in one plan. Their
// screened quartets are evaluated and digested by the per-class kernels that
// single molecules use (one launch per class for all replicas); this file holds
// the density and DIIS solvers of all replicas at once.
//
// Matrices of a batch live in a padded layout: replica r's (nset x) ld x ld
// block starts at (r * nset + x) * ld^2; rows and columns past n_r stay zero.

#include "aimdhf_internal.h"

namespace aimdhf {

namespace {

// Trace-correcting purification of nmat symmetric ld x ld matrices (ld <= 64), one
// workgroup per matrix held in LDS for all steps: X0 = (e_max - F) / (e_max -
// e_min) with F's Gershgorin bounds, then X <- X^2 if tr X > nocc else 2X - X^2,
// up to `steps` times while |tr X - tr X^2| >= tol (more steps would amplify the
// rounding errors), and two final steps that square the remaining error. err[i]
// receives the idempotency error |tr X - tr X^2| before those two steps.
//
// X^2 on the matrix cores: X sits zero-padded to 64 x 64 in LDS (row stride 65
// doubles, so the 16 rows one operand load touches fall in distinct banks); the
// 16 x 16 tiles of its upper triangle, up to ceil(ld / 16) a side, go round the four
// wavefronts (10 tiles, 3 at most in one, at ld > 48) and are written on both sides,
// each 4 ceil(ld / 16) steps of v_mfma_f64_16x16x4f64 over k. Operand and result
// lanes (measured on gfx950): A(i, k) from lane i + 16 k, B(k, j) from lane j + 16 k,
// D(i, j) in register i / 4 of lane j + 16 (i % 4). Both traces are summed by every
// wavefront for itself in DPP steps, so a step has two barriers.
// Bound by the serial chain of steps, each the MFMA issue of one CU (1.3 us of 64 x 64)
// and the latencies of LDS and barriers: 24 matrices of 50 orbitals 268 -> 201 us (full
// tiles, six barriers and all 62 steps before), one of 19 orbitals 99 -> 56 us.
constexpr int PUR_THREADS = 256;
constexpr int PUR_MAXLD = 64;
constexpr int PUR_LS = PUR_MAXLD + 1;       // LDS row stride (doubles)
constexpr int PUR_TILES = 3;                // tiles of one wavefront

typedef double v4d __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return v + __hiloint2double(hi, lo);
}

__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the wavefront: neighbours, pairs, half rows and rows of 16 lanes, then the four rows
__device__ __forceinline__ double wave_sum(double v) {
    v = dpp_add<0xB1>(v);               // quad_perm 1 0 3 2
    v = dpp_add<0x4E>(v);               // quad_perm 2 3 0 1
    v = dpp_add<0x141>(v);              // row_half_mirror
    v = dpp_add<0x140>(v);              // row_mirror
    return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

__global__ __launch_bounds__(PUR_THREADS) void k_batch_purify(int ld, const double* __restrict__ F,
                                                              const double* __restrict__ nocc, double* __restrict__ P,
                                                              int steps, double tol, double* __restrict__ err) {
    __shared__ double X[PUR_MAXLD * PUR_LS];
    __shared__ double diag2[PUR_MAXLD];
    const int mat = blockIdx.x, t = threadIdx.x, n2 = ld * ld;
    const int w = t >> 6, lane = t & 63, li = lane & 15, lk = lane >> 4;
    const int nt = (ld + 15) / 16, ntile = nt * (nt + 1) / 2;
    const double* Fm = F + (size_t)mat * n2;
    // all loads of F in flight at once, then symmetrised in place
    double f[16];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int i = 16 * r + (t >> 4), j = 16 * c + (t & 15);
            f[4 * r + c] = i < ld && j < ld ? Fm[i * ld + j] : 0.0;
        }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) X[(16 * r + (t >> 4)) * PUR_LS + 16 * c + (t & 15)] = f[4 * r + c];
    if (t < PUR_MAXLD) diag2[t] = 0.0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            f[4 * r + c] = 0.5 * (f[4 * r + c] + X[(16 * c + (t & 15)) * PUR_LS + 16 * r + (t >> 4)]);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) X[(16 * r + (t >> 4)) * PUR_LS + 16 * c + (t & 15)] = f[4 * r + c];
    __syncthreads();
    // Gershgorin bounds, lane per row, each wavefront for itself (min / max do not depend on the order)
    double mn = 1e300, mx = -1e300;
    if (lane < ld) {
        double r = 0.0;
        const double d = X[lane * PUR_LS + lane];
#pragma unroll 8
        for (int j = 0; j < ld; ++j) r += j == lane ? 0.0 : fabs(X[lane * PUR_LS + j]);
        mn = d - r;
        mx = d + r;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        mn = fmin(mn, __shfl_xor(mn, o, 64));
        mx = fmax(mx, __shfl_xor(mx, o, 64));
    }
    const double inv = 1.0 / (mx - mn);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int i = 16 * r + (t >> 4), j = 16 * c + (t & 15);
            X[i * PUR_LS + j] = i < ld && j < ld ? ((i == j ? mx : 0.0) - f[4 * r + c]) * inv : 0.0;
        }
    __syncthreads();
    const double ne = nocc[mat];
    // the wavefront's tiles w, w + 4, w + 8 of the upper triangle (row by row)
    int ti[PUR_TILES], tj[PUR_TILES];
#pragma unroll
    for (int s = 0; s < PUR_TILES; ++s) {
        int q = w + 4 * s, i = 0;
        while (i < nt && q >= nt - i) q -= nt - i++;
        ti[s] = __builtin_amdgcn_readfirstlane(i);
        tj[s] = __builtin_amdgcn_readfirstlane(i + q);
    }
    const int mine = __builtin_amdgcn_readfirstlane(w < ntile ? (ntile - w + 3) / 4 : 0);
    double last = 0.0;
    for (int it = 0; it < steps + 2; ++it) {
        v4d acc[PUR_TILES];
#pragma unroll
        for (int s = 0; s < PUR_TILES; ++s) acc[s] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int k0 = 0; k0 < 16 * nt; k0 += 4)
#pragma unroll
            for (int s = 0; s < PUR_TILES; ++s)
                if (s < mine)
                    acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(X[(16 * ti[s] + li) * PUR_LS + k0 + lk],
                                                                  X[(k0 + lk) * PUR_LS + 16 * tj[s] + li], acc[s], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < PUR_TILES; ++s)
            if (s < mine && ti[s] == tj[s])
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (lk + 4 * v == li) diag2[16 * ti[s] + li] = acc[s][v];
        const double dx = X[lane * PUR_LS + lane];
        __syncthreads();                            // X read by all, diagonal of X^2 complete
        const double tr = wave_sum(dx), tr2 = wave_sum(diag2[lane]);
        if (it < steps && fabs(tr - tr2) < tol) it = steps;
        if (it == steps) last = fabs(tr - tr2);
        const bool square = tr > ne;
#pragma unroll
        for (int s = 0; s < PUR_TILES; ++s)
            if (s < mine)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * ti[s] + lk + 4 * v, j = 16 * tj[s] + li;
                    const double x = square ? acc[s][v] : 2.0 * X[i * PUR_LS + j] - acc[s][v];
                    X[i * PUR_LS + j] = x;
                    if (ti[s] != tj[s]) X[j * PUR_LS + i] = x;
                }
        __syncthreads();
    }
    double* Pm = P + (size_t)mat * n2;
    for (int e = t; e < n2; e += PUR_THREADS) {
        const int i = e / ld, j = e % ld;
        Pm[e] = 0.5 * (X[i * PUR_LS + j] + X[j * PUR_LS + i]);
    }
    if (t == 0) err[mat] = last;
}

// Pulay coefficients of nrep DIIS problems, thread per replica: the m x m system
// G c = r (G the Gram matrix of the error differences, r the right-hand side;
// rows of unused slots are identity rows with r = 0) by Gaussian elimination with
// partial pivoting; a singular pivot (below 1e-14 of the largest diagonal) leaves
// its unknown 0, as the reference's least-squares solve drops null directions.
__global__ void k_batch_diis_solve(int nrep, int m, const double* __restrict__ G, const double* __restrict__ r,
                                   double* __restrict__ c) {
    const int rep = blockIdx.x * blockDim.x + threadIdx.x;
    if (rep >= nrep) return;
    constexpr int MM = 12;
    double A[MM][MM + 1];
    const double* g = G + (size_t)rep * m * m;
    double scale = 0.0;
    for (int i = 0; i < m; ++i) {
        for (int j = 0; j < m; ++j) A[i][j] = g[i * m + j];
        A[i][m] = r[(size_t)rep * m + i];
        scale = fmax(scale, fabs(A[i][i]));
    }
    int piv_of[MM];
    for (int col = 0; col < m; ++col) {
        int best = col;
        for (int i = col + 1; i < m; ++i)
            if (fabs(A[i][col]) > fabs(A[best][col])) best = i;
        if (best != col)
            for (int j = 0; j <= m; ++j) {
                const double tmp = A[col][j];
                A[col][j] = A[best][j];
                A[best][j] = tmp;
            }
        piv_of[col] = fabs(A[col][col]) > 1e-14 * scale;
        if (!piv_of[col]) continue;
        for (int i = col + 1; i < m; ++i) {
            const double f = A[i][col] / A[col][col];
            for (int j = col; j <= m; ++j) A[i][j] -= f * A[col][j];
        }
    }
    double x[MM];
    for (int i = m - 1; i >= 0; --i) {
        if (!piv_of[i]) {
            x[i] = 0.0;
            continue;
        }
        double v = A[i][m];
        for (int j = i + 1; j < m; ++j) v -= A[i][j] * x[j];
        x[i] = v / A[i][i];
    }
    for (int i = 0; i < m; ++i) c[(size_t)rep * m + i] = x[i];
}

}  // namespace

void launch_batch_purify(int nmat, int ld, const double* F, const double* nocc, double* P, int steps, double tol,
                         double* err, hipStream_t st) {
    if (nmat > 0) k_batch_purify<<<dim3(nmat), dim3(PUR_THREADS), 0, st>>>(ld, F, nocc, P, steps, tol, err);
}

void launch_batch_diis_solve(int nrep, int m, const double* G, const double* r, double* c, hipStream_t st) {
    if (nrep > 0) k_batch_diis_solve<<<dim3((nrep + 63) / 64), dim3(64), 0, st>>>(nrep, m, G, r, c);
}

}  // namespace aimdhf
