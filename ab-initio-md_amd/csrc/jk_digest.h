// Screened quartet list, integral store and its J/K digestion: argument blocks
// and launchers (quartet_list.hip, eri_store.hip, jk_digest.hip, jk_prep.hip).
//
// Shell pairs are ranked class by class (cls_pairs), within a class replica by
// replica, the most contracted pairs first, then along the diagonals of the
// shell-pair triangle, so that consecutive pairs of one rank range name
// different first and different second shells. The quartet list holds, class
// by class (heavier pair as bra) and per precision part, one run of kets per
// bra in rank order.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace aimdhf {

constexpr int DIG_NQC = 21;         // quartet classes
constexpr int JK_CELLS = 4;         // words of dcell per density
constexpr int LIST_WAVES = 4;       // wavefronts (list cells) per run

struct QListArgs {
    int npair, nrep, nparts;        // nparts 2: quartets with q_P q_Q >= sw first, then the rest
    double thr, sw;
    int cls_off[7];                 // rank range of each pair class
    long long runbase[DIG_NQC];     // first run of each class; run = runbase[k] + part * n_bra + bra
    const int* seg;                 // (6 nrep + 1) first rank of each class's replica segment
    const int* rank_rep;            // replica of each rank (null: one molecule)
    const double* rq;               // screening value by rank
    long long* cnt;                 // quartets per cell (LIST_WAVES cells per run)
    const long long* off;           // their exclusive scan
    int* lbra;                      // per quartet: rank of the bra and of the ket
    int* lket;
};

struct EriArgs {
    const double* recs;
    const long long* rec_off;       // by pair
    const int* npp;
    const int* cls_pairs;           // rank -> pair
    const double* boys;
    const int* lbra;                // the evaluated part's quartets
    const int* lket;
    double* out64;                  // its blocks: quartet t, value v = cd NAB + ab at
    float* out32;                   // (t / 64) 64 NAB NCD + 64 v + t % 64
};

// AO offsets of a ranked pair's shells (within the replica), 16 bits each; equal offsets are the same shell
constexpr int MAX_LD = (1 << 16) - 1;
__host__ __device__ inline unsigned oab_pack(int first, int second) { return (unsigned)first | (unsigned)second << 16; }
__host__ __device__ inline int oab_first(unsigned o) { return (int)(o & 0xffffu); }
__host__ __device__ inline int oab_second(unsigned o) { return (int)(o >> 16); }
__host__ __device__ inline bool oab_same(unsigned o) { return oab_first(o) == oab_second(o); }

// What of a digestion depends on the geometry; read from device memory, so a captured
// launch stays valid when the geometry moves (batched SCF iterations are replayed)
struct DigestGeo {
    long long t64, t32;             // list index of the first FP64 and FP32 block
    long long lo64, hi64, lo32, hi32;   // list ranges that are held (direct mode: a piece of the list)
    const long long* off;           // list offsets of the class's runs (LIST_WAVES apart)
    const int* lket;
    const double* s64;              // the class's blocks, FP64 part
    const float* s32;               // and FP32 part
};

struct DigestArgs {
    const DigestGeo* geo;           // by quartet class
    int ld, nset, ncopy;
    int lds_limit;                  // LDS bytes a workgroup may take
    int nparts, nchunk, unit;       // pieces a long run is cut into, each of at least unit quartets
    int cls_off[7];                 // rank range and component base (dket / jacc) of each pair class
    long long koff[7];
    const unsigned* oab;            // by rank
    const int* rank_rep;
    const double* dsym;             // (nrep, nset, ld, ld)
    const double* dket;             // (nset, npao): densities by pair component
    long long npao;
    unsigned long long* kacc;       // (ncopy, nrep, nset, ld, ld)
    unsigned long long* jacc;       // (ncopy, nset, npao)
    long long kstride;              // nrep nset ld^2
    const unsigned long long* dcell;   // (nrep, nset, 4): largest row sum of |D|, of D^2, largest |D| (bits),
                                       // sum of q |D| (2^24 fixed, rounded up)
    const unsigned long long* gcell;   // (nrep, 3): largest q, largest row sum of q^2 (bits), sum of q^2 (2^20 fixed)
    const int* rep_nao;             // null: ld
    int delta;                      // density-difference build: skip quartets below dthr
    double dthr;
    const double* rq;
};

struct PrepArgs {
    int ld, nset, nrep, ncopy, npair;
    int cls_off[7];
    long long koff[7];              // component base of each pair class
    long long npao, kstride;
    const unsigned* oab;
    const int* rank_rep;
    const int* rep_nao;
    const double* dens;
    double* dsym;
    double* dket;
    unsigned long long *kacc, *jacc, *dcell;
    const unsigned long long* gcell;
    double *J, *K;
    const double* rq;
};

struct GeoArgs {
    int nshell, npair;
    const int* shell_l;
    const int* shell_rep;           // null: one molecule
    const int* shell_first;
    const int* shell_pair0;
    const int* rep_shell;           // nrep + 1 (null: 0 .. nshell)
    const int* cls_pairs;
    const double* qscr;             // by pair
    double* rq;                     // by rank
    unsigned long long* gcell;
    int nrep;
};

void launch_geo_bounds(const GeoArgs& a, hipStream_t st);
void launch_qlist_count(const QListArgs& a, hipStream_t st);
void launch_qlist_fill(const QListArgs& a, hipStream_t st);
void launch_list_scan(const long long* in, long long* out, long long n, long long* bsum, hipStream_t st);
long long list_scan_blocks(long long n);
// out[i] = off[at[i]] of n (<= 128) list cells, at by value
struct PickArgs {
    int n;
    long long at[128];
};
void launch_pick(const PickArgs& a, const long long* off, long long* out, hipStream_t st);
// out[r] = first quartet of run r
void launch_run_starts(const long long* off, long long nrun, long long* out, hipStream_t st);

// n64 FP64 quartets from the list position of a, n32 FP32 ones after them; the first h64 / h32
// of each have contracted bras (ERI_HEAVY primitive pairs or more)
constexpr int ERI_HEAVY = 6;
void launch_eri(int k, const EriArgs& a, long long n64, long long h64, long long n32, long long h32, hipStream_t st);
long long store_block(int k);       // integrals per block of quartet class k
void launch_jk_prep(const PrepArgs& a, hipStream_t st);
void launch_jk_finish(const PrepArgs& a, hipStream_t st);
void launch_digest(int k, const DigestArgs& a, int threads, hipStream_t st);
// every class in one launch (matrices small enough for the rows of any bra in LDS)
void launch_digest_all(const DigestArgs& a, int threads, hipStream_t st);
bool digest_all_fits(int ld, int lds_limit);

#ifdef __HIPCC__
// Exponents of the fixed-point words that J and K sums are held in. Every sum
// of contributions to a K element is bounded by sum_ls q_ml |D_ls| q_ns <=
// max_m |q_m|^2 max_l sum_s |D_ls| (the spectral norm of |D| is at most its
// largest row sum), to a J element by q_max sum_ls q_ls |D_ls| (a fixed-point sum,
// so the smaller of it and its Cauchy-Schwarz bound q_max |q|_F |D|_F); scaled
// below 2^62 no sum overflows, and the resolution is at most 2^-61 of the bound
// (J and K of (H2O)32/6-31G* agree with two-word sums of 2^-80 resolution to 2e-13).
__device__ inline int jk_exponent(double bound) {
    if (!(bound > 0.0)) return 0;
    const int e = 61 - ilogb(bound);
    return e > 1000 ? 1000 : e < -1000 ? -1000 : e;
}
__device__ inline double jk_bound_k(const unsigned long long* g, const unsigned long long* d) {
    return __longlong_as_double((long long)g[1]) * __longlong_as_double((long long)d[0]);
}
__device__ inline double jk_bound_j(const unsigned long long* g, const unsigned long long* d, int n) {
    // |q|_F^2: the fixed-point sum, whose words neither saturate nor wrap while n times the
    // largest row is below their range, or that bound (larger integrals; and much smaller
    // ones, of which the sum only counts the rounded-up units)
    const double rows = n * __longlong_as_double((long long)g[1]), fq = (double)g[2] * (1.0 / 1048576.0);
    const double cs = sqrt((rows < 1e12 && fq < rows ? fq : rows) * (n * __longlong_as_double((long long)d[1])));
    const double sum = (double)d[3] * (1.0 / 16777216.0);
    // the fixed-point sum cannot have wrapped while the other bound is below its range
    return __longlong_as_double((long long)g[0]) * (cs < 1e9 && sum < cs ? sum : cs);
}
// 2^e; 0 where the bound is not finite (the sums then read NaN)
__device__ inline double jk_scale(double bound) { return isfinite(bound) ? ldexp(1.0, jk_exponent(bound)) : 0.0; }

// x (|x| < 2^62, scaled) rounded to the nearest integer, for 64-bit integer sums:
// adding 1.5 2^(52+k) to a double leaves its value in units of 2^k in the low
// mantissa bits, so the part above 2^20 and the rest cost two additions each
// and no conversion
__device__ __forceinline__ unsigned long long jk_fixed(double x) {
    constexpr double HI = 6755399441055744.0 * 1048576.0, LO = 6755399441055744.0;     // 1.5 2^72, 1.5 2^52
    const double h = x + HI;
    const double l = (x - (h - HI)) + LO;
    return ((unsigned long long)__double_as_longlong(h) << 20) + (unsigned long long)__double_as_longlong(l) -
           (((0x4478000000000000ull) << 20) + 0x4338000000000000ull);
}
#endif

}  // namespace aimdhf
