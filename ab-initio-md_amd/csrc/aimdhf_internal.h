// Argument blocks shared by the kernels and the host-side plan code.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace aimdhf {

struct PairArgs {
    int npair;                  // shell pairs (s1 >= s2), index s1 (s1+1)/2 + s2
    int nbpair;                 // contraction-block pairs
    const int* pair_a;          // shell with the higher l (ties: the higher index)
    const int* pair_b;
    const int* pair_cls;        // pair class (ss, ps, pp, ds, dp, dd) = 0..5
    const int* shell_l;
    const int* shell_atom;
    const int* shell_prim;      // nshell + 1
    const double* prim_exp;
    const double* prim_coef;
    const double* pos;          // (natm, 3) bohr
    const long long* rec_off;   // first record of each pair, in doubles
    const int* rec_size;        // doubles per record of each pair
    double* recs;
    int* npp;                   // kept primitive pairs per pair
    const int* cls_pairs;       // pairs grouped by class
    const int* cls_pair_off;    // 7 offsets into cls_pairs
    const int* ncls_pairs;      // 6 counts
    double* qshell;             // Schwarz bound of each shell pair
    double* qblock;             // of each block pair
    double* qscr;               // screening value of each shell pair (its block pair's bound)
    const int* bp_off;          // nbpair + 1
    const int* bp_list;         // shell pairs of each block pair
    const double* boys;         // 402 x 43 table
    const int* pair_lo;         // batched plans: first pair of each pair's replica (quartets pair
                                // within a replica only); null: every pair Q <= P
};

struct OneElArgs {
    int npair;                  // shell pairs s1 >= s2
    int nao;
    int natm;
    int ncls_host[6];           // pairs per class
    int cls_off_host[6];        // first pair of each class in cls_pairs
    const int* cls_pairs;
    const int* pair_a;          // l_A >= l_B orientation
    const int* pair_b;
    const int* shell_atom;
    const int* shell_l;
    const int* shell_prim;
    const int* shell_ao;
    const double* prim_exp;
    const double* prim_coef;
    const double* pos;
    const double* charges;
    const double* boys;
    int parts;                  // one-electron gradient: 1 overlap/kinetic, 2 nuclear attraction, 3 both
    // matrix layout: element (m, n) of a shell pair's matrices sits at
    // rep * ld^2 + m * ld + n (m, n: AO offsets within the replica, shell_ao);
    // the dipole components are mstride apart. A single molecule: rep 0, ld nao.
    int ld;
    long long mstride;
    const int* shell_rep;       // replica of each shell (null: 0)
    const int* rep_atom;        // nrep + 1: atoms of each replica (null: all atoms)
};

struct GradArgs {
    int nao;
    int natm;
    int nx;
    double kfac;
    double thr;
    const int* pair_a;
    const int* pair_b;
    const int* shell_ao;
    const int* shell_atom;
    const int* npp;
    const long long* rec_off;
    const double* recs;
    const double* boys;
    const double* pos;
    const double* qscr;
    const double* dc;           // (nao, nao), symmetric
    const double* dx;           // (nx, nao, nao), symmetric
    int npair;                  // shell pairs (s1 >= s2, index s1 (s1 + 1) / 2 + s2)
    const double* dmc;          // per shell pair: max |dc| over its block
    const double* dmx;          // (nx, npair): max |dx| over each block
    double fp32_switch;         // quartets with Q_P Q_Q max|Gamma| below: FP32 derivative integrals
    unsigned char* keep;        // per quartet of the launched class: 0 dropped, 1 FP64, 2 FP32
    int* sel64;                 // selected quartets (indices into the class list), FP64
    int* sel32;                 // and FP32
    int* nsel;                  // their counts (2 ints)
    int* bcnt;                  // pre-pass block counts (2 ints per 256 quartets)
    int* boff;                  // and their exclusive prefix sums
    long long* out;             // (natm, 3) fixed point, hi/lo interleaved
    // batched plans (see OneElArgs): dc of replica r at r ld^2, dx set x at (r nx + x) ld^2;
    // shell pair (s, t) of a replica at shell_pair0[s] + tri(s - shell_first[s], t - shell_first[t])
    int ld;
    const int* shell_rep;       // null: one molecule
    const int* shell_first;
    const int* shell_pair0;
};

void launch_batch_purify(int nmat, int ld, const double* F, const double* nocc, double* P, int steps, double tol,
                         double* err, hipStream_t st);
void launch_batch_diis_solve(int nrep, int m, const double* G, const double* r, double* c, hipStream_t st);

void launch_tc2_step(int n, const double* X, const double* X2, double* Xout, double nocc, double freeze,
                     hipStream_t st);
void launch_tc2_init(int n, const double* F, double* X0, hipStream_t st);
void launch_tc2_error(int n, const double* X, double* out, hipStream_t st);
void launch_zero_d(double* p, size_t n, hipStream_t st);

void launch_build_pairs(const PairArgs& g, hipStream_t st);
void launch_schwarz(const PairArgs& g, const int* ncls_host, hipStream_t st);
// gradient quartet lists: per class, NCOSTBIN bins of primitive-quartet cost (heaviest first)
constexpr int NCOSTBIN = 5;
void launch_count_quartets(const PairArgs& g, double thr, int* counts, long long* offs, long long* totals,
                           long long* base, hipStream_t st);
void launch_fill_quartets(const PairArgs& g, double thr, const long long* offs, const long long* base, int2* list,
                          hipStream_t st);
// ---------------------------------------------------------------- runtime-l path (l <= GEN_LMAX)
constexpr int GEN_LMAX = 4;
struct GenArgs {
    int nao, natm, nset;
    const int* shell_atom;
    const int* shell_l;
    const int* shell_prim;
    const int* shell_ao;
    const double* prim_exp;
    const double* prim_coef;
    const double* pos;
    const double* charges;
    const double* boys;
    const int* pair_i;          // shell pairs P: pair_i[P] >= pair_j[P]
    const int* pair_j;
    const int2* quartets;       // unique (P, Q), P >= Q
    long long nq;
    const double* dens;         // J/K: nset symmetric densities
    long long* fx;              // fixed-point accumulators (J/K planes, or 3 natm gradient words)
    const double* dc;           // derivative ERIs: Coulomb density, nx exchange densities, factor
    const double* dx;
    int nx;
    double kfac;
    double *S, *T, *V, *M;      // one-electron outputs
    const double* D;            // one-electron gradient densities
    const double* W;
    int parts;                  // one-electron gradient terms: 1 kinetic, 2 nuclear attraction, 4 overlap
    double* q;                  // Schwarz bounds per shell pair
};
void launch_gen_schwarz(const GenArgs& g, int npair, hipStream_t st);
void launch_gen_jk(const GenArgs& g, hipStream_t st);
void launch_gen_grad2(const GenArgs& g, hipStream_t st);
void launch_gen_oneel(const GenArgs& g, int npair, hipStream_t st);
void launch_gen_grad1(const GenArgs& g, int npair, hipStream_t st);

void launch_zero64(long long* p, size_t n, hipStream_t st);
void launch_symmetrize(const double* D, int nset, int n, double* out, hipStream_t st);
void launch_grad_one_class(int k, const GradArgs& a, const int2* list, long long nq, hipStream_t st);
void launch_grad_keep(int k, const GradArgs& a, const int2* list, long long nq, hipStream_t st);
void launch_pair_dmax(const GradArgs& a, const int* shell_l, double* dmc, double* dmx, hipStream_t st);
// on: the stream of each of the six pair classes
void launch_oneel(const OneElArgs& g, double* S, double* T, double* M, double* V, const hipStream_t* on);
// device address of the fixed-size scratch array of the allocation-free entry
// points on the current device (resolved once per device), and its size
void* noalloc_scratch(size_t* bytes);
void launch_grad_one(const OneElArgs& g, const double* D, const double* Wneg, long long* out, const hipStream_t* on);
void launch_negate(const double* W, size_t n, double* out, hipStream_t st);
void launch_fx_to_double(const long long* fx, int n, double* out, hipStream_t st);
double device_absmax(const double* x, size_t n, double* scratch, hipStream_t st);
void launch_jk_finalize(const long long* fx, int nset, int n, double* J, double* K, hipStream_t st);

}  // namespace aimdhf
