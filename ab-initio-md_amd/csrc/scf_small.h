// SCF algebra of small matrices (scf_small.hip). Matrices are (nrep, nspin, ld, ld) or
// (nrep, ld, ld), ld <= 64.
#pragma once
#include <hip/hip_runtime.h>

namespace aimdhf {

struct SmallFock {
    int nspin, ld;
    double g;                   // 2 / nspin
    const double *H, *S, *X, *D, *J, *K;
    double* F;
    double *Fo, *E;             // orthogonal-basis Fock matrix and commutator of replica r at
    long long rep_stride, slot_stride;  // r rep_stride + slot slot_stride
    const long long* slot;      // device scalar (null: 0)
    double* energy;             // per replica
    double* err;                // largest |E| element
};

struct SmallDiis {
    int nspin, ld, m;           // ring of m <= 12 vectors
    const long long *slot, *count;      // device scalars: newest vector, vectors held
    const double *E, *Fo;       // (nrep, m, nspin, ld, ld)
    double* G;                  // (nrep, m, m), kept between calls
    const int* rep_nao;         // null: ld
    double pad;
    double* Fx;
};

struct SmallDensity {
    int nspin, ld;
    const double *X, *P;
    double* D;
    unsigned char* frozen;      // null: no convergence bookkeeping
    const double *energy, *err;
    double* e_prev;
    double conv_e, conv_g;
    long long *slot, *count;    // ring position to advance (null: none)
    int m;
};

void launch_small_fock(const SmallFock& a, int nrep, hipStream_t st);
void launch_small_diis(const SmallDiis& a, int nrep, hipStream_t st);
void launch_small_density(const SmallDensity& a, int nrep, hipStream_t st);
void launch_small_inv_sqrt(int nrep, int ld, const double* S, double* X, int iters, double tol, double* out,
                           hipStream_t st);

// sums: 2 doubles per 16 x 16 tile of the upper triangle
void launch_tc2_sums(int n, const double* X, double* sums, hipStream_t st);
void launch_tc2_fused(int n, const double* X, double* Xout, const double* sums, double* sums_out, double nocc,
                      double freeze, hipStream_t st);

}  // namespace aimdhf
