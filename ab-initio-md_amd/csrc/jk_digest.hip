// J and K of one quartet class from the integral store (compiled once per class
// with -DAIMDHF_QCLASS=k): one workgroup per bra pair and piece of its run.

#include "jk_digest_run.h"

#ifndef AIMDHF_QCLASS
#error "compile with -DAIMDHF_QCLASS=<0..20>"
#endif

namespace aimdhf {

namespace {
constexpr int QC = AIMDHF_QCLASS;
// threads of a workgroup: where its rows leave room for few workgroups on a CU, 512; the
// classes that need more than 128 registers a lane spill there and stay at 256. Alone,
// 256 : 512 threads, 6-31G*: (H2O)32 class 6 393 : 330 us, class 10 300 : 226, class 18
// 159 : 258; (H2O)16 class 10 49 : 42, class 15 54 : 43, class 16 75 : 120; the whole build
// of (H2O)32 4.31 ms with 256 in every class, 4.52 with 512, 4.19 so
constexpr int MAXT = QC == 4 || QC == 5 || QC == 8 || QC >= 16 ? 256 : 512;
// two densities in one workgroup (each integral read once) where the sums of both fit
// the registers, else a workgroup each: per build with each alone, so, and both up to
// class 9: (H2O)32 6-31G* 8.22, 8.06, 8.19 ms; (H2O)16 1.22, 1.17, 1.21; cc-pVDZ (H2O)12
// 1.48, 1.40, 1.40; (H2O)8 0.52, 0.51, 0.55 (up to class 15 0.78)
constexpr bool BOTH = QC < 5;

template <int QC_, int NSET, bool LDSROWS>
__global__ __launch_bounds__(MAXT) void k_digest(DigestArgs a, int bra0) {
    digest_run<QC_, NSET, LDSROWS>(a, bra0 + blockIdx.x, blockIdx.y / a.nchunk, blockIdx.y % a.nchunk, blockIdx.z * NSET,
                                   (int)((blockIdx.y * gridDim.x + blockIdx.x) % a.ncopy));
}

template <int NSET>
void launch(const DigestArgs& a, int nb, int threads, hipStream_t st) {
    using S = Dig<QC>;
    const size_t head = sizeof(double) * S::head(NSET);
    const size_t rows = head + sizeof(double) * S::colw(NSET) * (size_t)a.ld;
    const bool fit = rows <= (size_t)a.lds_limit;
    if (fit && threads == 256 && rows > 40 * 1024) threads = MAXT;
    if (fit && rows > 60 * 1024)
        (void)hipFuncSetAttribute((const void*)k_digest<QC, NSET, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)rows);
    // bras in slices: a grid of 2^32 work-items or more wraps without an error
    constexpr int SLICE = 1 << 21;
    for (int b0 = 0; b0 < nb; b0 += SLICE) {
        const dim3 grid(nb - b0 < SLICE ? nb - b0 : SLICE, a.nparts * a.nchunk, a.nset / NSET);
        if (fit) k_digest<QC, NSET, true><<<grid, dim3(threads), rows, st>>>(a, b0);
        else k_digest<QC, NSET, false><<<grid, dim3(threads), head, st>>>(a, b0);
    }
}

}  // namespace

#define CAT2(a, b) a##b
#define CAT(a, b) CAT2(a, b)

void CAT(launch_digest_, AIMDHF_QCLASS)(const DigestArgs& a, int threads, hipStream_t st) {
    const int nb = a.cls_off[Dig<QC>::CB + 1] - a.cls_off[Dig<QC>::CB];
    const int nk = a.cls_off[Dig<QC>::CK + 1] - a.cls_off[Dig<QC>::CK];
    if (nb <= 0 || nk <= 0) return;
    if (a.nset == 1 || !BOTH) launch<1>(a, nb, threads, st);
    else launch<2>(a, nb, threads, st);
}

}  // namespace aimdhf
