// J and K of one quartet class from the integral store (compiled once per class
// with -DAIMDHF_QCLASS=k): one workgroup per bra pair and piece of its run.

#include "jk_digest_run.h"

#ifndef AIMDHF_QCLASS
#error "compile with -DAIMDHF_QCLASS=<0..20>"
#endif

namespace aimdhf {

namespace {
constexpr int QC = AIMDHF_QCLASS;
// threads of a workgroup: where its rows leave room for few workgroups on a CU, 512;
// the classes that need more than 128 registers a lane stay at 256 (measured on 32
// waters, 6-31G*: class 6 674 -> 509 us, class 10 504 -> 350, class 18 194 -> 247)
constexpr int MAXT = QC == 4 || QC == 5 || QC == 8 || QC >= 16 ? 256 : 512;
// two densities in one workgroup (each integral read once) where the sums of both fit
// the registers, else a workgroup each: UHF (H2O)8/cc-pVDZ 0.59 ms per build, against
// 0.66 with both up to class 11 and 0.78 up to class 15
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
