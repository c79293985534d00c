// Every quartet class of a build in one launch, for small matrices: the runs are
// short there (tens of kets), and 21 launches cost more than the work in them. One
// workgroup per bra pair, ket class, precision part and density; the classes in
// falling order of work.

#include "jk_digest_run.h"

namespace aimdhf {

namespace {
constexpr int LIGHT = 12, WLIGHT = 3;

template <int K, int LAST>
__device__ __forceinline__ void dispatch(const DigestArgs& a, int x, int part, int set) {
    const int nb = a.cls_off[Dig<K>::CB + 1] - a.cls_off[Dig<K>::CB];
    if (x < nb) {
        digest_run<K, 1, true>(a, x, part, 0, set, (int)(blockIdx.x % a.ncopy));
        return;
    }
    if constexpr (K > LAST) dispatch<K - 1, LAST>(a, x - nb, part, set);
}

__global__ __launch_bounds__(256) void k_digest_all(DigestArgs a) {
    dispatch<20, 0>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// many runs: the light classes apart, at three wavefronts a SIMD instead of one
__global__ __launch_bounds__(256) void k_digest_heavy(DigestArgs a) {
    dispatch<20, LIGHT>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WLIGHT))) void k_digest_light(DigestArgs a) {
    dispatch<LIGHT - 1, 0>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

constexpr int HEAD = Dig<20>::head(1), COLW = Dig<20>::colw(1);     // the widest class

}  // namespace

bool digest_all_fits(int ld, int lds_limit) {
    return sizeof(double) * (HEAD + (size_t)COLW * ld) <= (size_t)(lds_limit < 61440 ? lds_limit : 61440);
}

void launch_digest_all(const DigestArgs& a, int threads, hipStream_t st) {
    int nl = 0, nh = 0;
    for (int k = 0; k < DIG_NQC; ++k) {
        const int cb = pc_hi(k);
        (k < LIGHT ? nl : nh) += a.cls_off[cb + 1] - a.cls_off[cb];
    }
    const size_t lds = sizeof(double) * (HEAD + (size_t)COLW * a.ld);
    // two launches from the runs on that keep all CUs busy at three wavefronts a SIMD: one
    // water 30 (one launch) : 39 us (two), 76 AOs 62 : 57, 114 AOs 131 : 94, 128 replicas
    // 690 : 450 us
    if (nl + nh > 1200) {
        if (nh > 0) k_digest_heavy<<<dim3(nh, a.nparts, a.nset), dim3(threads), lds, st>>>(a);
        if (nl > 0) k_digest_light<<<dim3(nl, a.nparts, a.nset), dim3(threads), lds, st>>>(a);
    } else if (nl + nh > 0)         // either may be zero: a basis of d shells alone has no light runs
        k_digest_all<<<dim3(nl + nh, a.nparts, a.nset), dim3(threads), lds, st>>>(a);
}

}  // namespace aimdhf
