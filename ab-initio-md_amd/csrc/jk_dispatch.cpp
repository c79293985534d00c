// Dispatch tables over the per-class / per-type kernel objects (one object
// per template configuration, see the Makefile).
#include "aimdhf_internal.h"
#include "jk_digest.h"

namespace aimdhf {

#define DECLG(k) void launch_grad_class_##k(const GradArgs&, const int2*, long long, hipStream_t); \
    void launch_grad_keep_##k(const GradArgs&, const int2*, long long, hipStream_t);
DECLG(0) DECLG(1) DECLG(2) DECLG(3) DECLG(4) DECLG(5) DECLG(6) DECLG(7) DECLG(8) DECLG(9) DECLG(10)
DECLG(11) DECLG(12) DECLG(13) DECLG(14) DECLG(15) DECLG(16) DECLG(17) DECLG(18) DECLG(19) DECLG(20)
#undef DECLG

void launch_grad_one_class(int k, const GradArgs& a, const int2* list, long long nq, hipStream_t st) {
    typedef void (*Fn)(const GradArgs&, const int2*, long long, hipStream_t);
    static const Fn fns[21] = {
        launch_grad_class_0, launch_grad_class_1, launch_grad_class_2, launch_grad_class_3,
        launch_grad_class_4, launch_grad_class_5, launch_grad_class_6, launch_grad_class_7,
        launch_grad_class_8, launch_grad_class_9, launch_grad_class_10, launch_grad_class_11,
        launch_grad_class_12, launch_grad_class_13, launch_grad_class_14, launch_grad_class_15,
        launch_grad_class_16, launch_grad_class_17, launch_grad_class_18, launch_grad_class_19,
        launch_grad_class_20};
    fns[k](a, list, nq, st);
}

void launch_grad_keep(int k, const GradArgs& a, const int2* list, long long nq, hipStream_t st) {
    typedef void (*Fn)(const GradArgs&, const int2*, long long, hipStream_t);
    static const Fn fns[21] = {
        launch_grad_keep_0, launch_grad_keep_1, launch_grad_keep_2, launch_grad_keep_3,
        launch_grad_keep_4, launch_grad_keep_5, launch_grad_keep_6, launch_grad_keep_7,
        launch_grad_keep_8, launch_grad_keep_9, launch_grad_keep_10, launch_grad_keep_11,
        launch_grad_keep_12, launch_grad_keep_13, launch_grad_keep_14, launch_grad_keep_15,
        launch_grad_keep_16, launch_grad_keep_17, launch_grad_keep_18, launch_grad_keep_19,
        launch_grad_keep_20};
    fns[k](a, list, nq, st);
}

#define DECLS(k) void launch_eri_##k(const EriArgs&, long long, long long, long long, long long, hipStream_t); \
    void launch_digest_##k(const DigestArgs&, int, hipStream_t);
DECLS(0) DECLS(1) DECLS(2) DECLS(3) DECLS(4) DECLS(5) DECLS(6) DECLS(7) DECLS(8) DECLS(9) DECLS(10)
DECLS(11) DECLS(12) DECLS(13) DECLS(14) DECLS(15) DECLS(16) DECLS(17) DECLS(18) DECLS(19) DECLS(20)
#undef DECLS

void launch_eri(int k, const EriArgs& a, long long n64, long long h64, long long n32, long long h32, hipStream_t st) {
    typedef void (*Fn)(const EriArgs&, long long, long long, long long, long long, hipStream_t);
    static const Fn fns[21] = {
        launch_eri_0, launch_eri_1, launch_eri_2, launch_eri_3, launch_eri_4, launch_eri_5, launch_eri_6,
        launch_eri_7, launch_eri_8, launch_eri_9, launch_eri_10, launch_eri_11, launch_eri_12, launch_eri_13,
        launch_eri_14, launch_eri_15, launch_eri_16, launch_eri_17, launch_eri_18, launch_eri_19, launch_eri_20};
    fns[k](a, n64, h64, n32, h32, st);
}

void launch_digest(int k, const DigestArgs& a, int threads, hipStream_t st) {
    typedef void (*Fn)(const DigestArgs&, int, hipStream_t);
    static const Fn fns[21] = {
        launch_digest_0, launch_digest_1, launch_digest_2, launch_digest_3, launch_digest_4, launch_digest_5,
        launch_digest_6, launch_digest_7, launch_digest_8, launch_digest_9, launch_digest_10, launch_digest_11,
        launch_digest_12, launch_digest_13, launch_digest_14, launch_digest_15, launch_digest_16, launch_digest_17,
        launch_digest_18, launch_digest_19, launch_digest_20};
    fns[k](a, threads, st);
}

// integrals per block of quartet class k (heavier pair as bra)
long long store_block(int k) {
    static const int ncp[6] = {1, 3, 9, 6, 18, 36};
    int hi = 0;
    while ((hi + 1) * (hi + 2) / 2 <= k) ++hi;
    int lo = k - hi * (hi + 1) / 2;
    return (long long)ncp[hi] * ncp[lo];
}

}  // namespace aimdhf
