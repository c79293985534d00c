// Evaluation of screened unique quartets of one class (compiled once per class
// with -DAIMDHF_QCLASS=k) into the integral store. Quartet t of a list part
// (bra = heavier pair) keeps value v = cd NAB + ab (ab / cd over the bra / ket
// pair records) at (t / 64) 64 NAB NCD + 64 v + t % 64: tiles of 64 quartets,
// value-major, so that every store of a wavefront here and every load of the J/K
// digestion covers 64 consecutive words. In mixed precision the quartets below
// the switch are evaluated and held in FP32. The lanes of a wavefront take 64
// consecutive quartets (one bra run of the list: the same bra records for most
// of them); classes whose block does not fit the registers take one ket
// component per wavefront.

#include "jk_digest.h"
#include "md_eri.h"

#ifndef AIMDHF_QCLASS
#error "compile with -DAIMDHF_QCLASS=<0..20>"
#endif

namespace aimdhf {
using namespace md;

namespace {
constexpr int QC = AIMDHF_QCLASS;
constexpr int pc_hi() { int h = 0; while ((h + 1) * (h + 2) / 2 <= QC) ++h; return h; }
constexpr int pc_lo() { return QC - pc_hi() * (pc_hi() + 1) / 2; }
constexpr int la_of(int pc) { return pc == 0 ? 0 : pc <= 2 ? 1 : 2; }
constexpr int lb_of(int pc) { return pc - la_of(pc) * (la_of(pc) + 1) / 2; }
constexpr int LA = la_of(pc_hi()), LB = lb_of(pc_hi()), LC = la_of(pc_lo()), LD = lb_of(pc_lo());
using Qt = Quartet<LA, LB, LC, LD>;
constexpr bool SPLIT = split_by_cd<LA, LB, LC, LD>();
constexpr int BLK = Qt::NAB * Qt::NCD;
constexpr int NSPLIT = SPLIT ? Qt::NCD : 1;

template <int LA_, int LB_, int LC_, int LD_, typename Real>
__global__ __launch_bounds__(256) void k_eri(EriArgs a, Real* __restrict__ store, long long nq) {
    __shared__ double btab[BOYS_NGRID * BOYS_SROW];
    boys_stage(a.boys, LA_ + LB_ + LC_ + LD_, btab);
    const long long it = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long g = it >> 6;                    // wavefront: tile g / NSPLIT, ket component g % NSPLIT
    const int lane = (int)(it & 63);
    const long long q = g / NSPLIT * 64 + lane;
    if (q >= nq) return;
    const int P = a.cls_pairs[a.lbra[q]], Q = a.cls_pairs[a.lket[q]];
    const double* rb = a.recs + a.rec_off[P];
    const double* rk = a.recs + a.rec_off[Q];
    Real* out = store + (q >> 6) * (64 * BLK) + lane;
    if constexpr (SPLIT) {
        const int cd = (int)(g % NSPLIT);
        Real acc[Qt::NAB];
        eri_quartet_cd<LA_, LB_, LC_, LD_, true, Real>(rb, a.npp[P], rk, a.npp[Q], btab, cd, acc);
#pragma unroll
        for (int ab = 0; ab < Qt::NAB; ++ab) out[(cd * Qt::NAB + ab) * 64] = acc[ab];
    } else {
        Real acc[BLK];
        eri_quartet<LA_, LB_, LC_, LD_, true, Real>(rb, a.npp[P], rk, a.npp[Q], btab, acc);
#pragma unroll
        for (int ab = 0; ab < Qt::NAB; ++ab)
#pragma unroll
            for (int cd = 0; cd < Qt::NCD; ++cd) out[(cd * Qt::NAB + ab) * 64] = acc[ab * Qt::NCD + cd];
    }
}
}  // namespace

#define CAT2(a, b) a##b
#define CAT(a, b) CAT2(a, b)

// n64 quartets from a.lbra in FP64, the n32 after them in FP32
void CAT(launch_eri_, AIMDHF_QCLASS)(const EriArgs& a, long long n64, long long n32, hipStream_t st) {
    auto blocks = [](long long n) { return dim3((unsigned)(((n + 63) / 64 * 64 * NSPLIT + 255) / 256)); };
    if (n64 > 0) k_eri<LA, LB, LC, LD, double><<<blocks(n64), dim3(256), 0, st>>>(a, a.out64, n64);
    if (n32 > 0) {
        EriArgs b = a;
        b.lbra += n64;
        b.lket += n64;
        k_eri<LA, LB, LC, LD, float><<<blocks(n32), dim3(256), 0, st>>>(b, a.out32, n32);
    }
}

}  // namespace aimdhf
