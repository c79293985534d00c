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

// wavefronts a tile of contracted bras is split over: an (s s) bra has up to 64
// primitive pairs (cc-pVDZ), a (p s) one 24, (p p) and (d s) ones 9 and 8
constexpr int WH = QC == 0 ? 16 : pc_hi() == 1 ? 8 : pc_hi() <= 3 ? 4 : 1;

// one tile of 64 quartets (and ket component) per wavefront
template <int LA_, int LB_, int LC_, int LD_, typename Real>
__global__ __launch_bounds__(256) void k_eri(EriArgs a, Real* __restrict__ store, long long nq) {
    __shared__ double btab[BOYS_NGRID * BOYS_SROW];
    boys_stage(a.boys, LA_ + LB_ + LC_ + LD_, btab);
    const int lane = threadIdx.x & 63;
    const long long ng = (nq + 63) / 64 * NSPLIT;
    for (long long g = (long long)blockIdx.x * 4 + (threadIdx.x >> 6); g < ng; g += (long long)gridDim.x * 4) {
        const long long q = g / NSPLIT * 64 + lane;     // ket component g % NSPLIT
        if (q >= nq) continue;
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
}

// one tile (and ket component) per workgroup: wavefront w takes the w-th part of each
// quartet's bra primitives, the parts are added in wavefront order. A lane alone walks
// up to 36 x 36 (6-31G*) or 64 x 64 (cc-pVDZ) dependent primitive quartets, 0.28 us each:
// 0.36 ms for one water's (ss|ss), 2.5 ms for (H2O)8/cc-pVDZ, most of it this chain
// (four waters' geometry and first Fock matrix, with the Schwarz bounds split alike: 2.87 -> 1.43 ms)
template <int LA_, int LB_, int LC_, int LD_, typename Real>
__global__ __launch_bounds__(64 * WH) void k_eri_split(EriArgs a, Real* __restrict__ store, long long nq) {
    constexpr int NV = SPLIT ? Qt::NAB : BLK;           // values per lane
    constexpr int CH = NV < WH ? NV : WH;               // summed at a time
    __shared__ double btab[BOYS_NGRID * BOYS_SROW];
    __shared__ Real part[WH][CH][64];
    boys_stage(a.boys, LA_ + LB_ + LC_ + LD_, btab);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long g = blockIdx.x;
    const int cd = SPLIT ? (int)(g % NSPLIT) : 0;
    const long long q = g / NSPLIT * 64 + lane;
    const bool in = q < nq;
    const int P = a.cls_pairs[a.lbra[in ? q : nq - 1]], Q = a.cls_pairs[a.lket[in ? q : nq - 1]];
    const int np = in ? a.npp[P] : 0, ch = (np + WH - 1) / WH;
    const int b0 = w * ch < np ? w * ch : np, nb = b0 + ch < np ? ch : np - b0;
    const double* rb = a.recs + a.rec_off[P] + (size_t)b0 * Qt::RSB;
    const double* rk = a.recs + a.rec_off[Q];
    Real acc[NV];
    if constexpr (SPLIT)
        eri_quartet_cd<LA_, LB_, LC_, LD_, true, Real>(rb, nb, rk, a.npp[Q], btab, cd, acc);
    else
        eri_quartet<LA_, LB_, LC_, LD_, true, Real>(rb, nb, rk, a.npp[Q], btab, acc);
    Real* out = store + (q >> 6) * (64 * BLK) + lane;
    static_for<0, (NV + CH - 1) / CH>([&](auto cc) {
        constexpr int v0 = decltype(cc)::value * CH;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (v0 + i < NV) part[w][i][lane] = acc[v0 + i < NV ? v0 + i : 0];
        __syncthreads();
        if (w < CH && v0 + w < NV && in) {
            Real s = Real(0);
#pragma unroll
            for (int k = 0; k < WH; ++k) s += part[k][w][lane];
            const int v = v0 + w;
            out[(SPLIT ? cd * Qt::NAB + v : (v % Qt::NCD) * Qt::NAB + v / Qt::NCD) * 64] = s;
        }
    });
}

// quartets [0, nh) of the part split over wavefronts, [nh, n) one tile per wavefront
template <typename Real>
void launch_part(const EriArgs& a, Real* out, long long n, long long nh, hipStream_t st) {
    if (WH == 1) nh = 0;
    nh = (nh + 63) / 64 * 64;
    if (nh > n) nh = n;
    if constexpr (WH > 1) {
        // a launch takes fewer than 2^32 work-items, and past that the grid wraps without an
        // error: at most 2^21 workgroups (of up to 1024) at a time
        constexpr long long SLICE = (1 << 21) / NSPLIT * 64;
        for (long long q0 = 0; q0 < nh; q0 += SLICE) {
            EriArgs b = a;
            b.lbra += q0;
            b.lket += q0;
            const long long nq = q0 + SLICE < nh ? SLICE : nh - q0;
            k_eri_split<LA, LB, LC, LD, Real>
                <<<dim3((unsigned)((nq + 63) / 64 * NSPLIT)), dim3(64 * WH), 0, st>>>(b, out + q0 * BLK, nq);
        }
    }
    if (n > nh) {
        EriArgs b = a;
        b.lbra += nh;
        b.lket += nh;
        const long long blocks = ((n - nh + 63) / 64 * NSPLIT + 3) / 4;
        k_eri<LA, LB, LC, LD, Real><<<dim3((unsigned)(blocks > 8192 ? 8192 : blocks)), dim3(256), 0, st>>>(
            b, out + nh * BLK, n - nh);
    }
}
}  // namespace

#define CAT2(a, b) a##b
#define CAT(a, b) CAT2(a, b)

// n64 quartets from a.lbra in FP64 (the first h64 of contracted bras), the n32 after
// them in FP32 (the first h32)
void CAT(launch_eri_, AIMDHF_QCLASS)(const EriArgs& a, long long n64, long long h64, long long n32, long long h32,
                                     hipStream_t st) {
    if (n64 > 0) launch_part<double>(a, a.out64, n64, h64, st);
    if (n32 > 0) {
        EriArgs b = a;
        b.lbra += n64;
        b.lket += n64;
        launch_part<float>(b, a.out32, n32, h32, st);
    }
}

}  // namespace aimdhf
