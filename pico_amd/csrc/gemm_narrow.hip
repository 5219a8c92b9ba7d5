// pico_amd/csrc/gemm_narrow.hip -- the opt-in bf16 and split-bf16 products of fp32
// operands, staged as the fp32 product's (gemm_split.h).
//
//  * P = 1: operands rounded to bf16 (nearest even), one matrix instruction per
//    block and 16 k.  P = 2: hi = bf16(x) and lo = bf16(x - hi), and hi.hi +
//    hi.lo + lo.hi per 16 k, in that order.
//  * Bound: P = 1 by staging -- an fp32 operand value costs 4 bytes of loads for
//    as many matrix cycles as 2 of a bf16 operand -- P = 2 by the matrix cores
//    (834 TFLOP/s nominal) and the split.  Eight waves of 128x64, two per
//    SIMD, hide a 256x256 tile's staging behind each other's matrix instructions.
//  * A slice is 32 k, two steps of 16: the second step's fragments are read
//    under the first step's products, the next slice's first ones under the
//    second's; one barrier.
//  * One group of waves per tile, so that every shape and epilogue adds K in the
//    same order: the composed and fused operations agree bit for bit, and so do
//    the split product here and on operands split beforehand.
//  * Ragged sizes go through the buffer resources' own bounds, as there; those of
//    a row-contiguous operand, which cost a resource per k row, only in the last
//    slices (bounded in every slice, scalar instructions were the bound: A^T.B
//    of [192, 6464], K 1984, bf16 73 -> 41 us, [266, 1340], K 5136, A.B split 130 ->
//    98).
//
// Bf16 against the four-wave kernel it replaces, us: 4096^3 A.B / A.B^T / A^T.B
// 173 / 145 / 190 -> 166 / 136 / 175, [8192, 4096] K 768 87 -> 79.  Ragged:
// [2000, 1503] K 1001 54 -> 26 (split bf16 64 -> 37), its A.B^T 73 -> 27 (77 ->
// 36), [333, 517] K 1201 32 -> 15 (35 -> 18).  gemm.hip keeps that kernel for
// the whole tiles where it is the faster one (narrow_here).
#include <type_traits>

#include "gemm_common.h"

namespace {

using namespace pkg;

#include "gemm_split.h"

constexpr int W = 32;  // k per slice

template <bool TA, bool TB, int EDGE, class T, int P, int EPI>
__global__ __launch_bounds__(T::THREADS, T::WPS) void gemm_narrow_kernel(GemmParams p) {
    constexpr int BM = T::BM, BN = T::BN, TM = T::TM, TN = T::TN, NT_ = T::THREADS;
    constexpr bool AK = !TA, BKF = TB, PAIR = EPI == kEpiSwigluFwd;
    using OA = SplitOperand<AK, BM, NT_, W>;
    using OB = SplitOperand<BKF, BN, NT_, W>;
    constexpr int PART = (BM + BN) * SK, STEP = P * PART, STAGE = 2 * STEP;
    // (the epilogue stages at least 32 rows of floats)
    constexpr int EPI_SHORTS = EPI == kEpiPlain ? 0 : 32 * (BN + 4) * 2;
    __shared__ __attribute__((aligned(16))) short lds[2 * STAGE > EPI_SHORTS ? 2 * STAGE : EPI_SHORTS];

    const TileJob job = tile_job<T>(p);
    if(job.skip) return;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64;
    const int wm = w / T::WGN, wn = w % T::WGN;
    const int lr = l & 31, lh = l >> 5;
    const int ar0 = wm * TM * 32, br0 = wn * TN * 32;
    const int nslices = (int)((job.kend - job.kbeg + W - 1) / W);

    f32x16 acc[TM][TN];
#pragma unroll
    for(int i = 0; i < TM; ++i)
#pragma unroll
        for(int j = 0; j < TN; ++j)
#pragma unroll
            for(int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    if(nslices > 0) {
        const SplitSource sa = {reinterpret_cast<const char*>(job.A + (AK ? job.row0 * p.lda : job.row0)),
                                4 * ((AK ? (p.M - 1 - job.row0) * p.lda + p.K
                                         : (p.K - 1) * p.lda + p.M - job.row0)),
                                AK ? 4 : p.lda * 4};
        const SplitSource sb = {reinterpret_cast<const char*>(job.B + (BKF ? job.col0 * p.ldb : job.col0)),
                                4 * ((BKF ? (p.N - 1 - job.col0) * p.ldb + p.K
                                          : (p.K - 1) * p.ldb + p.N - job.col0)),
                                BKF ? 4 : p.ldb * 4};
        const int64_t shift = p.pair_F - BN / 2;
        // the slices before this one lie inside the operands with their whole
        // tile rows: a row-contiguous operand's rows past its last one are read
        // from the next k rows, `past` of them behind the end
        // (a loop of their own, which the split-bf16 256x256 and A^T.B 128x128 tiles
        // have no registers for)
        constexpr bool TWO = EDGE == kPartial && !(AK && BKF) &&
                             !(P == 2 && (TM * TN == 8 || (TM * TN == 2 && !AK)));
        int inside = 0;
        if constexpr(TWO) {
            auto past = [](int64_t over, int64_t ld) {
                return over > 0 ? (int)(((unsigned)over + (unsigned)ld - 1) / (unsigned)ld) : 0;
            };
            const int pa = AK ? 0 : past(job.row0 + BM - p.M, p.lda);
            const int pb = BKF ? 0 : past(job.col0 + BN + (PAIR ? shift : 0) - p.N, p.ldb);
            inside = (int)(max(min(job.kend, p.K - max(pa, pb)) - job.kbeg, (int64_t)0) / W);
        }
        float ra[OA::ITEMS][OA::KPI], rb[OB::ITEMS][OB::KPI];
        // (TAIL: slices from `inside` on)
        auto load = [&](int s, auto tail) {
            constexpr bool TAIL = decltype(tail)::value;
            const int64_t k0 = job.kbeg + (int64_t)min(s, nslices - 1) * W;
            if constexpr(EDGE == kFar) {
                far_load<AK, BM, NT_, false, W>(job.A, p.lda, job.row0, p.M, k0, job.kend, 0, ra);
                far_load<BKF, BN, NT_, PAIR, W>(job.B, p.ldb, job.col0, p.N, k0, job.kend, shift, rb);
            } else {
                constexpr bool EA = EDGE == kPartial && (AK || TAIL), EB = EDGE == kPartial && (BKF || TAIL);
                split_load<AK, EA, BM, NT_, false, W>(sa, p.lda, k0, 0, ra);
                split_load<BKF, EB, BN, NT_, PAIR, W>(sb, p.ldb, k0, shift, rb);
            }
        };
        auto store = [&](int stage) {
            split_store<P, AK, BM, NT_, PART, W>(lds + stage * STAGE, ra, 1.0f);
            split_store<P, BKF, BN, NT_, PART, W>(lds + stage * STAGE + BM * SK, rb, 1.0f);
        };
        auto mask = [&](int s, auto tail) {
            if constexpr(decltype(tail)::value && EDGE == kPartial && (AK || BKF)) {
                const int64_t limit = job.kend - job.kbeg - (int64_t)min(s, nslices - 1) * W;
                if(limit < W) {
                    if(AK) split_mask<AK, BM, NT_, W>((int)limit, ra);
                    if(BKF) split_mask<BKF, BN, NT_, W>((int)limit, rb);
                }
            }
        };
        const int fo = lr * SK + ((lh ^ (lr >> 2)) & 1) * 8;
        auto read = [&](SplitFrag<TM, TN>& f, int stage, int step, int part) {
            const short* t = lds + stage * STAGE + step * STEP + part * PART + fo;
#pragma unroll
            for(int i = 0; i < TM; ++i)
                f.a[i] = *reinterpret_cast<const bf16x8*>(t + (ar0 + i * 32) * SK);
#pragma unroll
            for(int j = 0; j < TN; ++j)
                f.b[j] = *reinterpret_cast<const bf16x8*>(t + (BM + br0 + j * 32) * SK);
        };
        auto mma = [&](const SplitFrag<TM, TN>& x, const SplitFrag<TM, TN>& y) {
#pragma unroll
            for(int i = 0; i < TM; ++i)
#pragma unroll
                for(int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.a[i], y.b[j], acc[i][j], 0,
                                                                        0, 0);
        };
        using Bounded = std::integral_constant<bool, EDGE != kWhole>;
        load(0, Bounded());
        mask(0, Bounded());
        store(0);
        load(1, Bounded());
        __syncthreads();
        SplitFrag<TM, TN> h0, h1, lo;
        read(h0, 0, 0, 0);
        constexpr int NB = TM * TN, RD = TM + TN;
        constexpr int CV = (OA::ITEMS * OA::KPI + OB::ITEMS * OB::KPI) * (P == 2 ? 7 : 1) / 2;
        constexpr int WR = P * (OA::ITEMS + OB::ITEMS);
        constexpr int LD = OA::ITEMS * OA::LOADS + OB::ITEMS * OB::LOADS;
        auto slice = [&](int s, auto tail) {
            const int cur = s & 1;
            mask(s + 1, tail);
            if constexpr(P == 2) read(lo, cur, 0, 1);
            read(h1, cur, 1, 0);
            store(cur ^ 1);
            load(s + 2, tail);
            mma(h0, h0);
            if constexpr(P == 2) {
                mma(h0, lo);
                mma(lo, h0);
            }
            split_sched<(P == 2 ? 3 : 1) * NB, P * RD, CV, WR, LD>();
            __builtin_amdgcn_sched_barrier(0);
            if constexpr(P == 2) {
                read(lo, cur, 1, 1);
                mma(h1, h1);
                mma(h1, lo);
                split_sched<2 * NB, RD, 0, 0, 0>();
                __builtin_amdgcn_sched_barrier(0);
            }
            __syncthreads();
            read(h0, cur ^ 1, 0, 0);
            if constexpr(P == 2) mma(lo, h1);
            else mma(h1, h1);
            split_sched<NB, RD, 0, 0, 0>();
            __builtin_amdgcn_sched_barrier(0);
        };
        int s = 0;
        if constexpr(TWO) {
#pragma unroll 1
            for(; s + 2 < inside; ++s) slice(s, std::false_type());
        }
#pragma unroll 1
        for(; s < nslices; ++s) slice(s, Bounded());
    }
    if constexpr(EPI == kEpiPlain)
        store_tile<EDGE == kWhole ? kEdgeNone : kEdgeScalar, TM, TN, 1>(p, job, acc, ar0, br0, lr, lh, 0);
    else
        staged_epilogue<EPI, T, (int)sizeof(lds) / 4>(p, job, acc, reinterpret_cast<float*>(lds), ar0,
                                                      br0, lr, lh);
}

using Narrow256 = SplitTile<2, 4, 4, 2, 1, 2, 1>;
using Narrow128 = SplitTile<2, 4, 2, 1, 1, 4, 1>;
using Narrow64 = SplitTile<2, 2, 1, 1, 1, 4, 1>;

template <bool TA, bool TB, int EDGE, class T, int P>
void launch_narrow_kernel(const GemmParams& gp, dim3 grid, hipStream_t st) {
    if constexpr(!TA && TB) {
        if(gp.sg_a) {
            gemm_narrow_kernel<TA, TB, EDGE, T, P, kEpiSwiglu><<<grid, T::THREADS, 0, st>>>(gp);
            return;
        }
    }
    if constexpr(!TA && !TB) {
        if(gp.sf_h) {
            gemm_narrow_kernel<TA, TB, EDGE, T, P, kEpiSwigluFwd><<<grid, T::THREADS, 0, st>>>(gp);
            return;
        }
        if(gp.Cin) {
            gemm_narrow_kernel<TA, TB, EDGE, T, P, kEpiAdd><<<grid, T::THREADS, 0, st>>>(gp);
            return;
        }
    }
    gemm_narrow_kernel<TA, TB, EDGE, T, P, kEpiPlain><<<grid, T::THREADS, 0, st>>>(gp);
}

template <bool TA, bool TB, class T, int P>
void launch_narrow_tile(const GemmParams& gp, int64_t batch, bool edge, hipStream_t st) {
    dim3 grid((unsigned)(gp.tiles_m * gp.tiles_n), (unsigned)(gp.splits > 1 ? gp.splits : batch));
    // (whole split-bf16 tiles come here only when unaligned or too large for the
    // other kernel)
    constexpr int kFull = P == 1 ? kWhole : kPartial;
    if(edge)
        launch_narrow_kernel<TA, TB, kPartial, T, P>(gp, grid, st);
    else
        launch_narrow_kernel<TA, TB, kFull, T, P>(gp, grid, st);
}

template <bool TA, bool TB, int P>
int launch_layout(const GemmParams& gp, int64_t batch, bool edge, TileKind kind, hipStream_t st) {
    switch(kind) {
    case kTile256: launch_narrow_tile<TA, TB, Narrow256, P>(gp, batch, edge, st); break;
    case kTile64: {
        if(!gp.far) {
            launch_narrow_tile<TA, TB, Narrow64, P>(gp, batch, edge, st);
            break;
        }
        dim3 grid((unsigned)(gp.tiles_m * gp.tiles_n),
                  (unsigned)(gp.splits > 1 ? gp.splits : batch));
        launch_narrow_kernel<TA, TB, kFar, Narrow64, P>(gp, grid, st);
        break;
    }
    default: launch_narrow_tile<TA, TB, Narrow128, P>(gp, batch, edge, st);
    }
    return pk::launch_status(P == 1 ? "pk_gemm_bf16_f32" : "pk_gemm_bf16x3_f32");
}

template <int P>
int launch_parts(bool ta, bool tb, const GemmParams& gp, int64_t batch, bool edge, TileKind kind,
                 hipStream_t st) {
    if(!ta && !tb) return launch_layout<false, false, P>(gp, batch, edge, kind, st);
    if(!ta && tb) return launch_layout<false, true, P>(gp, batch, edge, kind, st);
    if(ta && !tb) return launch_layout<true, false, P>(gp, batch, edge, kind, st);
    return launch_layout<true, true, P>(gp, batch, edge, kind, st);
}

}  // namespace

namespace pkg {

int launch_narrow(bool ta, bool tb, int parts, const GemmParams& gp, int64_t batch, bool edge,
                  TileKind kind, hipStream_t st) {
    return parts == 1 ? launch_parts<1>(ta, tb, gp, batch, edge, kind, st)
                      : launch_parts<2>(ta, tb, gp, batch, edge, kind, st);
}

}  // namespace pkg
