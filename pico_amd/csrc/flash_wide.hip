// pico_amd/csrc/flash_wide.hip -- fused causal attention for head sizes 32, 96 and
// 128 (flash_attention.hip holds head size 64).
//
// The chain of products that served these sizes writes and reads the [T, T]
// probabilities of every head five times and pads every causal product to its
// tiles (batch 4, 8 heads of 128, T 1000: products of 4.1 GFLOP in 87-139 us each).
// Here scores and probabilities stay in registers, as in the head-64 kernels and
// with their layout: S^T = K.Q^T puts one query (backward: one key) in a lane, so
// the softmax is lane-local but for one exchange between the wave's halves, and
// P^T is already the B operand of the next product, the contraction taken in the
// accumulator's row order acc_row.  fp32 matrix instructions throughout.
//
// What differs from head size 64:
//  * A streamed block is 32 rows (two 64-row tiles of K and V at 128 dims would
//    leave one workgroup per CU), double-buffered, loaded straight into LDS.
//  * A workgroup is four waves: 128 rows, or, while that leaves fewer than two
//    workgroups per CU, 64 rows with the streamed blocks dealt to two waves per
//    row group, whose sums meet at the end (batch 4, 8 heads of 128, T 1000: two-wave
//    workgroups left the heaviest rows' chain on two SIMDs of a CU, forward 160 us,
//    backward 385; dealt to four 129 and 284, dispatched as below 105 and 242).
//  * Workgroups run heaviest first; where two or more share a CU from the start,
//    every second round of 256 is reversed, pairing the heaviest with the lightest.
//  * Two score chains (even and odd dims) alternate, since a wave may have a SIMD
//    to itself: the backward's K and V fragments and its dK and dV accumulators
//    alone are 256 registers at 128 dims.
// Bound by the fp32 matrix cores, and at few rows by the longest one's chain.
// Forward / backward us, then the chain on the bf16 matrix cores:
//    batch 4, 8 heads of 128, T 1000   105 / 242   175 / 282
//    batch 8, 8 heads of 96, T 1024    143 / 372   340 / 547
//    batch 8, 24 heads of 32, T 1024   142 / 455   885 / 1512
//    batch 1, 6 heads of 128, T 2048   169 / 380   154 / 284 (the chain runs)
#include <math.h>

#include "pk_common.h"

namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr int64_t kCUs = 256;
constexpr float kTau = 8.0f;  // the running max is raised when a block exceeds it by this (log2)
constexpr int QB = 32;        // rows of a streamed block, and of a wave

struct WideParams {
    const float *q, *k, *v, *o, *dout, *lse;
    float *out, *lse_out, *dq, *dk, *dv;
    float *consts, *ds;  // [B*H][Tp/32][2][32] L2 and D rows; dS tiles
    int64_t B, H, T, Tp, D, ld;
    float scale;
    int flags;
};

__device__ __forceinline__ f32x16 mfma(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 splat16(float x) {
    f32x16 z;
#pragma unroll
    for(int r = 0; r < 16; ++r) z[r] = x;
    return z;
}
__device__ __forceinline__ int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// dS tiles (32 x 32) of a head's causal triangle, packed by rows of tiles; inside a
// tile the 16 values of a dQ lane (q, half) are consecutive: (2q + half)*16 + s
__host__ __device__ __forceinline__ int64_t ds_tiles(int64_t Tp) {
    return (Tp / 32) * (Tp / 32 + 1) / 2;
}

// workgroup b's place in heaviest-first order.  A CU that holds one workgroup
// (LDS or registers) takes the next heaviest as it frees; where it holds two or
// more (SHARED), b and b + 256 run on one CU from the start, so every second
// round of 256 is reversed.
template <bool SHARED>
__device__ __forceinline__ int64_t place(int64_t b, int64_t n) {
    if(!SHARED) return b;
    const int64_t round = b / kCUs, lo = round * kCUs, hi = min(lo + kCUs, n);
    return (round & 1) ? lo + hi - 1 - b : b;
}

typedef __attribute__((address_space(3))) void lds_ptr_t;

// rows of HDT + 4 floats: 16 bytes apart modulo 128, so 128-bit reads down a column
// of rows touch every bank once.  A tile is filled by LOADS 1 KB direct loads, the
// last of which runs past row 31 into the tile's tail.
template <int HDT>
struct WideTile {
    static constexpr int LDT = HDT + 4;
    static constexpr int LOADS = (QB * LDT * 4 + 1023) / 1024;
    static constexpr int FLOATS = LOADS * 256;
};

template <int HDT, int NW>
struct WideLoad {
    using Tl = WideTile<HDT>;
    static constexpr int N = (Tl::LOADS + NW - 1) / NW;
    unsigned off[N];
    __device__ __forceinline__ WideLoad(int64_t ld, int w, int l) {
#pragma unroll
        for(int i = 0; i < N; ++i) {
            const int f = 256 * (w + NW * i) + 4 * l, r = f / Tl::LDT, c = f % Tl::LDT;
            off[i] = (unsigned)((r * ld + (c < HDT ? c : 0)) * 4);
        }
    }
    // rows row0.. of a head of T rows; those at or past T read as zeros (the resource
    // ends at the head's last element, and the whole lane offset is bounds-checked)
    __device__ __forceinline__ void issue(const float* head, int64_t T, int64_t ld, int64_t row0,
                                          float* tile, int w) const {
        const int64_t bytes = T > row0 ? ((T - 1 - row0) * ld + HDT) * 4 : 0;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(head + row0 * ld), (short)0, (int)bytes, 0x00020000);
#pragma unroll
        for(int i = 0; i < N; ++i)
            if(NW * i + NW <= Tl::LOADS || w + NW * i < Tl::LOADS)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rs, (lds_ptr_t*)(tile + 256 * (w + NW * i)), 16, off[i], 0, 0, 0);
    }
};

__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// a lane's half of one row: dims HDT/2*h .. +HDT/2-1, times mul; zeros past the end
template <int HDT>
__device__ __forceinline__ void load_frag(const float* __restrict__ row, int h, float (&f)[HDT / 2],
                                          float mul, bool ok) {
    const f32x4* p = reinterpret_cast<const f32x4*>(row + HDT / 2 * h);
#pragma unroll
    for(int i = 0; i < HDT / 8; ++i) {
        const f32x4 x = ok ? p[i] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for(int e = 0; e < 4; ++e) f[4 * i + e] = x[e] * mul;
    }
}

// out[row][d] = acc * mul (+ out): one row per lane, 4 consecutive d per float4
template <int NB>
__device__ __forceinline__ void store_rowT(float* dst, const f32x16 (&acc)[NB], int lh,
                                           float mul, bool accumulate) {
#pragma unroll
    for(int cb = 0; cb < NB; ++cb)
#pragma unroll
        for(int g = 0; g < 4; ++g) {
            f32x4 v;
#pragma unroll
            for(int e = 0; e < 4; ++e) v[e] = acc[cb][4 * g + e] * mul;
            f32x4* p = reinterpret_cast<f32x4*>(dst + cb * 32 + 8 * g + 4 * lh);
            if(accumulate) v += *p;
            *p = v;
        }
}

// three LDS reads ahead, then one more per PER matrix instructions
template <int N, int PER>
__device__ __forceinline__ void read_ahead() {
    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
    for(int i = 0; i < N; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
}

// ------------------------------------------------------------------- forward
template <int HDT, int RG, int KS>
__global__ __launch_bounds__(256, KS == 1 || HDT == 32 ? 2 : 1) void wide_fwd(WideParams p) {
    using Tl = WideTile<HDT>;
    constexpr int NB = HDT / 32, LDT = Tl::LDT, ROWS = 32 * RG;
    __shared__ __attribute__((aligned(16))) float sK[2][KS][Tl::FLOATS];
    __shared__ __attribute__((aligned(16))) float sV[2][KS][Tl::FLOATS];
    const int64_t BH = p.B * p.H, nqb = (p.Tp + ROWS - 1) / ROWS;
    const int64_t rank = place<(KS == 1 || HDT == 32)>(blockIdx.x, gridDim.x);
    const int64_t qb = nqb - 1 - rank / BH, bh = rank % BH, b = bh / p.H, h = bh % p.H;
    const int64_t base = b * p.T * p.ld + h * HDT;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63, lq = l & 31, lh = l >> 5;
    const int rg = w % RG, ks = w / RG;
    const int64_t q0 = qb * ROWS + rg * QB, qi = q0 + lq;
    const int steps = (int)((qb + 1) * RG / KS), nw = (int)(q0 / QB) + 1;

    const WideLoad<HDT, 4> blk(p.ld, w, l);
    const float *K = p.k + base, *V = p.v + base;
    auto issue = [&](int it, int st) {
#pragma unroll
        for(int x = 0; x < KS; ++x) {
            blk.issue(K, p.T, p.ld, (int64_t)(it * KS + x) * QB, sK[st][x], w);
            blk.issue(V, p.T, p.ld, (int64_t)(it * KS + x) * QB, sV[st][x], w);
        }
    };
    issue(0, 0);
    float qf[HDT / 2];
    load_frag<HDT>(p.q + base + qi * p.ld, lh, qf, p.scale * kLog2e, qi < p.T);
    f32x16 o[NB];
#pragma unroll
    for(int cb = 0; cb < NB; ++cb) o[cb] = splat16(0.0f);
    // m: the running max, raised when a block's max passes it by kTau; ref: what is
    // subtracted, m or 0 while every score has been -inf
    float m = -INFINITY, ref = 0.0f, ls = 0.0f;
    auto block = [&](int j, const float* __restrict__ tk, const float* __restrict__ tv) {
        // scores in log2 units.  ref is taken off the finished sum, 16 subtractions a
        // block: as the sum's start it would absorb the scores of a row whose
        // first keys lie far below the others
        f32x16 s = splat16(0.0f), s1 = splat16(0.0f);
        const f32x4* a4 = reinterpret_cast<const f32x4*>(tk + lq * LDT + HDT / 2 * lh);
#pragma unroll
        for(int i = 0; i < HDT / 8; ++i) {
            const f32x4 a = a4[i];
            s = mfma(a[0], qf[4 * i + 0], s);
            s1 = mfma(a[1], qf[4 * i + 1], s1);
            s = mfma(a[2], qf[4 * i + 2], s);
            s1 = mfma(a[3], qf[4 * i + 3], s1);
        }
        read_ahead<HDT / 8 - 3, 4>();
        __builtin_amdgcn_sched_barrier(0);
        float mx = -INFINITY;
#pragma unroll
        for(int r = 0; r < 16; ++r) {
            s[r] += s1[r];
            if(j == nw - 1 && acc_row(r, lh) > lq) s[r] = -INFINITY;  // the diagonal block
            mx = fmaxf(mx, s[r]);
        }
        if(__builtin_amdgcn_ballot_w64(mx > m + kTau)) {
            mx = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
            ref = mx == -INFINITY ? 0.0f : mx;
            const float alpha = __builtin_amdgcn_exp2f(m - ref);
#pragma unroll
            for(int cb = 0; cb < NB; ++cb)
#pragma unroll
                for(int r = 0; r < 16; ++r) o[cb][r] *= alpha;
            ls *= alpha;
            m = mx;
        }
#pragma unroll
        for(int r = 0; r < 16; ++r) s[r] -= ref;
        float l0 = 0.0f, l1 = 0.0f;
#pragma unroll
        for(int r = 0; r < 16; r += 2) {
            s[r] = __builtin_amdgcn_exp2f(s[r]);
            s[r + 1] = __builtin_amdgcn_exp2f(s[r + 1]);
            l0 += s[r];
            l1 += s[r + 1];
        }
        ls += l0 + l1;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for(int r = 0; r < 16; ++r)
#pragma unroll
            for(int cb = 0; cb < NB; ++cb)
                o[cb] = mfma(tv[acc_row(r, lh) * LDT + cb * 32 + lq], s[r], o[cb]);
        read_ahead<16 * NB - 3, 1>();
        __builtin_amdgcn_sched_barrier(0);
    };
    for(int it = 0; it < steps; ++it) {
        wait_loads();
        __syncthreads();  // this step's blocks are in; the other buffers are free
        if(it + 1 < steps) issue(it + 1, (it + 1) & 1);
        if(it * KS + ks < nw) block(it * KS + ks, sK[it & 1][ks], sV[it & 1][ks]);
    }
    if constexpr(KS == 2) {
        // the second wave of a row group hands over its keys' sums
        __syncthreads();
        float* mine = &sK[0][0][0] + rg * (NB * 16 + 2) * 64 + l;
        static_assert(RG * (NB * 16 + 2) * 64 <= 4 * Tl::FLOATS, "the sums fit");
        if(ks == 1) {
#pragma unroll
            for(int cb = 0; cb < NB; ++cb)
#pragma unroll
                for(int r = 0; r < 16; ++r) mine[(cb * 16 + r) * 64] = o[cb][r];
            mine[NB * 16 * 64] = m;
            mine[(NB * 16 + 1) * 64] = ls;
        }
        __syncthreads();
        if(ks == 1) return;
        const float m1 = mine[NB * 16 * 64], l1 = mine[(NB * 16 + 1) * 64], mt = fmaxf(m, m1);
        const float a0 = __builtin_amdgcn_exp2f(m - mt), a1 = __builtin_amdgcn_exp2f(m1 - mt);
#pragma unroll
        for(int cb = 0; cb < NB; ++cb)
#pragma unroll
            for(int r = 0; r < 16; ++r) o[cb][r] = o[cb][r] * a0 + mine[(cb * 16 + r) * 64] * a1;
        ls = ls * a0 + l1 * a1;
        m = mt;
    }
    if(qi >= p.T) return;
    const float lsum = ls + __shfl_xor(ls, 32, 64);
    store_rowT<NB>(p.out + b * p.T * p.D + h * HDT + qi * p.D, o, lh, 1.0f / lsum, false);
    if(lh == 0 && p.lse_out) p.lse_out[bh * p.T + qi] = (m + log2f(lsum)) * kLn2;
}

// ------------------------------------------------------------------ backward
// L2 = lse*log2(e) and D = rowsum(dO*O) of every row, 32 lanes a row; rows T..Tp-1
// get L2 = +inf and D = 0: no probability
template <int HDT>
__global__ void wide_consts(WideParams p) {
    const int64_t n = p.B * p.H * p.Tp;
    const int c = threadIdx.x & 31;
    for(int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 5; i < n;
        i += ((int64_t)gridDim.x * blockDim.x) >> 5) {
        const int64_t bh = i / p.Tp, t = i % p.Tp, b = bh / p.H, h = bh % p.H;
        float s = 0.0f;
        if(t < p.T && c < HDT / 4) {
            const int64_t off = (b * p.T + t) * p.D + h * HDT;
            const f32x4 a = reinterpret_cast<const f32x4*>(p.dout + off)[c];
            const f32x4 o = reinterpret_cast<const f32x4*>(p.o + off)[c];
            s = a[0] * o[0] + a[1] * o[1] + a[2] * o[2] + a[3] * o[3];
        }
#pragma unroll
        for(int e = 16; e > 0; e >>= 1) s += __shfl_xor(s, e, 32);
        if(c == 0) {
            float* blk = p.consts + (bh * (p.Tp / QB) + t / QB) * 2 * QB + t % QB;
            blk[0] = t < p.T ? p.lse[bh * p.T + t] * kLog2e : INFINITY;
            blk[QB] = s;
        }
    }
}

// one lane's 16 bytes of a head's row constants; past their end: zeros
__device__ __forceinline__ void load_consts(const float* consts, int nq, int offset, float* lds) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(consts), (short)0, nq * 2 * QB * 4, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t*)lds, 16, offset, 0, 0, 0);
}

// dK, dV: one key per lane; query blocks with q >= key stream through LDS
//   P = exp2(S - L2)   dV^T += dO^T.P   dS = P*(dP - D)   dK^T += Q^T.dS
template <int HDT, int RG, int KS>
__global__ __launch_bounds__(256, 1) void wide_bwd_dkdv(WideParams p) {
    using Tl = WideTile<HDT>;
    constexpr int NB = HDT / 32, LDT = Tl::LDT, ROWS = 32 * RG;
    __shared__ __attribute__((aligned(16))) float sQ[2][KS][Tl::FLOATS];
    __shared__ __attribute__((aligned(16))) float sO[2][KS][Tl::FLOATS];
    __shared__ __attribute__((aligned(16))) float sC[2][KS][256];  // L2, then D (a 1 KB load)
    const int64_t BH = p.B * p.H, rank = place<(HDT == 32)>(blockIdx.x, gridDim.x);
    const int64_t kb = rank / BH, bh = rank % BH, b = bh / p.H, h = bh % p.H;
    const int64_t base = b * p.T * p.ld + h * HDT, obase = b * p.T * p.D + h * HDT;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63, lq = l & 31, lh = l >> 5;
    const int rg = w % RG, ks = w / RG;
    const int64_t k0 = kb * ROWS + rg * QB, ki = k0 + lq, kg = k0 / QB;
    const WideLoad<HDT, 4> blq(p.ld, w, l), blo(p.D, w, l);
    const float *Q = p.q + base, *O = p.dout + obase;
    const int nq = (int)(p.Tp / QB), j0 = (int)(kb * RG);
    const float* consts = p.consts + bh * nq * 2 * QB;
    auto issue = [&](int it, int st) {
#pragma unroll
        for(int x = 0; x < KS; ++x) {
            const int j = j0 + it * KS + x;
            blq.issue(Q, p.T, p.ld, (int64_t)j * QB, sQ[st][x], w);
            blo.issue(O, p.T, p.D, (int64_t)j * QB, sO[st][x], w);
            if(w == 3)  // 16 lanes' worth is used
                load_consts(consts, nq, 16 * l + j * 2 * QB * 4, sC[st][x]);
        }
    };
    issue(0, 0);
    float kf[HDT / 2], vf[HDT / 2];
    load_frag<HDT>(p.k + base + ki * p.ld, lh, kf, p.scale * kLog2e, ki < p.T);
    load_frag<HDT>(p.v + base + ki * p.ld, lh, vf, 1.0f, ki < p.T);
    f32x16 dv[NB], dk[NB];
#pragma unroll
    for(int cb = 0; cb < NB; ++cb) dv[cb] = dk[cb] = splat16(0.0f);
    float* dsk = p.ds + bh * ds_tiles(p.Tp) * 1024 + ((lq >> 2) & 1) * 16 + 4 * (lq >> 3) + (lq & 3);
    auto block = [&](int j, const float* __restrict__ tq, const float* __restrict__ to,
                     const float* __restrict__ tc) {
        f32x16 sc = splat16(0.0f), dp = splat16(0.0f);
        const f32x4* q4 = reinterpret_cast<const f32x4*>(tq + lq * LDT + HDT / 2 * lh);
        const f32x4* o4 = reinterpret_cast<const f32x4*>(to + lq * LDT + HDT / 2 * lh);
#pragma unroll
        for(int i = 0; i < HDT / 8; ++i) {
            const f32x4 a = q4[i], c = o4[i];
#pragma unroll
            for(int e = 0; e < 4; ++e) {
                sc = mfma(a[e], kf[4 * i + e], sc);
                dp = mfma(c[e], vf[4 * i + e], dp);
            }
        }
        read_ahead<HDT / 4 - 3, 4>();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for(int r = 0; r < 16; ++r) {
            const int qr = acc_row(r, lh);
            const bool hidden = j == kg && qr < lq;  // the diagonal block: query before key
            const float pr = __builtin_amdgcn_exp2f(sc[r] - tc[qr]);
            const float g = pr * (dp[r] - tc[QB + qr]);
            sc[r] = hidden ? 0.0f : pr;
            dp[r] = hidden ? 0.0f : g;
        }
        float* t = dsk + ((int64_t)j * (j + 1) / 2 + kg) * 1024;
#pragma unroll
        for(int r = 0; r < 16; ++r) t[acc_row(r, lh) * 32] = dp[r];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for(int r = 0; r < 16; ++r)
#pragma unroll
            for(int cb = 0; cb < NB; ++cb) {
                const int at = acc_row(r, lh) * LDT + cb * 32 + lq;
                dv[cb] = mfma(to[at], sc[r], dv[cb]);
                dk[cb] = mfma(tq[at], dp[r], dk[cb]);
            }
        read_ahead<32 * NB - 3, 1>();
        __builtin_amdgcn_sched_barrier(0);
    };
    const int steps = (nq - j0 + KS - 1) / KS;
    for(int it = 0; it < steps; ++it) {
        const int j = j0 + it * KS + ks, st = it & 1;
        wait_loads();
        __syncthreads();
        if(it + 1 < steps) issue(it + 1, st ^ 1);
        // (j < kg: every query of the block precedes this wave's keys)
        if(j >= kg && j < nq) block(j, sQ[st][ks], sO[st][ks], sC[st][ks]);
    }
    if constexpr(KS == 2) {
        __syncthreads();
        float* mine = &sQ[0][0][0] + rg * 16 * 64 + l;
        static_assert(RG * 16 * 64 <= 4 * Tl::FLOATS, "one accumulator of every row group fits");
#pragma unroll
        for(int cb = 0; cb < 2 * NB; ++cb) {
            f32x16& x = cb < NB ? dv[cb % NB] : dk[cb % NB];
            if(ks == 1) {
#pragma unroll
                for(int r = 0; r < 16; ++r) mine[r * 64] = x[r];
            }
            __syncthreads();
            if(ks == 0) {
#pragma unroll
                for(int r = 0; r < 16; ++r) x[r] += mine[r * 64];
            }
            __syncthreads();
        }
        if(ks == 1) return;
    }
    if(ki >= p.T) return;
    store_rowT<NB>(p.dv + base + ki * p.ld, dv, lh, 1.0f, (p.flags & PK_ACCUM3) != 0);
    store_rowT<NB>(p.dk + base + ki * p.ld, dk, lh, p.scale, (p.flags & PK_ACCUM2) != 0);
}

// dQ: one query per lane, dQ^T += K^T.dS^T over the stored dS tiles
template <int HDT, int RG, int KS>
__global__ __launch_bounds__(256, 2) void wide_bwd_dq(WideParams p) {
    using Tl = WideTile<HDT>;
    constexpr int NB = HDT / 32, LDT = Tl::LDT, ROWS = 32 * RG;
    __shared__ __attribute__((aligned(16))) float sK[2][KS][Tl::FLOATS];
    const int64_t BH = p.B * p.H, nqb = (p.Tp + ROWS - 1) / ROWS;
    const int64_t rank = place<true>(blockIdx.x, gridDim.x);
    const int64_t qb = nqb - 1 - rank / BH, bh = rank % BH, b = bh / p.H, h = bh % p.H;
    const int64_t base = b * p.T * p.ld + h * HDT;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = threadIdx.x & 63, lq = l & 31, lh = l >> 5;
    const int rg = w % RG, ks = w / RG;
    const int64_t q0 = qb * ROWS + rg * QB, qi = q0 + lq, qg = q0 / QB;
    const int steps = (int)((qb + 1) * RG / KS);
    const WideLoad<HDT, 4> blk(p.ld, w, l);
    const float* K = p.k + base;
    auto issue = [&](int it, int st) {
#pragma unroll
        for(int x = 0; x < KS; ++x)
            blk.issue(K, p.T, p.ld, (int64_t)(it * KS + x) * QB, sK[st][x], w);
    };
    issue(0, 0);
    // (a wave past Tp would read tiles past the triangle: it has none)
    const bool live = q0 < p.Tp;
    const float* ds = p.ds + (bh * ds_tiles(p.Tp) + qg * (qg + 1) / 2) * 1024 + (2 * lq + lh) * 16;
    auto fetch = [&](int64_t kg, f32x16& x) {
        const f32x4* src = reinterpret_cast<const f32x4*>(ds + kg * 1024);
#pragma unroll
        for(int i = 0; i < 4; ++i) {
            const f32x4 v = src[i];
#pragma unroll
            for(int e = 0; e < 4; ++e) x[4 * i + e] = v[e];
        }
    };
    f32x16 dq[NB];
#pragma unroll
    for(int cb = 0; cb < NB; ++cb) dq[cb] = splat16(0.0f);
    f32x16 cur = splat16(0.0f), nxt = splat16(0.0f);
    if(live && ks <= qg) fetch(ks, cur);
    auto block = [&](int j, const float* __restrict__ tk) {
        if(j + KS <= qg) fetch(j + KS, nxt);
#pragma unroll
        for(int r = 0; r < 16; ++r)
#pragma unroll
            for(int cb = 0; cb < NB; ++cb)
                dq[cb] = mfma(tk[acc_row(r, lh) * LDT + cb * 32 + lq], cur[r], dq[cb]);
        cur = nxt;
    };
    for(int it = 0; it < steps; ++it) {
        const int j = it * KS + ks;
        wait_loads();
        __syncthreads();
        if(it + 1 < steps) issue(it + 1, (it + 1) & 1);
        if(live && j <= qg) block(j, sK[it & 1][ks]);
    }
    if constexpr(KS == 2) {
        __syncthreads();
        float* mine = &sK[0][0][0] + rg * 16 * 64 + l;
        static_assert(RG * 16 * 64 <= 4 * Tl::FLOATS, "one accumulator of every row group fits");
#pragma unroll
        for(int cb = 0; cb < NB; ++cb) {
            if(ks == 1) {
#pragma unroll
                for(int r = 0; r < 16; ++r) mine[r * 64] = dq[cb][r];
            }
            __syncthreads();
            if(ks == 0) {
#pragma unroll
                for(int r = 0; r < 16; ++r) dq[cb][r] += mine[r * 64];
            }
            __syncthreads();
        }
        if(ks == 1) return;
    }
    if(qi >= p.T) return;
    store_rowT<NB>(p.dq + base + qi * p.ld, dq, lh, p.scale, (p.flags & PK_ACCUM) != 0);
}

// (hipcc leaves the launch stubs of these out unless they are instantiated by name)
#define WIDE_KERNELS(HDT, RG, KS)                                    \
    template __global__ void wide_fwd<HDT, RG, KS>(WideParams);      \
    template __global__ void wide_bwd_dkdv<HDT, RG, KS>(WideParams); \
    template __global__ void wide_bwd_dq<HDT, RG, KS>(WideParams);
WIDE_KERNELS(32, 2, 2)
WIDE_KERNELS(32, 4, 1)
WIDE_KERNELS(96, 2, 2)
WIDE_KERNELS(96, 4, 1)
WIDE_KERNELS(128, 2, 2)
WIDE_KERNELS(128, 4, 1)
#undef WIDE_KERNELS

int wide_check(const char* who, int64_t B, int64_t H, int64_t T, int64_t hd, int64_t ld,
               const void* a, const void* b, const void* c) {
    if(B < 0 || H < 1 || T < 0) return pk::fail("%s: bad sizes", who);
    if(!pk_flash_wide_supported(T > 0 ? T : 1, hd))
        return pk::fail("%s: head size %lld (these kernels handle 32, 96 and 128)", who, (long long)hd);
    if(ld < H * hd || ld % 4)
        return pk::fail("%s: row stride %lld of q, k, v must be >= %lld and a multiple of 4", who,
                        (long long)ld, (long long)(H * hd));
    if(!pk::aligned16(a) || !pk::aligned16(b) || !pk::aligned16(c))
        return pk::fail("%s: q, k, v must be 16-byte aligned", who);
    const int64_t Tp = (T + QB - 1) / QB * QB;
    if(B * H * (Tp / QB) > 0x7fffffff || (Tp + QB) * ld * 4 > 0x7fffffff)
        return pk::fail("%s: problem too large", who);
    return PK_OK;
}

// 128-row workgroups once they give every CU two
bool four_waves(int64_t B, int64_t H, int64_t T) { return B * H * ((T + 127) / 128) >= 2 * kCUs; }

template <int HDT, int RG, int KS>
int launch_fwd(const WideParams& p, hipStream_t st) {
    const unsigned grid = (unsigned)(p.B * p.H * ((p.Tp + 32 * RG - 1) / (32 * RG)));
    wide_fwd<HDT, RG, KS><<<grid, 256, 0, st>>>(p);
    return pk::launch_status("pk_flash_wide_fwd_f32");
}

template <int HDT, int RG, int KS>
int launch_bwd(const WideParams& p, hipStream_t st) {
    const unsigned grid = (unsigned)(p.B * p.H * ((p.Tp + 32 * RG - 1) / (32 * RG)));
    wide_consts<HDT><<<pk::grid_for(p.B * p.H * p.Tp * 32, 256), 256, 0, st>>>(p);
    int rc = pk::launch_status("pk_flash_wide_bwd_f32");
    if(rc) return rc;
    wide_bwd_dkdv<HDT, RG, KS><<<grid, 256, 0, st>>>(p);
    if((rc = pk::launch_status("pk_flash_wide_bwd_f32"))) return rc;
    wide_bwd_dq<HDT, RG, KS><<<grid, 256, 0, st>>>(p);
    return pk::launch_status("pk_flash_wide_bwd_f32");
}

}  // namespace

extern "C" int pk_flash_wide_supported(int64_t T, int64_t hd) {
    return T > 0 && (hd == 32 || hd == 96 || hd == 128);
}

extern "C" size_t pk_flash_wide_bwd_workspace(int64_t B, int64_t H, int64_t T) {
    if(B <= 0 || H <= 0 || T <= 0) return 0;
    const int64_t Tp = (T + QB - 1) / QB * QB;
    return (size_t)(2 * B * H * Tp + B * H * ds_tiles(Tp) * 1024) * sizeof(float);
}

extern "C" int pk_flash_wide_fwd_f32(int64_t B, int64_t H, int64_t T, int64_t hd, int64_t ld,
                                     float scale, const float* q, const float* k, const float* v,
                                     float* o, float* lse, pk_stream_t stream) {
    const char* who = "pk_flash_wide_fwd_f32";
    int rc = wide_check(who, B, H, T, hd, ld, q, k, v);
    if(rc) return rc;
    if(B == 0 || T == 0) return PK_OK;
    if(!q || !k || !v || !o || !pk::aligned16(o)) return pk::fail("%s: NULL or unaligned pointer", who);
    WideParams p = {};
    p.q = q;
    p.k = k;
    p.v = v;
    p.out = o;
    p.lse_out = lse;
    p.B = B;
    p.H = H;
    p.T = T;
    p.Tp = (T + QB - 1) / QB * QB;
    p.D = H * hd;
    p.ld = ld;
    p.scale = scale;
    hipStream_t st = pk::as_stream(stream);
    const bool four = four_waves(B, H, T);
    if(hd == 32) return four ? launch_fwd<32, 4, 1>(p, st) : launch_fwd<32, 2, 2>(p, st);
    if(hd == 96) return four ? launch_fwd<96, 4, 1>(p, st) : launch_fwd<96, 2, 2>(p, st);
    return four ? launch_fwd<128, 4, 1>(p, st) : launch_fwd<128, 2, 2>(p, st);
}

extern "C" int pk_flash_wide_bwd_f32(int64_t B, int64_t H, int64_t T, int64_t hd, int64_t ld,
                                     float scale, const float* q, const float* k, const float* v,
                                     const float* o, const float* lse, const float* dout, float* dq,
                                     float* dk, float* dv, void* workspace, size_t workspace_bytes,
                                     int flags, pk_stream_t stream) {
    const char* who = "pk_flash_wide_bwd_f32";
    int rc = wide_check(who, B, H, T, hd, ld, q, k, v);
    if(rc) return rc;
    if(B == 0 || T == 0) return PK_OK;
    if(!q || !k || !v || !o || !lse || !dout || !dq || !dk || !dv) return pk::fail("%s: NULL pointer", who);
    if(!pk::aligned16(o) || !pk::aligned16(dout) || !pk::aligned16(dq) || !pk::aligned16(dk) ||
       !pk::aligned16(dv))
        return pk::fail("%s: o, dout, dq, dk, dv must be 16-byte aligned", who);
    const size_t need = pk_flash_wide_bwd_workspace(B, H, T);
    if(!workspace || workspace_bytes < need || !pk::aligned16(workspace))
        return pk::fail("%s: needs a 16-byte aligned workspace of %zu bytes", who, need);
    WideParams p = {};
    p.q = q;
    p.k = k;
    p.v = v;
    p.o = o;
    p.lse = lse;
    p.dout = dout;
    p.dq = dq;
    p.dk = dk;
    p.dv = dv;
    p.B = B;
    p.H = H;
    p.T = T;
    p.Tp = (T + QB - 1) / QB * QB;
    p.consts = static_cast<float*>(workspace);
    p.ds = p.consts + 2 * B * H * p.Tp;
    p.D = H * hd;
    p.ld = ld;
    p.scale = scale;
    p.flags = flags & (PK_ACCUM | PK_ACCUM2 | PK_ACCUM3);
    hipStream_t st = pk::as_stream(stream);
    const bool four = four_waves(B, H, T);
    if(hd == 32) return four ? launch_bwd<32, 4, 1>(p, st) : launch_bwd<32, 2, 2>(p, st);
    if(hd == 96) return four ? launch_bwd<96, 4, 1>(p, st) : launch_bwd<96, 2, 2>(p, st);
    return four ? launch_bwd<128, 4, 1>(p, st) : launch_bwd<128, 2, 2>(p, st);
}
