// pico_amd/csrc/gemm_common.h -- what the GEMM kernels share: the launch
// parameters, a workgroup's tile and K range, and the epilogues.
#pragma once

#include "pk_common.h"

namespace pkg {

constexpr int BK = 32, NT = 256;
constexpr int GROUP_M = 8;

struct GemmParams {
    const float* A;
    const float* B;
    float* C;
    int64_t M, N, K, lda, ldb, ldc;
    int64_t sAo, sAi, sBo, sBi, sCo, sCi, inner;
    float alpha, beta;
    int causal;
    int tiles_m, tiles_n;
    int splits;      // > 1: blockIdx.y is a K slice of kchunk, partials go to ws
    int64_t kchunk;
    float* ws;
    // the beta term's source: C itself, or another matrix (batch 1 only)
    const float* Cin;
    int64_t ldcin;
    // SwiGLU-backward epilogue (sg_a non-null, batch 1, no K split): the
    // product is the upstream gradient dh of h = silu(a) * u and is not
    // stored; the tile writes da (+)= dh*u*s*(1 + a*(1-s)) and du (+)= dh*a*s
    // (s = sigmoid(a)), accumulating per sg_flags bit 0 (da) and bit 1 (du)
    const float *sg_a, *sg_u;
    float *sg_da, *sg_du;
    int64_t sg_lda, sg_ldu, sg_ldd;
    int sg_flags;
    // the staged epilogue may use float4 accesses: every matrix it touches is
    // 16-byte aligned with a row stride that is a multiple of 4
    int epi_vec;
    // fp8 products: the device address of the two operand scales (NULL: 1, 1)
    const float* fp8_scale;
    // SwiGLU-forward epilogue (pair_F > 0, 'N','N', batch 1, no K split): C is
    // [gate | up], N = 2 pair_F columns.  A tile takes BN/2 gate columns and
    // the BN/2 up columns pair_F to their right, so it holds matching pairs;
    // it writes both to C and h = silu(gate) * up to sf_h
    int64_t pair_F;
    float* sf_h;
    int64_t sf_ldh;
    // 1: an operand's rows are too far apart for buffer offsets, so tiles (64x64
    // ones only) load with 64-bit addresses
    int far;
};

// Bounds handling of a tile's loads and stores: none (whole tiles), per float4
// (M, N, K, the leading dimensions and batch strides multiples of 4, 16-byte
// aligned operands: a float4 is wholly inside or wholly outside), or per element.
constexpr int kEdgeNone = 0, kEdgeVec = 1, kEdgeScalar = 2;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// One workgroup's job: its tile, operand bases, output, K range.
struct TileJob {
    const float* A;
    const float* B;
    float* C;
    const float* Cin;
    int64_t ldc, ldcin, row0, col0, kbeg, kend;
    float alpha, beta;
    int nslices;
    bool skip;
};

template <class T>
__device__ __forceinline__ TileJob tile_job(const GemmParams& p) {
    TileJob j;
    // tile selection: XCD-contiguous runs, grouped by GROUP_M tile-rows
    const int ntiles = p.tiles_m * p.tiles_n;
    int bid = blockIdx.x;
    if((ntiles & 7) == 0) bid = (bid & 7) * (ntiles >> 3) + (bid >> 3);
    const int group_span = GROUP_M * p.tiles_n;
    const int first_m = (bid / group_span) * GROUP_M;
    const int gm = min(p.tiles_m - first_m, GROUP_M);
    const int local = bid % group_span;
    const int tm = first_m + local % gm;
    const int tn = local / gm;

    // blockIdx.y is the batch index, or the K slice of a split product
    const int64_t z = p.splits > 1 ? 0 : blockIdx.y;
    const int64_t zo = z / p.inner, zi = z % p.inner;
    j.A = p.A + zo * p.sAo + zi * p.sAi;
    j.B = p.B + zo * p.sBo + zi * p.sBi;
    j.C = p.C + zo * p.sCo + zi * p.sCi;
    j.ldc = p.ldc;
    j.Cin = p.Cin ? p.Cin : j.C;
    j.ldcin = p.Cin ? p.ldcin : p.ldc;
    j.alpha = p.alpha;
    j.beta = p.beta;

    j.row0 = (int64_t)tm * T::BM;
    j.col0 = (int64_t)tn * (p.pair_F ? T::BN / 2 : T::BN);
    j.kbeg = 0;
    j.kend = p.K;
    j.skip = p.causal == 1 && j.col0 > j.row0 + T::BM - 1;  // wholly above the diagonal
    if(p.causal == 2) j.kend = min(p.K, j.row0 + T::BM);
    if(p.causal == 3) j.kbeg = min(p.K, (j.row0 / BK) * BK);
    if(p.splits > 1) {
        // slice s of K; its partial product goes to workspace plane s
        j.kbeg = (int64_t)blockIdx.y * p.kchunk;
        j.kend = min(p.K, j.kbeg + p.kchunk);
        j.C = p.ws + (int64_t)blockIdx.y * p.M * p.N;
        j.ldc = p.N;
        j.Cin = j.C;
        j.ldcin = p.N;
        j.alpha = 1.0f;
        j.beta = 0.0f;
    }
    j.nslices = (int)((j.kend - j.kbeg + BK - 1) / BK);
    return j;
}

// C block = alpha * acc (+ beta * C).  32x32 block accumulator r of lane l is
// row 8*(r/4) + 4*(l/32) + r%4, column l%32: each half-wave writes 128
// contiguous bytes per register.
template <int EDGE, bool NT_STORE>
__device__ __forceinline__ void store_block(const GemmParams& p, const TileJob& j, const f32x16& acc,
                                            int ar, int br, int lr, int lh) {
    const int64_t col = j.col0 + br + lr;
#pragma unroll
    for(int r = 0; r < 16; ++r) {
        const int64_t row = j.row0 + ar + (r >> 2) * 8 + lh * 4 + (r & 3);
        if(EDGE != kEdgeNone && (row >= p.M || col >= p.N)) continue;
        float v = j.alpha * acc[r];
        float* c = j.C + row * j.ldc + col;
        if(j.beta != 0.0f) v += j.beta * *c;
        // 64x64 tiles (products of about 1024^2 outputs, where the
        // launch's end is a large share of its time) store C
        // non-temporally: 1024^3 1.1-1.6 % and 768^3 0.6-1.1 % faster,
        // config-4 and config-5 steps unchanged (same box, alternating);
        // for every tile they cost a config-5 step 0.05 ms
        if constexpr(NT_STORE) __builtin_nontemporal_store(v, c);
        else *c = v;
    }
}

// The tile's blocks but those of the bits of `skip`.
// G > 1: of the tile's blocks, the K group g stores those it finished.
template <int EDGE, int TM, int TN, int G = 1>
__device__ __forceinline__ void store_tile(const GemmParams& p, const TileJob& j,
                                           const f32x16 (&acc)[TM][TN], int ar0, int br0, int lr,
                                           int lh, int g = 0, unsigned skip = 0) {
#pragma unroll
    for(int b = 0; b < TM * TN; ++b) {
        if((G > 1 && b % G != g) || (skip >> b & 1)) continue;
        store_block<EDGE, TM * TN == 1>(p, j, acc[b / TN][b % TN], ar0 + b / TN * 32,
                                        br0 + b % TN * 32, lr, lh);
    }
}

// Epilogues that read other matrices: the tile goes through LDS (free once
// the main loop is done) in passes of RP rows, and all its threads then walk
// the staged rows in float4 runs, so every global access is a coalesced
// 128-bit one and no per-element loads wait inside the accumulator loops
// (which, in the 256x256 tile, also pushed the accumulators out of
// registers).
//   kEpiAdd:    C = alpha * acc + beta * Cin
//   kEpiSwiglu: dh = alpha * acc; da (+)= dh*u*s*(1 + a*(1-s)), du (+)= dh*a*s
//   kEpiSwigluFwd: the tile's two column halves are matching gate and up
//               columns: C gets g = alpha * acc and u alike (as the plain
//               store writes them), sf_h gets silu(g) * u
constexpr int kEpiPlain = 0, kEpiAdd = 1, kEpiSwiglu = 2, kEpiSwigluFwd = 3;

template <int EPI>
__device__ __forceinline__ void epi_one(const GemmParams& p, const TileJob& j, int64_t row,
                                        int64_t col, float x) {
    if constexpr(EPI == kEpiAdd) {
        float v = j.alpha * x;
        if(j.beta != 0.0f) v += j.beta * j.Cin[row * j.ldcin + col];
        j.C[row * j.ldc + col] = v;
    } else {
        float ga, gu;
        pk::swiglu_bwd1(p.sg_a[row * p.sg_lda + col], p.sg_u[row * p.sg_ldu + col], j.alpha * x,
                        ga, gu);
        float* da = p.sg_da + row * p.sg_ldd + col;
        float* du = p.sg_du + row * p.sg_ldd + col;
        if(p.sg_flags & PK_ACCUM) ga = pk::add_nc(*da, ga);
        if(p.sg_flags & PK_ACCUM2) gu = pk::add_nc(*du, gu);
        *da = ga;
        *du = gu;
    }
}

template <int EPI>
__device__ __forceinline__ void epi_four(const GemmParams& p, const TileJob& j, int64_t row,
                                         int64_t col, f32x4 x) {
    if constexpr(EPI == kEpiAdd) {
        f32x4 v;
#pragma unroll
        for(int e = 0; e < 4; ++e) v[e] = j.alpha * x[e];
        if(j.beta != 0.0f) {
            const f32x4 c = *reinterpret_cast<const f32x4*>(j.Cin + row * j.ldcin + col);
#pragma unroll
            for(int e = 0; e < 4; ++e) v[e] += j.beta * c[e];
        }
        *reinterpret_cast<f32x4*>(j.C + row * j.ldc + col) = v;
    } else {
        const f32x4 a = *reinterpret_cast<const f32x4*>(p.sg_a + row * p.sg_lda + col);
        const f32x4 u = *reinterpret_cast<const f32x4*>(p.sg_u + row * p.sg_ldu + col);
        f32x4* dap = reinterpret_cast<f32x4*>(p.sg_da + row * p.sg_ldd + col);
        f32x4* dup = reinterpret_cast<f32x4*>(p.sg_du + row * p.sg_ldd + col);
        f32x4 pa = {0.f, 0.f, 0.f, 0.f}, pu = {0.f, 0.f, 0.f, 0.f};
        if(p.sg_flags & PK_ACCUM) pa = *dap;
        if(p.sg_flags & PK_ACCUM2) pu = *dup;
        f32x4 ga, gu;
#pragma unroll
        for(int e = 0; e < 4; ++e) {
            float y, z;
            pk::swiglu_bwd1(a[e], u[e], j.alpha * x[e], y, z);
            ga[e] = (p.sg_flags & PK_ACCUM) ? pk::add_nc(pa[e], y) : y;
            gu[e] = (p.sg_flags & PK_ACCUM2) ? pk::add_nc(pu[e], z) : z;
        }
        *dap = ga;
        *dup = gu;
    }
}

// Blocks of the bits of `skip` come from block(index) instead of acc.
struct NoBlock {
    __device__ f32x16 operator()(int) const { return f32x16{}; }
};

template <int EPI, class T, int LDS_FLOATS, class Block = NoBlock>
__device__ __forceinline__ void staged_epilogue(const GemmParams& p, const TileJob& j,
                                                const f32x16 (&acc)[T::TM][T::TN], float* lds,
                                                int ar0, int br0, int lr, int lh, int g = 0,
                                                unsigned skip = 0, const Block& block = Block()) {
    constexpr int BN = T::BN, LDE = BN + 4, TM = T::TM, TN = T::TN, NTHR = T::THREADS;
    // rows per pass: whole 32-row blocks that fit in the operand buffers
    constexpr int rp = (LDS_FLOATS / LDE) / 32 * 32 < T::BM ? (LDS_FLOATS / LDE) / 32 * 32 : T::BM;
    static_assert(rp >= 32, "the staging buffer must hold at least one 32-row block");
    __syncthreads();  // every wave is done reading the operand tiles
    auto put = [&](const f32x16& x, int row, int col) {
#pragma unroll
        for(int r = 0; r < 16; ++r)
            lds[(row + (r >> 2) * 8 + lh * 4 + (r & 3)) * LDE + col + lr] = x[r];
    };
    for(int lo = 0; lo < T::BM; lo += rp) {
#pragma unroll
        for(int i = 0; i < TM; ++i) {
            const int rb = ar0 + i * 32;
            if(rb < lo || rb >= lo + rp) continue;
#pragma unroll
            for(int jj = 0; jj < TN; ++jj) {
                if((T::G > 1 && (i * TN + jj) % T::G != g) || (skip >> (i * TN + jj) & 1)) continue;
                put(acc[i][jj], rb - lo, br0 + jj * 32);
            }
        }
        for(unsigned left = skip; left; left &= left - 1) {
            const int b = __builtin_ctz(left), rb = ar0 + b / TN * 32;
            if(rb >= lo && rb < lo + rp) put(block(b), rb - lo, br0 + b % TN * 32);
        }
        __syncthreads();
        const int rows = rp < T::BM - lo ? rp : T::BM - lo;
        if constexpr(EPI == kEpiSwigluFwd) {
            // column c of the gate half pairs with column BN/2 + c; pair_F is a
            // multiple of 4, so a float4 is wholly inside or outside
            constexpr int HB = BN / 2;
            for(int idx = threadIdx.x; idx < rows * (HB / 4); idx += NTHR) {
                const int rr = idx / (HB / 4), c = (idx % (HB / 4)) * 4;
                const int64_t row = j.row0 + lo + rr, col = j.col0 + c;
                if(row >= p.M || col >= p.pair_F) continue;
                const f32x4 g4 = *reinterpret_cast<const f32x4*>(lds + rr * LDE + c);
                const f32x4 u = *reinterpret_cast<const f32x4*>(lds + rr * LDE + HB + c);
                f32x4 gv, uv, hv;
#pragma unroll
                for(int e = 0; e < 4; ++e) {
                    gv[e] = j.alpha * g4[e];
                    uv[e] = j.alpha * u[e];
                    hv[e] = pk::swiglu_fwd1(gv[e], uv[e]);
                }
                float* cg = j.C + row * j.ldc + col;
                float* hp = p.sf_h + row * p.sf_ldh + col;
                if(p.epi_vec) {
                    *reinterpret_cast<f32x4*>(cg) = gv;
                    *reinterpret_cast<f32x4*>(cg + p.pair_F) = uv;
                    *reinterpret_cast<f32x4*>(hp) = hv;
                } else {
#pragma unroll
                    for(int e = 0; e < 4; ++e) {
                        cg[e] = gv[e];
                        cg[p.pair_F + e] = uv[e];
                        hp[e] = hv[e];
                    }
                }
            }
        } else {
            for(int idx = threadIdx.x; idx < rows * (BN / 4); idx += NTHR) {
                const int rr = idx / (BN / 4), c = (idx % (BN / 4)) * 4;
                const int64_t row = j.row0 + lo + rr, col = j.col0 + c;
                const f32x4 x = *reinterpret_cast<const f32x4*>(lds + rr * LDE + c);
                if(row >= p.M) continue;
                if(p.epi_vec && col + 3 < p.N) {
                    epi_four<EPI>(p, j, row, col, x);
                } else {
#pragma unroll
                    for(int e = 0; e < 4; ++e)
                        if(col + e < p.N) epi_one<EPI>(p, j, row, col + e, x[e]);
                }
            }
        }
        __syncthreads();
    }
}

// (128x96 tiles: not for fp32; 128x64 and 64x64 tiles of two and one wave groups:
// fp32 only)
enum TileKind { kTile128, kTile96, kTile256, kTile64, kTile256x96, kTile128x64, kTile64x2, kTile64x1 };

// the fp32 product (gemm_split.hip): K groups a shape's workgroups split K into,
// and the launch; with gp.far, kTile64x2 only
int split_groups(TileKind kind);
int launch_split(bool ta, bool tb, const GemmParams& gp, int64_t batch, bool edge, TileKind kind,
                 hipStream_t st);

// the bf16 (parts 1) and split-bf16 (parts 2) products (gemm_narrow.hip); with
// gp.far, 64x64 tiles only
int launch_narrow(bool ta, bool tb, int parts, const GemmParams& gp, int64_t batch, bool edge,
                  TileKind kind, hipStream_t st);

}  // namespace pkg
