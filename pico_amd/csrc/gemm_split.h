// pico_amd/csrc/gemm_split.h -- the fp32 product on the bf16 matrix cores.
// Included inside the anonymous namespace of gemm_split.hip, which launches it,
// and of gemm_narrow.hip, whose kernel shares the staging.
//
// The fp32 matrix cores are 16 times slower than the bf16 ones, and a SIMD's
// vector instructions do not overlap fp32 matrix instructions while they do
// overlap bf16 ones (up to about six per 32x32x16 instruction, measured with
// independent streams of both).  So an fp32 operand is taken as the exact sum
// of three bf16 parts, x = h + m + l (8 significant bits each, rounded to
// nearest, 24 in all), on its way to LDS, and
//     a.b = hh + hm + mh + mm + hl + lh
// in six matrix instructions per 16 k; ml, lm and ll, together below 2^-24 of
// |a||b|, are left out (below 0.87 2^-24 of one product at the worst).  Nothing is
// held in less than fp32's 24 bits, and the sums are fp32.  Against float64,
// relative 2-norm on random operands, the error is below that of the fp32 matrix
// instructions (which round after every k) from K 4 on: normal operands, K 4 / 32 /
// 768 / 2048 / 4096 3.2e-8 / 4.2e-8 / 2.9e-7 / 6.9e-7 / 9.7e-7 against 4.0e-8 /
// 1.03e-7 / 5.0e-7 / 8.1e-7 / 1.15e-6.  Products of one and two k, whose few
// roundings they do better (2.5e-8 against 3.5e-8, 3.1e-8 against 3.4e-8), run
// on the fp32 cores (exact_block).  Half-zero operands (a relu's output) leave the
// fp32 cores half as many roundings: there 256x256 tiles, which have one sum to a
// block, are up to 14 % above them (6.5e-7 against 5.7e-7 at K 2048), the others below.
//  * Range: operands are scaled by 2^16, so that the parts of every normal and
//    subnormal fp32 number are exact bf16 numbers (l of a 2^-126 would need
//    2^-149), and the sums by 2^-32 at the end.  What overflows (values above
//    2^111, sums above 2^96, infinities) or is NaN leaves a non-finite sum: a
//    wave that sees one computes that 32x32 block again on the fp32 cores, from
//    global memory (exact_block).
//  * Sign: the matrix unit drops the low bits of products much smaller than the
//    accumulator towards minus infinity.  One sum loses less than its
//    roundings, but the loss has the same sign in every output, so it would
//    add up in a sum over outputs (a bias gradient, an attention average:
//    the mean error of [8192, 2304] outputs with K 768 was 2e-6 of the value
//    in such a sum).  So the parts of op(A) change sign with the sums every
//    128 k (K group by K group, or set by set, where a workgroup splits K), and
//    the loss cancels: mean error below 3e-9 of the root mean square from K 128 on.
//    Before the first turn (one slice of 16, 64 k in 256x256 tiles) nothing
//    cancels, up to 1.2e-8, and outputs of one sign keep some of it: probabilities
//    times values around 1 2e-8 to 4e-8 of the value (the fp32 instructions 2e-9
//    at K 128, 2e-8 at K 512).
//  * Bound: 6 instructions of 32 cycles per 32x32 block and 16 k, 2.5 PFLOP/s /
//    6 = 417 TFLOP/s at the nominal clock; the card settles near 2.06 GHz under
//    bf16 matrix load (358).  The split costs 6.5 vector instructions per staged
//    value, 1.1-4.6 per matrix instruction depending on the tile.  Splitting
//    when the fragments are read instead would stage 4 bytes a value, but each
//    value is read by several waves.
//  * Tiles: at least two waves per SIMD, so that one wave's staging and LDS
//    latency hides under the other's matrix work; where a tile has only four
//    waves, G groups of them take every G-th slice of K into LDS buffers of
//    their own and add their sums at the end (256x96: 166 -> 197 TFLOP/s at
//    [8192, 768] K 2304; 64x64 with G 4: 84 -> 114 at 1024^3).
//    64x64 tiles of short K have two groups or one, each with several sets of
//    sums: the same four sums, bit for bit, without a thousand threads' start and
//    the groups' meeting (256 tiles, us, G 4 / 2 / 1: K 32 9.6 / 7.2 / 5.3, K 256 9.4 /
//    9.0 / 10.3, K 512 12.8 / 13.1 / 16.1).
//  * A slice is 16 k.  Its first half multiplies m.m, m.h, h.m while l is read,
//    the next slice is split and stored and the slice after it fetched; one
//    barrier; then h.l, l.h, h.h while the next slice's m and h are read into
//    the fragments that are free by then.
//  * Loads go through buffer resources that end where the operand ends, 128 bits
//    at any 4-byte alignment, so ragged sizes take the same path: what lies
//    behind the end reads as zero, and only a partial last slice is masked.
//    (The per-element edge path this replaces ran 2000x1503x1001, forward and
//    backward, at 59 TFLOP/s; now 118-127.)
//
// TFLOP/s of A.B, A.B^T and A^T.B by card and box: 4096^3 223-250 (149 on the fp32
// cores), 8192^3 222-243 (151), 2048^3 174-197 (142), 1024^3 100-118 (98-115).

// A tile shape: WM x WN waves, each TM x TN blocks of 32 x 32; WPS waves per SIMD;
// G groups of them, each with A sets of sums (slice s of K goes to group s % G and
// there to set s / G % A).
template <int WM_, int WN_, int TM_, int TN_, int G_, int WPS_, int PF_, int A_ = 1>
struct SplitTile {
    static constexpr int WGM = WM_, WGN = WN_, TM = TM_, TN = TN_, G = G_, A = A_;
    static_assert(A_ == 1 || (TM_ * TN_ == 1 && PF_ == 1), "one block to a wave");
    static constexpr int WPS = WPS_, PF = PF_;
    static constexpr int BM = WM_ * TM_ * 32, BN = WN_ * TN_ * 32;
    static constexpr int WAVES = WM_ * WN_;                    // of one K group
    static constexpr int GTHREADS = 64 * WAVES, THREADS = GTHREADS * G_;
};

constexpr int SK = 16;  // k per slice: one v_mfma_f32_32x32x16_bf16 step

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));

// One operand's R x W slice as staged by THREADS threads: items of KPI
// consecutive k of one row, ITEMS per thread (threads past the last item
// repeat an earlier one).
template <bool KFAST, int R, int THREADS, int W = SK>
struct SplitOperand {
    static constexpr int KPI = KFAST ? 4 : (R * W / 8 >= THREADS ? 8 : 4);
    static constexpr int COUNT = R * W / KPI;
    static constexpr int ITEMS = (COUNT + THREADS - 1) / THREADS;
    static constexpr int LOADS = KFAST ? 1 : KPI;

    static __device__ __forceinline__ void origin(int item, int& rr, int& kk) {
        int u = threadIdx.x % THREADS + item * THREADS;
        if(ITEMS * THREADS != COUNT) u %= COUNT;
        if(KFAST) {
            rr = u / (W / 4);
            kk = u % (W / 4) * 4;
        } else {
            rr = u % R;
            kk = (u / R) * KPI;
        }
    }
};

// The operand as buffer loads see it: bytes from `base` to its end.
struct SplitSource {
    const char* base;  // element (first row of the tile, k 0)
    int64_t left;      // bytes from base to the end of the operand
    int64_t kstep;     // bytes per k
};

template <bool KFAST, bool EDGE, int R, int THREADS, bool PAIR, int W = SK>
__device__ __forceinline__ void split_load(const SplitSource& src, int64_t ld, int64_t k0,
                                           int64_t shift,
                                           float (&v)[SplitOperand<KFAST, R, THREADS, W>::ITEMS]
                                                     [SplitOperand<KFAST, R, THREADS, W>::KPI]) {
    using O = SplitOperand<KFAST, R, THREADS, W>;
    const int64_t off = k0 * src.kstep;
    const int64_t left = src.left - off;
    // the operand from the slice's k row t on.  Only slices of 32 k ask for more than
    // the first: their size stops at 2^31 - 1, which no offset of theirs reaches,
    // so that taking k rows off it stays a 32-bit subtraction
    auto rest = [&](int t) {
        const int skip = W == SK ? 0 : t * (int)src.kstep;
        int num = (int)0xfffffff0u;
        if(EDGE && W == SK)
            num = (int)(left <= 0 ? 0u : left > 0xfffffff0ll ? 0xfffffff0u : (unsigned)left);
        else if(EDGE)
            num = max((int)min(max(left, (int64_t)0), (int64_t)INT32_MAX) - skip, 0);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(src.base + off + skip), (short)0,
                                                 num, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rs = rest(0);
#pragma unroll
    for(int i = 0; i < O::ITEMS; ++i) {
        int rr, kk;
        O::origin(i, rr, kk);
        const unsigned row = (unsigned)rr + (PAIR && rr >= R / 2 ? (unsigned)shift : 0u);
        if(KFAST) {
            const int voff = (int)((row * (unsigned)ld + kk) * 4u);
            const f32x4 x =
                __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, 0, 0));
#pragma unroll
            for(int t = 0; t < 4; ++t) v[i][t] = x[t];
        } else {
            // whole tiles reach their k rows by the scalar offset; bounded loads do
            // not, as only the vector offset is sure to be checked.  Slices of 16 k
            // add it up anew each time (kept over the loop, the offsets spill in
            // 256-row tiles), those of 32 k, with no vector register to spare and
            // few bounded slices, take a resource per k row (which would spill
            // scalar registers in the other)
            unsigned voff = (kk * (unsigned)ld + row) * 4u;
            const unsigned step = (unsigned)ld * 4u;
            if(EDGE && W == SK) asm volatile("" : "+v"(voff));
#pragma unroll
            for(int t = 0; t < O::KPI; ++t) {
                int x;
                if(!EDGE)
                    x = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)voff, (int)(t * step), 0);
                else if(W == SK)
                    x = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)(voff + t * step), 0, 0);
                else
                    x = __builtin_amdgcn_raw_buffer_load_b32(rest(t), (int)voff, 0, 0);
                v[i][t] = __builtin_bit_cast(float, x);
            }
        }
    }
}

// How a tile's operands are read: buffer loads without bounds (whole tiles), bounded
// by the operand's end, or with 64-bit addresses (leading dimensions beyond the
// reach of buffer offsets)
constexpr int kWhole = 0, kPartial = 1, kFar = 2;

// the slice at k0 of rows row0.., zeros past `rows` and kend
template <bool KFAST, int R, int THREADS, bool PAIR, int W>
__device__ __forceinline__ void far_load(const float* x, int64_t ld, int64_t row0, int64_t rows,
                                         int64_t k0, int64_t kend, int64_t shift,
                                         float (&v)[SplitOperand<KFAST, R, THREADS, W>::ITEMS]
                                                   [SplitOperand<KFAST, R, THREADS, W>::KPI]) {
    using O = SplitOperand<KFAST, R, THREADS, W>;
    typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for(int i = 0; i < O::ITEMS; ++i) {
        int rr, kk;
        O::origin(i, rr, kk);
        const int64_t row = row0 + rr + (PAIR && rr >= R / 2 ? shift : 0), k = k0 + kk;
        const float* q = x + (KFAST ? row * ld + k : k * ld + row);
        if(KFAST && row < rows && k + 3 < kend) {
            const f32x4 y = *reinterpret_cast<const f32x4u*>(q);
#pragma unroll
            for(int t = 0; t < 4; ++t) v[i][t] = y[t];
            continue;
        }
#pragma unroll
        for(int t = 0; t < O::KPI; ++t)
            v[i][t] = row < rows && k + t < kend ? q[KFAST ? t : t * ld] : 0.0f;
    }
}

// zero the values at k >= limit (limit < W: the last, partial slice)
template <bool KFAST, int R, int THREADS, int W = SK>
__device__ __forceinline__ void split_mask(int limit,
                                           float (&v)[SplitOperand<KFAST, R, THREADS, W>::ITEMS]
                                                     [SplitOperand<KFAST, R, THREADS, W>::KPI]) {
    using O = SplitOperand<KFAST, R, THREADS, W>;
#pragma unroll
    for(int i = 0; i < O::ITEMS; ++i) {
        int rr, kk;
        O::origin(i, rr, kk);
#pragma unroll
        for(int t = 0; t < O::KPI; ++t) v[i][t] = kk + t < limit ? v[i][t] : 0.0f;
    }
}

// two values as three bf16 pairs: x * scale = h + m + l exactly (scale a power of two)
__device__ __forceinline__ void split3(float x0, float x1, float scale, int& h, int& m, int& l) {
    const f32x2 x = {x0 * scale, x1 * scale};
    const bf16x2 hv = __builtin_convertvector(x, bf16x2);
    const f32x2 r = {x[0] - (float)hv[0], x[1] - (float)hv[1]};
    const bf16x2 mv = __builtin_convertvector(r, bf16x2);
    const f32x2 q = {r[0] - (float)mv[0], r[1] - (float)mv[1]};
    const bf16x2 lv = __builtin_convertvector(q, bf16x2);
    h = __builtin_bit_cast(int, hv);
    m = __builtin_bit_cast(int, mv);
    l = __builtin_bit_cast(int, lv);
}

// LDS: [part][row][16 k], rows of 32 bytes whose two 16-byte halves swap places
// every 4 rows.  8 rows 32 bytes apart then fall in distinct banks, but rows r and
// r + 8 share theirs: 3.8e7 conflict cycles over 1.3e7 LDS instructions at 4096^3, 72 a
// wave and slice or 4 to a fragment read, in every layout.  Under 256x256 tiles'
// matrix instructions that is hidden; in the small tiles the reads take as long
// as those.  Offset in 16-bit elements of (row, k):
__device__ __forceinline__ int split_off(int row, int k) {
    return row * SK + ((((k >> 3) ^ (row >> 2)) & 1) << 3) + (k & 7);
}

// P parts of every value into [k / 16][part][row][16]: 3 as above, 2 hi and lo
// (lo = bf16(x - hi)), 1 rounded to bf16
template <int P, bool KFAST, int R, int THREADS, int PART, int W = SK>
__device__ __forceinline__ void split_store(short* lds,
                                            const float (&v)[SplitOperand<KFAST, R, THREADS, W>::ITEMS]
                                                            [SplitOperand<KFAST, R, THREADS, W>::KPI],
                                            float scale) {
    using O = SplitOperand<KFAST, R, THREADS, W>;
#pragma unroll
    for(int i = 0; i < O::ITEMS; ++i) {
        int rr, kk;
        O::origin(i, rr, kk);
        const int off = split_off(rr, kk % SK) + kk / SK * (P * PART);
        int w[3][O::KPI / 2];
#pragma unroll
        for(int t = 0; t < O::KPI / 2; ++t) {
            if constexpr(P == 3) {
                split3(v[i][2 * t], v[i][2 * t + 1], scale, w[0][t], w[1][t], w[2][t]);
            } else {
                const f32x2 x = {v[i][2 * t], v[i][2 * t + 1]};
                const bf16x2 h = __builtin_convertvector(x, bf16x2);
                w[0][t] = __builtin_bit_cast(int, h);
                if constexpr(P == 2) {
                    const f32x2 r = {x[0] - (float)h[0], x[1] - (float)h[1]};
                    w[1][t] = __builtin_bit_cast(int, __builtin_convertvector(r, bf16x2));
                }
            }
        }
#pragma unroll
        for(int q = 0; q < P; ++q) {
            if constexpr(O::KPI == 8)
                *reinterpret_cast<i32x4*>(lds + q * PART + off) =
                    i32x4{w[q][0], w[q][1], w[q][2], w[q][3]};
            else
                *reinterpret_cast<i32x2*>(lds + q * PART + off) = i32x2{w[q][0], w[q][1]};
        }
    }
}

template <int TM, int TN>
struct SplitFrag {
    bf16x8 a[TM], b[TN];
};

// one 32x32 block again on the fp32 matrix cores, from global memory with 64-bit
// addresses: for blocks whose split sums are not finite.  8 k at a time (lanes
// 0-31 take four of them, lanes 32-63 the others), D such steps in flight.  An
// infinity in one row of 4096^3 costs 813-843 us in all (1060 with one step in
// flight; the whole tile again 1340-1865; fp32 cores throughout 915), one in every
// row 2000-2600 (bound by the loads, which only one block shares)
template <bool KFAST>
__device__ __forceinline__ void exact_load(const float* x, int64_t ld, float (&f)[4]) {
    typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
    if constexpr(KFAST) {
        const f32x4 y = *reinterpret_cast<const f32x4u*>(x);
#pragma unroll
        for(int e = 0; e < 4; ++e) f[e] = y[e];
    } else {
#pragma unroll
        for(int e = 0; e < 4; ++e) f[e] = x[e * ld];
    }
}

template <bool TA, bool TB, bool PAIR, class T, int D>
__device__ __forceinline__ f32x16 exact_block(const GemmParams& p, const TileJob& j, int ar, int br,
                                              int lr, int lh) {
    const int64_t m = min(j.row0 + ar + lr, p.M - 1);
    const int c = br + lr;
    const int64_t n = min(j.col0 + c + (PAIR && c >= T::BN / 2 ? p.pair_F - T::BN / 2 : 0), p.N - 1);
    const int64_t sa = TA ? p.lda : 1, sb = TB ? 1 : p.ldb;
    const float* const a = j.A + (TA ? m : m * p.lda) + (j.kbeg + 4 * lh) * sa;
    const float* const b = j.B + (TB ? n * p.ldb : n) + (j.kbeg + 4 * lh) * sb;
    const int64_t klen = j.kend - j.kbeg;
    const int64_t whole = klen / 8;  // steps
    f32x16 acc;
#pragma unroll
    for(int r = 0; r < 16; ++r) acc[r] = 0.0f;
    float fa[D][4], fb[D][4];
    int64_t s = 0;
    if(whole >= D) {
        auto load = [&](int d, int64_t step) {
            const int64_t k = 8 * min(step, whole - 1);
            exact_load<!TA>(a + k * sa, p.lda, fa[d]);
            exact_load<TB>(b + k * sb, p.ldb, fb[d]);
        };
#pragma unroll
        for(int d = 0; d < D; ++d) load(d, d);
#pragma unroll 1
        for(; s + D <= whole; s += D) {
#pragma unroll
            for(int d = 0; d < D; ++d) {
#pragma unroll
                for(int i = 0; i < 4; ++i)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[d][i], fb[d][i], acc, 0, 0, 0);
                load(d, s + d + D);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
#pragma unroll 1
    for(int64_t k = 8 * s; k < klen; k += 8) {
#pragma unroll
        for(int i = 0; i < 4; ++i) {
            const bool in = k + 4 * lh + i < klen;
            fa[0][i] = in ? a[(k + i) * sa] : 0.0f;
            fb[0][i] = in ? b[(k + i) * sb] : 0.0f;
        }
#pragma unroll
        for(int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[0][i], fb[0][i], acc, 0, 0, 0);
    }
    return acc;
}

// one MFMA, then its share of the phase's other instructions
template <int N, int DSR, int VALU, int DSW, int VM, int I = 0>
__device__ __forceinline__ void split_sched() {
    if constexpr(I < N) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        constexpr int r = (I + 1) * DSR / N - I * DSR / N, v = (I + 1) * VALU / N - I * VALU / N,
                      w = (I + 1) * DSW / N - I * DSW / N, g = (I + 1) * VM / N - I * VM / N;
        if constexpr(r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
        if constexpr(v > 0) __builtin_amdgcn_sched_group_barrier(0x002, v, 0);
        if constexpr(w > 0) __builtin_amdgcn_sched_group_barrier(0x200, w, 0);
        if constexpr(g > 0) __builtin_amdgcn_sched_group_barrier(0x020, g, 0);
        split_sched<N, DSR, VALU, DSW, VM, I + 1>();
    }
}

template <bool TA, bool TB, int EDGE, class T, int EPI>
__global__ __launch_bounds__(T::THREADS, T::WPS) void gemm_split_kernel(GemmParams p) {
    constexpr int BM = T::BM, BN = T::BN, TM = T::TM, TN = T::TN, NT_ = T::GTHREADS, G = T::G,
                  SETS = T::A;
    constexpr bool AK = !TA, BKF = TB, PAIR = EPI == kEpiSwigluFwd;
    using OA = SplitOperand<AK, BM, NT_>;
    using OB = SplitOperand<BKF, BN, NT_>;
    constexpr int PART = (BM + BN) * SK, STAGE = 3 * PART;  // 16-bit elements
    __shared__ __attribute__((aligned(16))) short lds_all[G * 2 * STAGE];

    const TileJob job = tile_job<T>(p);
    if(job.skip) return;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), l = threadIdx.x % 64;
    const int g = G > 1 ? wv / T::WAVES : 0, w = G > 1 ? wv % T::WAVES : wv;
    const int wm = w / T::WGN, wn = w % T::WGN;
    const int lr = l & 31, lh = l >> 5;
    const int ar0 = wm * TM * 32, br0 = wn * TN * 32;
    short* const lds = lds_all + g * 2 * STAGE;
    // slices per group, an even number unless one group has several sets of sums
    constexpr int STEP = G == 1 && SETS > 1 ? 1 : 2;
    // (K of 1 or 2 runs on the fp32 cores)
    const bool cores = p.K <= 2;
    const int nslices =
        cores ? 0 : (int)((job.kend - job.kbeg + STEP * G * SK - 1) / (STEP * G * SK)) * STEP;

    f32x16 acc[TM][TN], more[SETS > 1 ? SETS - 1 : 1];  // the first set, the others
#pragma unroll
    for(int i = 0; i < TM; ++i)
#pragma unroll
        for(int j = 0; j < TN; ++j)
#pragma unroll
            for(int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
#pragma unroll
    for(int i = 0; i + 1 < SETS; ++i) more[i] = acc[0][0];

    // the scale of op(A)'s parts, whose sign the sums share: one sign to a group,
    // or to a set of sums
    float scale = G > 1 && (g & 1) ? -0x1p16f : 0x1p16f;
    auto set_sign = [&](int a) { return G == 1 && (a & 1) ? -1.0f : 1.0f; };
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
        constexpr int PF = T::PF;
        struct Regs {
            float a[OA::ITEMS][OA::KPI], b[OB::ITEMS][OB::KPI];
        };
        Regs r0, r1;
        const int64_t klen = job.kend - job.kbeg;
        auto load = [&](Regs& r, int s) {
            const int64_t k0 = job.kbeg + ((int64_t)(EDGE ? s : min(s, nslices - 1)) * G + g) * SK;
            if constexpr(EDGE == kFar) {
                far_load<AK, BM, NT_, false, SK>(job.A, p.lda, job.row0, p.M, k0, job.kend, 0, r.a);
                far_load<BKF, BN, NT_, PAIR, SK>(job.B, p.ldb, job.col0, p.N, k0, job.kend, shift, r.b);
            } else {
                split_load<AK, EDGE == kPartial, BM, NT_, false>(sa, p.lda, k0, 0, r.a);
                split_load<BKF, EDGE == kPartial, BN, NT_, PAIR>(sb, p.ldb, k0, shift, r.b);
            }
        };
        auto store = [&](const Regs& r, int stage, float scale_a) {
            split_store<3, AK, BM, NT_, PART>(lds + stage * STAGE, r.a, scale_a);
            split_store<3, BKF, BN, NT_, PART>(lds + stage * STAGE + BM * SK, r.b, 0x1p16f);
        };
        auto mask = [&](Regs& r, int s) {
            if constexpr(EDGE == kPartial) {
                const int64_t limit = klen - ((int64_t)s * G + g) * SK;
                // (k rows of a row-contiguous operand past K lie behind its end)
                if((AK || BKF) && limit < SK) {
                    if(AK) split_mask<AK, BM, NT_>((int)max(limit, (int64_t)0), r.a);
                    if(BKF) split_mask<BKF, BN, NT_>((int)max(limit, (int64_t)0), r.b);
                }
            }
        };
        const int fo = lr * SK + ((lh ^ (lr >> 2)) & 1) * 8;
        auto read = [&](SplitFrag<TM, TN>& f, int stage, int part) {
            const short* t = lds + stage * STAGE + part * PART + fo;
#pragma unroll
            for(int i = 0; i < TM; ++i)
                f.a[i] = *reinterpret_cast<const bf16x8*>(t + (ar0 + i * 32) * SK);
#pragma unroll
            for(int j = 0; j < TN; ++j)
                f.b[j] = *reinterpret_cast<const bf16x8*>(t + (BM + br0 + j * 32) * SK);
        };
        auto mma = [&](f32x16 (&c)[TM][TN], const SplitFrag<TM, TN>& x, const SplitFrag<TM, TN>& y) {
#pragma unroll
            for(int i = 0; i < TM; ++i)
#pragma unroll
                for(int j = 0; j < TN; ++j)
                    c[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x.a[i], y.b[j], c[i][j], 0, 0, 0);
        };
        load(r0, 0);
        mask(r0, 0);
        store(r0, 0, scale);
        load(PF == 2 ? r1 : r0, 1);
        if constexpr(PF == 2) load(r0, 2);
        __syncthreads();
        SplitFrag<TM, TN> f0, f1, m;
        read(f0, 0, 0);
        read(m, 0, 1);
        constexpr int NB = TM * TN, RD = TM + TN;
        constexpr int CV = (OA::ITEMS * OA::KPI + OB::ITEMS * OB::KPI) * 13 / 2;
        constexpr int WR = 3 * (OA::ITEMS + OB::ITEMS);
        constexpr int LD = OA::ITEMS * OA::LOADS + OB::ITEMS * OB::LOADS;
        // scale_a: of the next slice, which is split here
        auto slice = [&](int s, int cur, float scale_a, Regs& r, SplitFrag<TM, TN>& h,
                         SplitFrag<TM, TN>& q, f32x16 (&c)[TM][TN]) {
            mask(r, s + 1);
            read(q, cur, 2);
            store(r, cur ^ 1, scale_a);
            load(r, s + 1 + PF);
            mma(c, m, m);
            mma(c, m, h);
            mma(c, h, m);
            split_sched<3 * NB, RD, CV, WR, LD>();
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            read(m, cur ^ 1, 1);
            mma(c, h, q);
            mma(c, q, h);
            split_sched<2 * NB, RD, 0, 0, 0>();
            __builtin_amdgcn_sched_barrier(0);
            read(q, cur ^ 1, 0);
            mma(c, h, h);
            split_sched<NB, RD, 0, 0, 0>();
            __builtin_amdgcn_sched_barrier(0);
        };
        if constexpr(SETS > 1) {
            auto set = [&](int a) -> f32x16(&)[TM][TN] {
                return a == 0 ? acc : reinterpret_cast<f32x16(&)[TM][TN]>(more[a - 1]);
            };
#pragma unroll 1
            for(int s = 0; s < nslices; s += SETS) {
#pragma unroll
                for(int a = 0; a < SETS; ++a) {
                    if(a % STEP == 0 && a > 0 && s + a >= nslices) break;
                    slice(s + a, a & 1, scale * set_sign(a + 1), r0, a & 1 ? f1 : f0,
                          a & 1 ? f0 : f1, set(a));
                }
            }
        } else {
            int flip = 4;
#pragma unroll 1
            for(int s = 0; s < nslices; s += 2) {
                slice(s, 0, scale, PF == 2 ? r1 : r0, f0, f1, acc);
                const bool turn = G == 1 && s + 2 == flip;
                if(turn) scale = -scale;
                slice(s + 1, 1, scale, r0, f1, f0, acc);
                if(turn) {
                    flip += 8;
#pragma unroll
                    for(int i = 0; i < TM; ++i)
#pragma unroll
                        for(int j = 0; j < TN; ++j) acc[i][j] = -acc[i][j];
                }
            }
        }
    }
    const float unscale = scale * 0x1p-48f;
    // every set of every group is scaled back, and they are added in the order of
    // their first slices, so the tile shapes that deal K to four sums agree bit
    // for bit
    if constexpr(G > 1 || SETS > 1) {
#pragma unroll
        for(int i = 0; i < TM; ++i)
#pragma unroll
            for(int j = 0; j < TN; ++j) acc[i][j] *= unscale;
#pragma unroll
        for(int a = 1; a < SETS; ++a) {
            more[a - 1] *= unscale * set_sign(a);
            if(G == 1) acc[0][0] += more[a - 1];
        }
    }
    if constexpr(G > 1) {
        // the groups' sums meet in LDS: group b % G finishes block b, adding in
        // group order
        f32x4* red = reinterpret_cast<f32x4*>(lds_all);
        constexpr int BLK = T::WAVES * TM * TN * SETS * 4 * 64;  // f32x4 of one group's tile
        auto slot = [&](int from, int b, int a, int r) {
            return (((from * T::WAVES + w) * TM * TN + b) * SETS + a) * 4 * 64 + r * 64 + l;
        };
        static_assert((G - 1) * BLK * 16 <= (int)sizeof(lds_all), "partial tiles fit");
        __syncthreads();
#pragma unroll
        for(int b = 0; b < TM * TN; ++b) {
            const int owner = b % G;
            if(g != owner) {
                const int from = (g - owner + G) % G - 1;
#pragma unroll
                for(int a = 0; a < SETS; ++a)
#pragma unroll
                    for(int r = 0; r < 4; ++r) {
                        const f32x16& x = a == 0 ? acc[b / TN][b % TN] : more[a - 1];
                        red[slot(from, b, a, r)] = f32x4{x[4 * r], x[4 * r + 1], x[4 * r + 2], x[4 * r + 3]};
                    }
            }
        }
        __syncthreads();
#pragma unroll
        for(int b = 0; b < TM * TN; ++b) {
            if(g == b % G) {
#pragma unroll
                for(int a = 0; a < SETS; ++a) {
                    if(a > 0) acc[0][0] += more[a - 1];
#pragma unroll
                    for(int from = 0; from < G - 1; ++from)
#pragma unroll
                        for(int r = 0; r < 4; ++r) {
                            const f32x4 x = red[slot(from, b, a, r)];
#pragma unroll
                            for(int e = 0; e < 4; ++e) acc[b / TN][b % TN][4 * r + e] += x[e];
                        }
                }
            }
        }
    }
    // the wave's blocks with a sum that is not finite
    unsigned again = 0;
#pragma unroll
    for(int b = 0; b < TM * TN; ++b) {
        if(G > 1 && g != b % G) continue;
        float sum = 0.0f;
#pragma unroll
        for(int r = 0; r < 16; ++r) {
            if(G == 1 && SETS == 1) acc[b / TN][b % TN][r] *= unscale;
            sum = fmaf(acc[b / TN][b % TN][r], 0.0f, sum);
        }
        if(cores || __any(sum != 0.0f)) again |= 1u << b;
    }
    // ... among those it stores: a tile's rows and columns past M and N hold anything
    // (looked at only now: 300 instructions that finite tiles need not run)
    if(EDGE != kWhole && again && !cores) {
        unsigned stored = 0;
#pragma unroll
        for(int b = 0; b < TM * TN; ++b) {
            if(G > 1 && g != b % G) continue;
            const int left = (int)min(p.M - job.row0 - ar0 - b / TN * 32 - lh * 4, (int64_t)32);
            const int c = br0 + b % TN * 32 + lr;
            float sum = 0.0f;
#pragma unroll
            for(int r = 0; r < 16; ++r)
                sum = fmaf((r >> 2) * 8 + (r & 3) < left ? acc[b / TN][b % TN][r] : 0.0f, 0.0f, sum);
            const bool in = PAIR ? job.col0 + c % (BN / 2) < p.pair_F : job.col0 + c < p.N;
            if(__any(in && sum != 0.0f)) stored |= 1u << b;
        }
        again = stored;
    }
    again = __builtin_amdgcn_readfirstlane(again);
    auto exact = [&](int b) {
        // (staged epilogues hold the tile's sums meanwhile)
        constexpr int D = EPI == kEpiPlain || T::WPS <= 2 ? 4 : 2;
        return exact_block<TA, TB, PAIR, T, D>(p, job, ar0 + b / TN * 32, br0 + b % TN * 32, lr, lh);
    };
    if constexpr(EPI == kEpiPlain) {
        constexpr int EDGES = EDGE == kWhole ? kEdgeNone : kEdgeScalar;
        store_tile<EDGES, TM, TN, G>(p, job, acc, ar0, br0, lr, lh, g, again);
        // (last, when the sums' registers are free)
        for(; again; again &= again - 1) {
            const int b = __builtin_ctz(again);
            store_block<EDGES, TM * TN == 1>(p, job, exact(b), ar0 + b / TN * 32, br0 + b % TN * 32,
                                             lr, lh);
        }
    } else {
        staged_epilogue<EPI, T, (int)sizeof(lds_all) / 4>(p, job, acc, reinterpret_cast<float*>(lds_all),
                                                         ar0, br0, lr, lh, g, again, exact);
    }
}
