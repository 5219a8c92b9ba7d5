// pico_amd/csrc/gemm_split.hip -- launches of the fp32 product (gemm_split.h).
#include "gemm_common.h"

namespace {

using namespace pkg;

#include "gemm_split.h"

// the fp32 products' shapes of the same names (gemm_split.h)
using Split256 = SplitTile<2, 4, 4, 2, 1, 2, 1>;
using Split128 = SplitTile<2, 4, 2, 1, 2, 4, 1>;
using Split256x96 = SplitTile<4, 1, 2, 3, 2, 2, 1>;
using Split128x64 = SplitTile<2, 2, 2, 1, 2, 4, 1>;
using Split64 = SplitTile<2, 2, 1, 1, 4, 4, 2>;
using Split64x2 = SplitTile<2, 2, 1, 1, 2, 4, 1, 2>;
using Split64x1 = SplitTile<2, 2, 1, 1, 1, 4, 1, 4>;

template <bool TA, bool TB, int EDGE, class T>
void launch_split_kernel(const GemmParams& gp, dim3 grid, hipStream_t st) {
    if constexpr(!TA && TB) {
        if(gp.sg_a) {
            gemm_split_kernel<TA, TB, EDGE, T, kEpiSwiglu><<<grid, T::THREADS, 0, st>>>(gp);
            return;
        }
    }
    if constexpr(!TA && !TB) {
        if(gp.sf_h) {
            gemm_split_kernel<TA, TB, EDGE, T, kEpiSwigluFwd><<<grid, T::THREADS, 0, st>>>(gp);
            return;
        }
        if(gp.Cin) {
            gemm_split_kernel<TA, TB, EDGE, T, kEpiAdd><<<grid, T::THREADS, 0, st>>>(gp);
            return;
        }
    }
    gemm_split_kernel<TA, TB, EDGE, T, kEpiPlain><<<grid, T::THREADS, 0, st>>>(gp);
}

template <bool TA, bool TB, class T>
int launch_split_tile(const GemmParams& gp, int64_t batch, bool edge, hipStream_t st) {
    dim3 grid((unsigned)(gp.tiles_m * gp.tiles_n), (unsigned)(gp.splits > 1 ? gp.splits : batch));
    if(edge)
        launch_split_kernel<TA, TB, kPartial, T>(gp, grid, st);
    else
        launch_split_kernel<TA, TB, kWhole, T>(gp, grid, st);
    return pk::launch_status("pk_gemm_f32");
}

template <bool TA, bool TB>
int launch_layout(const GemmParams& gp, int64_t batch, bool edge, TileKind kind, hipStream_t st) {
    switch(kind) {
    case kTile256: return launch_split_tile<TA, TB, Split256>(gp, batch, edge, st);
    case kTile256x96: return launch_split_tile<TA, TB, Split256x96>(gp, batch, edge, st);
    case kTile128x64: return launch_split_tile<TA, TB, Split128x64>(gp, batch, edge, st);
    case kTile64: return launch_split_tile<TA, TB, Split64>(gp, batch, edge, st);
    case kTile64x2: {
        if(!gp.far) return launch_split_tile<TA, TB, Split64x2>(gp, batch, edge, st);
        dim3 grid((unsigned)(gp.tiles_m * gp.tiles_n),
                  (unsigned)(gp.splits > 1 ? gp.splits : batch));
        launch_split_kernel<TA, TB, kFar, Split64x2>(gp, grid, st);
        return pk::launch_status("pk_gemm_f32");
    }
    case kTile64x1: return launch_split_tile<TA, TB, Split64x1>(gp, batch, edge, st);
    default: return launch_split_tile<TA, TB, Split128>(gp, batch, edge, st);
    }
}

}  // namespace

namespace pkg {

int split_groups(TileKind kind) {
    return kind == kTile64 ? Split64::G : kind == kTile256 || kind == kTile64x1 ? 1 : 2;
}

int launch_split(bool ta, bool tb, const GemmParams& gp, int64_t batch, bool edge, TileKind kind,
                 hipStream_t st) {
    if(!ta && !tb) return launch_layout<false, false>(gp, batch, edge, kind, st);
    if(!ta && tb) return launch_layout<false, true>(gp, batch, edge, kind, st);
    if(ta && !tb) return launch_layout<true, false>(gp, batch, edge, kind, st);
    return launch_layout<true, true>(gp, batch, edge, kind, st);
}

}  // namespace pkg
