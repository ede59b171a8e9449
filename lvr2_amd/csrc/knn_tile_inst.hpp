// Definition of launch_tile_p and its explicit instantiations for TILE_P lanes per query (defined by
// the including knn_tile_p*.hip).
#pragma once

#include <algorithm>

#include "adjoint.hpp"
#include "knn_tile.hpp"
#include "sinks.hpp"
#include "tile_launch.hpp"

namespace lvrhip {

template <int P, template <int> class SinkT>
void launch_tile_p(const BvhView& bv, const QueryView& qv, const TileParams& prm, const SinkT<P>& sink,
                   hipStream_t st, int64_t resident)
{
    constexpr int Q = kWave / P;
    const int64_t ntiles = ceil_div(qv.nq, Q);
    int64_t grid = ceil_div(ntiles, prm.tiles_per_wave);
    if (grid == 0) return;
    if (prm.queue) {
        grid = std::min(grid, resident);
        if (!prm.queue_zeroed) {
            fill_u32_kernel<<<1, 256, 0, st>>>(prm.queue, QUEUE_SEGS * QUEUE_STRIDE, 0u);
            LVRHIP_LAUNCH_CHECK();
        }
    }
    if (prm.stats)
        knn_tile_kernel<P, SinkT<P>, true><<<(unsigned)grid, kWave, 0, st>>>(bv, qv, prm, sink);
    else
        knn_tile_kernel<P, SinkT<P>, false><<<(unsigned)grid, kWave, 0, st>>>(bv, qv, prm, sink);
    LVRHIP_LAUNCH_CHECK();
}

#define LVRHIP_TILE_INST(SINK)                                                                               \
    template void launch_tile_p<TILE_P, SINK>(const BvhView&, const QueryView&, const TileParams&,            \
                                              const SINK<TILE_P>&, hipStream_t, int64_t)
LVRHIP_TILE_INST(SinkNormals);
LVRHIP_TILE_INST(SinkMoments);
LVRHIP_TILE_INST(SinkLevels);
LVRHIP_TILE_INST(SinkSdf);
LVRHIP_TILE_INST(SinkList);
LVRHIP_TILE_INST(SinkKiOnly);
LVRHIP_TILE_INST(SinkSdfAdjoint);
LVRHIP_TILE_INST(SinkPcaAdjoint);
#undef LVRHIP_TILE_INST

}  // namespace lvrhip
