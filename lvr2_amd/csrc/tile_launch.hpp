// Launch of the kNN tile kernel for P lanes per query.  The kernel's instantiations (every sink, with and
// without work counters) are compiled in translation units of their own, one per P
// (knn_tile_p2.hip, knn_tile_p4.hip, knn_tile_p8.hip), so that the library builds in parallel.
#pragma once

#include "knn_tile.hpp"

namespace lvrhip {

// With a work queue the grid is capped at `resident` waves (the ones the device holds at once):
// they drain the queue; without, one wave per run of tiles.
template <int P, template <int> class SinkT>
void launch_tile_p(const BvhView& bv, const QueryView& qv, const TileParams& prm, const SinkT<P>& sink,
                   hipStream_t st, int64_t resident);

}  // namespace lvrhip
