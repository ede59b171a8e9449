// The kNN tile kernel with eight lanes per query, for every sink.
#define TILE_P 8
#include "knn_tile_inst.hpp"
