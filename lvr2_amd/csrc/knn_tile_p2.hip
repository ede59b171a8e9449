// The kNN tile kernel with two lanes per query, for every sink.
#define TILE_P 2
#include "knn_tile_inst.hpp"
