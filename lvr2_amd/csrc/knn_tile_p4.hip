// The kNN tile kernel with four lanes per query, for every sink.
#define TILE_P 4
#include "knn_tile_inst.hpp"
