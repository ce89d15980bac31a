// The contraction kernels with activation SUB_EPI (1 .. 6) in their epilogue.
#include "sub_ring.hpp"
#include "sub_wide.hpp"

namespace sub {

template <>
void launch_act<SUB_EPI>(const TileProduct& p, int form, hipStream_t st) {
    TileGroup<1> G;
    int k1, k2;
    list_tiles<1>(G, &p, 1, form, nullptr, k1, k2);
    if (form == TILE_256x256) launch_wide_as<1, SUB_EPI>(G, k1, k2, G.workers, st);
    // (k_gemm_ring takes keep bits drawn ahead, where there are any, in the same instance)
    else if constexpr (SUB_EPI != EPI_RELU_DROPOUT_PRE) launch_ring_as<1, SUB_EPI>(G, form, k1, k2, G.workers, st);
    else launch_act<EPI_RELU_DROPOUT>(p, form, st);
}

}  // namespace sub
