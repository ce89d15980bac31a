// The 256 x 256 contraction kernel (sub_wide.hpp) with activation SUB_EPI (1 .. 5) in its epilogue.
#include "sub_wide.hpp"

namespace sub {

template <>
void launch_wide_act<SUB_EPI>(const TileProduct& p, hipStream_t st) {
    TileGroup<1> G;
    int k1, k2;
    list_tiles<1>(G, &p, 1, 256, 256, 256, nullptr, k1, k2);
    launch_wide_as<1, SUB_EPI>(G, k1, k2, G.workers, st);
}

}  // namespace sub
