// The 256 x 256 contraction kernel (sub_wide.hpp) without an activation.
#include "sub_wide.hpp"

namespace sub {

namespace {

template <int NP>
void launch_plain(const TileProduct* p, int n, FinishJobs* tail, unsigned side_blocks, hipStream_t st) {
    TileGroup<NP> G;
    int k1, k2;
    list_tiles<NP>(G, p, n, TILE_256x256, tail, k1, k2);
    launch_wide_as<NP, EPI_PLAIN>(G, k1, k2, G.workers + (unsigned)G.tail.n * G.tail_groups + side_blocks, st);
}

}  // namespace

// Operands contiguous along k in whole steps (the words behind a remainder would need masks of their own; of others, k rows
// beyond the last lie beyond the operand), not split, and 2^31 bytes from a tile's first element to its last.
bool wide_takes(const TileProduct& p) {
    const GemmArgs& a = p.a;
    const long la = 255 * a.sAM + (long)(a.K1 + BK) * a.sAK1, lb = 255 * a.sBN + (long)(a.K1 + BK) * a.sBK1;
    return a.splits == 1 && (a.K1 % BK == 0 || !(p.akc || p.bkc)) && la < (1L << 30) && lb < (1L << 30);
}

void launch_wide(const TileProduct* p, int n, FinishJobs* tail, unsigned side_blocks, hipStream_t st) {
    if (n == 1 && !(tail && tail->n)) launch_plain<1>(p, n, tail, side_blocks, st);
    else if (side_blocks) fail("gemm: a side job has its product to itself");
    else launch_plain<kMaxProducts>(p, n, tail, 0, st);
}

}  // namespace sub
