// Self-attention without score-sized tensors in memory.
//
// The reference keeps five tensors of the size of the score matrix per layer
// (pytorch_module/encoder.cu:104-131 forward: BETA, ALPHA, ATTN_DROP_MASK,
// ATTN_DROP; :222-262 backward: DATTN_DROP, DBETA) and moves each of them
// through memory two or three times.  Here a tile of 32 x 32 scores lives only in
// the accumulator registers of one wave:
//
//   forward     per 32 queries, over all keys: S = a.Q.K^T, running softmax
//               (max and sum per query), dropout, O += P_drop.V; writes O, the
//               log-sum-exp of each score row and one keep bit per score
//   backward dQ per 32 queries, over all keys: recomputes P from the log-sum-exp,
//               dP = dO.V^T, dS = P (keep.dP - D), dQ += dS.K with D = rowsum(dO o O)
//   backward dK, dV  per 32 keys, over all queries: the same dS and P_drop,
//               dK += dS^T.Q, dV += P_drop^T.dO
//
// Scores are formed as D[key, query] (dQ, forward) so that everything that is
// per query -- running max, sum, log-sum-exp, D, the keep word -- is per lane,
// and as D[query, key] in the dK/dV kernel.  Either way the score tile is, as it
// lies in the accumulator registers, the B operand of the next product with the
// contraction index running over the registers in the order
//   element i of step s  <->  index (2s + i/4)*8 + 4*(lane/32) + i%4 ;
// the A operand is gathered in the same order from an LDS tile with the
// transposing read, so no score ever moves between lanes.
#include <type_traits>

#include "sub_ops.hpp"

namespace sub {

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef short s8v __attribute__((ext_vector_type(8)));
constexpr float LOG2E = 1.4426950408889634f;
constexpr int QB = 128;           // positions per workgroup: 4 waves x 32
constexpr float RESCALE_SLACK = 8.f;   // unnormalised probabilities stay below 2^8

template <int P>
struct Geo {
    static constexpr int NKS = P / 16;             // k-steps of a contraction over the features
    static constexpr int NPT = P / 32;             // 32-wide tiles of the feature dim
    static constexpr int TILE = 32 * P;            // halves of an LDS tile of 32 positions
    static constexpr int VL = (32 * (P / 8)) / 256; // 16-byte words per thread and tile (of 256 threads)

    // LDS tiles are [position][feature] without padding; the index of a 16-byte
    // chunk within its row is xor-ed with a function of the row chosen so that both
    // ways of reading a tile are free of bank conflicts: 16 consecutive rows at one
    // chunk (the features as contraction index, ds_read_b128) and 4 consecutive
    // rows x 4 adjacent chunks (the positions as contraction index, transposing read).
    static __device__ __forceinline__ int swz(int row) {
        return P == 64 ? ((((row >> 1) & 1) << 2) | ((row >> 2) & 3)) : (((row & 3) << 2) | ((row >> 2) & 3));
    }
    // offset in halves of chunk c of a row
    static __device__ __forceinline__ int at(int row, int c) { return row * P + ((c ^ swz(row)) << 3); }
};

// Fragment of 32 rows (one per lane%32) with the features as contraction index:
// A or B operand of v_mfma_f32_32x32x16_f16, straight from global memory.
template <int P>
__device__ __forceinline__ void row_frags(const AttnSide& t, unsigned h, unsigned b, unsigned pos, int hi,
                                          h8 (&f)[P / 16]) {
    const half_t* p = t.p + (long)h * t.sh + (long)b * t.sb + (long)pos * t.sr + hi * 8;
#pragma unroll
    for (int ks = 0; ks < P / 16; ++ks) f[ks] = *reinterpret_cast<const h8*>(p + ks * 16);
}

// The same fragment from an LDS tile.
template <int P>
__device__ __forceinline__ void row_frags_lds(const half_t* tile, int l32, int hi, h8 (&f)[P / 16]) {
#pragma unroll
    for (int ks = 0; ks < P / 16; ++ks)
        f[ks] = *reinterpret_cast<const h8*>(tile + Geo<P>::at(l32, 2 * ks + hi));
}

// A tile of 32 positions x P features: global -> registers -> LDS, all threads.  RAGGED: positions from `limit` on
// read the last one that there is (their scores are taken out where they would count).
// PARTS: by 256 / PARTS threads.
template <int P, bool RAGGED, int PARTS = 1>
__device__ __forceinline__ void tile_fetch(const AttnSide& t, unsigned h, unsigned b, unsigned pos0, unsigned limit, int tid,
                                           h8 (&r)[Geo<P>::VL * PARTS]) {
#pragma unroll
    for (int i = 0; i < Geo<P>::VL * PARTS; ++i) {
        const int id = tid + i * (256 / PARTS), row = id / (P / 8), c = id % (P / 8);
        const unsigned pos = RAGGED ? min(pos0 + row, limit - 1) : pos0 + row;
        r[i] = *reinterpret_cast<const h8*>(t.p + (long)h * t.sh + (long)b * t.sb + (long)pos * t.sr + c * 8);
    }
}
// The tiles of 32 positions of one side.  WALK: one after the other from the first on, whole ones, by an address that moves
// along; else wherever they lie, by a 64-bit product for each row (four to eight quarter-rate multiplications a tile among
// vector work that bounds these kernels: H 16, P 64, 8 x 512 forward 24.8 -> 24.2 us, dK and dV 31.2 -> 30.6; H 32, P 128,
// 4 x 2048 forward 497 -> 487, dQ 528 -> 509).
template <int P, bool WALK, bool RAGGED, int PARTS>
struct Tiles {
    const half_t* p;
    __device__ __forceinline__ Tiles(const AttnSide& t, unsigned h, unsigned b, unsigned first, int tid)
        : p(WALK ? t.p + (long)h * t.sh + (long)b * t.sb + (long)(first * 32 + tid / (P / 8)) * t.sr + tid % (P / 8) * 8 : nullptr) {}
    __device__ __forceinline__ void fetch(const AttnSide& t, unsigned h, unsigned b, unsigned tile, unsigned limit, int tid,
                                          h8 (&r)[Geo<P>::VL * PARTS]) {
        if (!WALK) { tile_fetch<P, RAGGED, PARTS>(t, h, b, tile * 32, limit, tid, r); return; }
#pragma unroll
        for (int i = 0; i < Geo<P>::VL * PARTS; ++i) r[i] = *reinterpret_cast<const h8*>(p + i * (256 / PARTS / (P / 8)) * t.sr);
        p += 32 * t.sr;
    }
};
template <int P, int PARTS = 1>
__device__ __forceinline__ void tile_put(half_t* tile, int tid, const h8 (&r)[Geo<P>::VL * PARTS]) {
#pragma unroll
    for (int i = 0; i < Geo<P>::VL * PARTS; ++i) {
        const int id = tid + i * (256 / PARTS), row = id / (P / 8), c = id % (P / 8);
        *reinterpret_cast<h8*>(tile + Geo<P>::at(row, c)) = r[i];
    }
}

// A operand with the tile's positions as contraction index: lane%32 = feature
// m0 + lane%32, elements = positions in the register order of a score tile.
// ds_read_b64_tr_b16: within 16 lanes, lane i receives T[k0 + 0..3][m0 + i] when
// lane l addresses T[k0 + l/4][m0 + 4*(l%4)].
template <int P>
__device__ __forceinline__ h8 tr_frag(const half_t* tile, int m0, int s, int lane) {
    const int g = lane >> 4, l = lane & 15;
    const int k = 16 * s + 4 * (g >> 1) + (l >> 2);
    const int m = m0 + 16 * (g & 1) + 4 * (l & 3);
    typedef s4v __attribute__((address_space(3))) * lds_s4;
    s4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(tile + Geo<P>::at(k, m >> 3) + (m & 7)));
    s4v up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(tile + Geo<P>::at(k + 8, m >> 3) + (m & 7)));
    s8v r = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(h8, r);
}

// Workgroups are dealt to the 8 XCDs (each with its own L2) in turn.  Renumbered
// so that consecutive logical blocks -- the blocks of one head and sample, which
// read the same K, V (or Q, dO) -- run on one XCD and share its L2.
__device__ __forceinline__ unsigned logical_block() {
    const unsigned n = gridDim.x, bid = blockIdx.x;
    return (n % 8u) ? bid : (bid % 8u) * (n / 8u) + bid / 8u;
}

// Position (within a tile of 32) that accumulator register v of a lane holds.
__device__ __forceinline__ constexpr int reg_pos(int v, int hi) { return (v >> 2) * 8 + hi * 4 + (v & 3); }

// Output rows: D[feature, position] accumulators of a wave -> t[position][feature] for its 32 positions from pos0 on,
// those below `limit`, by way of LDS (`tile`: 32 * P halves, the wave's own): an accumulator holds a position per lane, so
// that straight from the registers an instruction writes 16 bytes to each of 32 rows, and from LDS whole rows.  On the way
// the columns of what is stored are summed, into `sums` (of the wave: 4 rows of P floats, one for each 16 lanes; or null).
// Straight from the registers 6 of the 35 us of dK and dV at H 16, P 64, 8 x 512 were the stores and 1 the sums (9
// instructions a value), at 96 x 128 17 and 1 of 48.  This way: 8 x 512: dK and dV 35.3 -> 32.4 us, forward 26.3 -> 25.7;
// 96 x 128: dK and dV 48.5 -> 38.3, dQ 41.9 -> 38.3, forward 31.5 -> 28.0.
// (Nothing of the addresses below is to be kept in registers while the tiles are worked on: the lane's index is made anew
// here, and the callers' wave index is a scalar.  Without that a lane needed 4 to 20 registers more, one wave per SIMD
// instead of two in the forward kernel of head size 128 at odd lengths: 4 x 1000, H 16, P 128: 104 us, with it 76.6.)
template <int P, bool RAGGED>
__device__ __forceinline__ void store_rows(const AttnSide& t, unsigned h, unsigned b, unsigned pos0, unsigned limit, int lane,
                                           const f16v (&acc)[P / 32], float scale, half_t* tile, float* sums) {
    constexpr int PER = P / 8, ROWS = WAVE / PER;      // 16-byte words of a row, rows of an instruction
    asm volatile("" : "+v"(lane));
    const int l32 = lane & 31, hi = lane >> 5, row = lane / PER, chunk = lane % PER;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int pt = 0; pt < P / 32; ++pt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            h4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = (half_t)(acc[pt][q * 4 + e] * scale);
            *reinterpret_cast<h4*>(tile + Geo<P>::at(l32, pt * 4 + q) + hi * 4) = w;
        }
    __builtin_amdgcn_wave_barrier();
    half_t* p = const_cast<half_t*>(t.p) + (long)h * t.sh + (long)b * t.sb + (long)(pos0 + row) * t.sr + chunk * 8;
    h8 w[32 / ROWS];
#pragma unroll
    for (int i = 0; i < 32 / ROWS; ++i) w[i] = *reinterpret_cast<const h8*>(tile + Geo<P>::at(i * ROWS + row, chunk));
#pragma unroll
    for (int i = 0; i < 32 / ROWS; ++i)
        if (!RAGGED || pos0 + i * ROWS + row < limit) *reinterpret_cast<h8*>(p + (long)(i * ROWS) * t.sr) = w[i];
    if (!sums) return;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 32 / ROWS; ++i) {
        const bool in = !RAGGED || pos0 + i * ROWS + row < limit;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += in ? (float)w[i][e] : 0.f;
    }
    if (P == 64) {          // two rows in 16 lanes
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += dpp<0x128>(x[e]);
        if (lane & 8) return;
    }
#pragma unroll
    for (int e = 0; e < 8; e += 4)
        *reinterpret_cast<float4*>(sums + (lane >> 4) * P + chunk * 8 + e) = make_float4(x[e], x[e + 1], x[e + 2], x[e + 3]);
}
// One value per feature of what WAVES waves have left in `sums`; behind a barrier.
template <int P, int WAVES>
__device__ __forceinline__ float column_sum(const float* sums, int feature) {
    float x[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4 * WAVES; ++i) x[i & 3] += sums[i * P + feature];
    return (x[0] + x[1]) + (x[2] + x[3]);
}

// x where bit `pos` of `bits` is set, else +0.0
__device__ __forceinline__ float keep_if(float x, uint32_t bits, int pos) {
    return __int_as_float(__float_as_int(x) & __builtin_amdgcn_sbfe((int)bits, pos, 1));
}
// The same of what a vector instruction has made (not of a product: nothing waits for one here).  Spelled out: as a choice it is
// three instructions, and that is what the compiler makes of a mask in the forward kernel (4 x 1024: 47.8 us, as a choice 50.5).
template <int pos>
__device__ __forceinline__ float keep_probability(float x, uint32_t bits) {
    float r;
    asm("v_bfe_i32 %0, %1, %2, 1\n\tv_and_b32 %0, %0, %3" : "=&v"(r) : "v"(bits), "n"(pos), "v"(x));
    return r;
}

// Scores of positions from `limit` on (the tile starts at tile0, register v of a lane holds position reg_pos(v, hi) of
// it) vanish from everything that is formed from them.
__device__ __forceinline__ void drop_past_end(f16v& s, unsigned tile0, unsigned limit, int hi) {
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = tile0 + reg_pos(v, hi) < limit ? s[v] : -INFINITY;
}

// Words of keep bits per score row: one per 32 keys, in whole groups of four (mha_keep_pitch).
__device__ __forceinline__ unsigned keep_pitch(unsigned K) { return (K + QB - 1) / QB * 4; }

// Additive attention mask (substation/attention.py:65-68: added to the raw scores,
// before the scaling) for the 16 scores of a lane.  QUERY_LANES: the lane holds
// one query and registers run over keys (forward, dQ); otherwise the lane holds
// one key and registers run over queries (dK/dV).  The values of a tile are loaded
// while the tile before it is worked on, ahead of that pass's K/V (Q/dO) loads:
// loads complete in order, so a wait for mask values issued after those would
// also wait for them.
struct MaskRegs { h4 q[4]; };

template <bool QUERY_LANES, bool RAGGED>
__device__ __forceinline__ void load_mask(const AttnArgs& a, unsigned lane_pos, unsigned tile0, int hi, MaskRegs& mk) {
    const long lane_stride = QUERY_LANES ? a.am_sj : a.am_sk, reg_stride = QUERY_LANES ? a.am_sk : a.am_sj;
    const half_t* m = a.amask + (long)lane_pos * lane_stride + (long)tile0 * reg_stride;
    const unsigned limit = QUERY_LANES ? a.K : a.J;
    if (RAGGED && (reg_stride != 1 || (lane_stride & 3) != 0 || tile0 + 32 > limit)) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
            mk.q[v >> 2][v & 3] = m[(long)(min(tile0 + reg_pos(v, hi), limit - 1) - tile0) * reg_stride];
    } else if (reg_stride == 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) mk.q[q] = *reinterpret_cast<const h4*>(m + q * 8 + hi * 4);
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) mk.q[v >> 2][v & 3] = m[(long)reg_pos(v, hi) * reg_stride];
    }
}

// The scores of a tile start from the mask's values instead of zero: the product
// accumulates on top of them.
__device__ __forceinline__ void start_from_mask(const MaskRegs& mk, f16v& s) {
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = (float)mk.q[v >> 2][v & 3];
}

// ---------------------------------------------------------------------------
// What a mask leaves to do.  Each 32x32 block of the mask is classed as mixed,
// dead (all -inf: the scores vanish) or clear (all zero: nothing to add).  Per
// workgroup of the attention kernels (128 queries, or 128 keys in the dK/dV
// kernel) a list names the tiles of the other side that are not dead for all
// four waves; the kernels walk that list instead of all tiles.
//   row of a list: [0] = number of entries, then the entries, then padding that
//   reads as "tile 0, dead for all waves" (the kernels read up to 4 past the end).
//   entry: bits 0..15 tile index, bits 16+2w.. the class of the block for wave w.
// ---------------------------------------------------------------------------
enum : uint32_t { BLOCK_MIXED = 0, BLOCK_DEAD = 1, BLOCK_CLEAR = 2 };
constexpr uint32_t kAllDead = BLOCK_DEAD * 0x55u << 16;
constexpr int kListPad = 5;       // the count and four entries of padding

// One wave per 32x32 block of the mask.
__global__ __launch_bounds__(64) void k_mha_mask_classes(const half_t* mask, long sj, long sk, int J, int K, uint8_t* cls) {
    const int lane = threadIdx.x, nkb = (K + 31) / 32;
    const int qb = blockIdx.x / nkb, kb = blockIdx.x % nkb;
    // positions past the end stand for the last one that there is: they change nobody's class
    const half_t* p = mask + (long)min(qb * 32 + (lane & 31), J - 1) * sj;
    bool dead = true, clear = true;
    for (int i = 0; i < 16; ++i) {
        const float x = (float)p[(long)min(kb * 32 + (lane >> 5) * 16 + i, K - 1) * sk];
        dead = dead && (x == -INFINITY);
        clear = clear && (x == 0.f);
    }
    const bool all_dead = __builtin_amdgcn_ballot_w64(dead) == ~0ull;
    const bool all_clear = __builtin_amdgcn_ballot_w64(clear) == ~0ull;
    if (lane == 0) cls[blockIdx.x] = all_dead ? BLOCK_DEAD : all_clear ? BLOCK_CLEAR : BLOCK_MIXED;
}

// One wave per list row: the first ceil(J/128) blocks build the key-tile lists of the query
// blocks, the others the query-tile lists of the key blocks.
__global__ __launch_bounds__(64) void k_mha_mask_lists(const uint8_t* cls, int J, int K, uint32_t* qlist, uint32_t* klist) {
    const int lane = threadIdx.x, nqb = (J + 31) / 32, nkb = (K + 31) / 32, nblk = (J + QB - 1) / QB;
    const bool by_query = (int)blockIdx.x < nblk;
    const int blk = by_query ? blockIdx.x : blockIdx.x - nblk;
    const int ntiles = by_query ? nkb : nqb;
    uint32_t* row = (by_query ? qlist : klist) + (size_t)blk * (ntiles + kListPad);
    unsigned count = 0;
    for (int t0 = 0; t0 < ntiles; t0 += 64) {
        const int t = t0 + lane;
        uint32_t e = kAllDead;
        if (t < ntiles) {
            e = (uint32_t)t;
            for (int w = 0; w < 4; ++w) {
                // (a wave whose 32 positions all lie past the end has nothing to do)
                uint32_t c = BLOCK_DEAD;
                if (blk * 4 + w < (by_query ? nqb : nkb))
                    c = by_query ? cls[(size_t)(blk * 4 + w) * nkb + t] : cls[(size_t)t * nkb + blk * 4 + w];
                e |= c << (16 + 2 * w);
            }
        }
        const bool live = (e & (0xffu << 16)) != kAllDead;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(live);
        if (live) row[1 + count + __builtin_popcountll(m & ((1ull << lane) - 1))] = e;
        count += (unsigned)__builtin_popcountll(m);
    }
    if (lane == 0) row[0] = count;
    for (int i = count + lane; i < ntiles + kListPad - 1; i += 64) row[1 + i] = kAllDead;
}

// Which block of 128 (and which head and sample) a workgroup takes when a mask has
// left the blocks unequal amounts to do.  Workgroups start in the order of their
// index.  The blocks of a head and sample are ranked long to short (the reverse of
// their positions when the last has more to do than the first: a causal mask seen
// from the queries) and dealt in four passes over the heads and samples of an XCD,
// a quarter of the ranks per pass, so that the launch does not end on a few long
// blocks running alone.
__device__ __forceinline__ void masked_order(const uint32_t* list, unsigned nblocks, unsigned ntiles, unsigned ngroups,
                                             unsigned lb, unsigned& blk, unsigned& hb) {
    blk = lb % nblocks; hb = lb / nblocks;
    if (!list) return;
    const bool rev = list[(size_t)(nblocks - 1) * (ntiles + kListPad)] > list[0];
    unsigned rank = blk;
    if (nblocks % 4 == 0 && ngroups % 8 == 0) {
        const unsigned gx = ngroups / 8, per = nblocks / 4;          // groups per XCD; blocks per pass and group
        const unsigned x = lb / (gx * nblocks), i = lb % (gx * nblocks);
        const unsigned pass = i / (gx * per), rem = i % (gx * per);
        hb = x * gx + rem / per;
        rank = pass * per + rem % per;
    }
    blk = rev ? nblocks - 1 - rank : rank;
}

// Entry i of a list row; without a list every tile is walked and treated as mixed.
template <bool MASKED>
__device__ __forceinline__ uint32_t live_entry(const uint32_t* row, unsigned i) {
    return (MASKED && row) ? row[1 + i] : i;
}
__device__ __forceinline__ unsigned entry_tile(uint32_t e) { return e & 0xffffu; }
__device__ __forceinline__ uint32_t entry_class(uint32_t e, int wave) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)((e >> (16 + 2 * wave)) & 3u));
}

// ---------------------------------------------------------------------------
// All three kernels stream tiles of 32 positions through a ring of three LDS
// buffers: while tile t is worked on, tile t+1 already lies in LDS (its row
// fragments are read ahead, during the vector work on tile t) and tile t+2 is on
// its way from memory in registers.  One barrier per tile.
//
// PARTS = 2 (head size 64): two waves of 32 positions and, for each, two waves that walk a half of the other side's tiles
// each, through a ring of their own.  What they have come to is added up at the end, by way of LDS.  Twice the workgroups
// with half the tiles each, where there are few (see parts).
// ---------------------------------------------------------------------------
constexpr int RING = 3;
constexpr long kFewBlocks = 128;  // workgroups of a launch without (see parts)

// The place of a wave: of `blocks` of QB positions, in PARTS pieces each.
template <int PARTS>
struct Place {
    static constexpr int WAVES = 4 / PARTS;          // of 32 positions
    int tid, lane, wave, half;                       // (tid, wave: within the half)
    __device__ __forceinline__ Place() : tid(threadIdx.x % (256 / PARTS)), lane(threadIdx.x & 63), wave((threadIdx.x >> 6) % WAVES),
                                         half(PARTS > 1 ? threadIdx.x / (256 / PARTS) : 0) {}
};

// A wave's accumulators to the other half's wave and back: 16 N words of 64 lanes.
template <int N>
__device__ __forceinline__ void leave(float* to, int lane, const f16v (&acc)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int v = 0; v < 16; v += 4)
            *reinterpret_cast<float4*>(to + ((i * 4 + v / 4) * 64 + lane) * 4) = make_float4(acc[i][v], acc[i][v + 1], acc[i][v + 2], acc[i][v + 3]);
}
// acc = acc * mine + (what is left there) * theirs; what lay there is no longer needed.
template <int N>
__device__ __forceinline__ void collect(const float* from, int lane, f16v (&acc)[N], float mine, float theirs) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            const float4 x = *reinterpret_cast<const float4*>(from + ((i * 4 + v / 4) * 64 + lane) * 4);
            acc[i][v] = acc[i][v] * mine + x.x * theirs; acc[i][v + 1] = acc[i][v + 1] * mine + x.y * theirs;
            acc[i][v + 2] = acc[i][v + 2] * mine + x.z * theirs; acc[i][v + 3] = acc[i][v + 3] * mine + x.w * theirs;
        }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // (halves are written there next, which the compiler takes for other memory)
}

// Every load issued so far has arrived.  Placed before a main loop: a load of the
// prologue whose first use is inside the loop would otherwise put its wait there,
// where on every later pass it waits for the loads that pass has just issued.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }   // vmcnt(0)

// ---------------------------------------------------------------------------
// forward.  grid = H * B * ceil(J / 128); wave = 32 queries.
//
// RAGGED: J or K is not a multiple of 128.  Loads of positions past the end are clamped, the scores of the last key
// tile's missing keys are set to -inf, and rows past the end are not written.  Without it such lengths took the operators
// one by one, with the score-sized tensors in memory and, for lengths that are not multiples of 8, products
// through the scalar kernel: the layer's forward and backward at B=13 L=201 E=768 took 3990 us.
// ---------------------------------------------------------------------------
template <int P, bool MASKED, bool RAGGED, int PARTS>
__device__ __forceinline__ void mha_fwd(const AttnArgs& a, const PhiloxKey& key_) {
    using G = Geo<P>;
    __shared__ __attribute__((aligned(16))) half_t kt_[PARTS][RING][G::TILE];
    __shared__ __attribute__((aligned(16))) half_t vt_[PARTS][RING][G::TILE];
    const PhiloxKey key = resolved(key_);
    const Place<PARTS> at;
    const int tid = at.tid, lane = at.lane, wave = at.wave, l32 = lane & 31, hi = lane >> 5;
    half_t (*const kt)[G::TILE] = kt_[at.half];
    half_t (*const vt)[G::TILE] = vt_[at.half];
    const unsigned qblocks = RAGGED ? (a.J + QB - 1) / QB : a.J / QB;
    const unsigned lb = logical_block() / PARTS;
    const unsigned nt = RAGGED ? (a.K + 31) / 32 : a.K / 32, pitch = RAGGED ? keep_pitch(a.K) : nt;
    unsigned qb = lb % qblocks, hb = lb / qblocks;
    if (MASKED) masked_order(a.qlist, qblocks, nt, a.H * a.B, lb, qb, hb);
    const unsigned b = hb % a.B, h = hb / a.B;
    const int piece = PARTS > 1 ? (int)(logical_block() % PARTS) * Place<PARTS>::WAVES : 0;      // its first wave's, of the block's four
    const unsigned j_ = qb * QB + (piece + wave) * 32 + l32;                   // this lane's query
    const bool mine_ = !RAGGED || j_ < (unsigned)a.J;                // (RAGGED: lanes past the end follow the last query)
    const unsigned j = RAGGED ? min(j_, (unsigned)a.J - 1) : j_;
    // waves whose queries all lie past the end only help with the tiles
    const bool working = !RAGGED || __builtin_amdgcn_readfirstlane((int)(qb * QB + (piece + wave) * 32)) < a.J;
    const unsigned row = (h * a.B + b) * a.J + j;                    // its score row
    const float c = a.alpha * LOG2E;
    // the key tiles to walk: all of them, or those a mask leaves for these 128 queries
    const uint32_t* live = (MASKED && a.qlist) ? a.qlist + (size_t)qb * (nt + kListPad) : nullptr;
    const unsigned all = live ? live[0] : nt, longest = (all + PARTS - 1) / PARTS;
    // (the second half's begin behind the first's; of an odd number it has one less)
    const unsigned begin = at.half ? longest : 0, n = at.half ? all - longest : longest;
    uint32_t e0 = live_entry<MASKED>(live, begin), e1 = live_entry<MASKED>(live, begin + 1), e2 = live_entry<MASKED>(live, begin + 2);

    h8 fq[G::NKS], fk[G::NKS], kr[G::VL * PARTS], vr[G::VL * PARTS];
    Tiles<P, !MASKED && !RAGGED, RAGGED, PARTS> tiles_k(a.k, h, b, begin, tid), tiles_v(a.v, h, b, begin, tid);
    {   // the first two tiles and the query rows: all loads in flight together
        h8 kr1[G::VL * PARTS], vr1[G::VL * PARTS];
        tiles_k.fetch(a.k, h, b, entry_tile(e0), a.K, tid, kr);
        tiles_v.fetch(a.v, h, b, entry_tile(e0), a.K, tid, vr);
        tiles_k.fetch(a.k, h, b, entry_tile(e1), a.K, tid, kr1);
        tiles_v.fetch(a.v, h, b, entry_tile(e1), a.K, tid, vr1);
        row_frags<P>(a.q, h, b, j, hi, fq);
        tile_put<P, PARTS>(kt[0], tid, kr);
        tile_put<P, PARTS>(vt[0], tid, vr);
        tile_put<P, PARTS>(kt[1], tid, kr1);
        tile_put<P, PARTS>(vt[1], tid, vr1);
    }
    __syncthreads();
    row_frags_lds<P>(kt[0], l32, hi, fk);

    f16v o[G::NPT];
#pragma unroll
    for (int pt = 0; pt < G::NPT; ++pt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[pt][v] = 0.f;
    float m_ref = -INFINITY, l_run = 0.f;                            // l_run: this lane's keys only
    const float slack = RESCALE_SLACK / c;
    int cur = 0, nxt = 1, nn = 2;
    MaskRegs mk = {};
    if (MASKED && n > 0 && entry_class(e0, piece + wave) != BLOCK_CLEAR) load_mask<true, RAGGED>(a, j, entry_tile(e0) * 32, hi, mk);
    // keep words drawn ahead of this launch are fetched a tile early: at the place of their
    // use the load would stand between the scores and their exponentials
    uint32_t word_ahead = 0;
    if (key.thr && n > 0 && entry_tile(e0) < a.keep_tiles_ready) word_ahead = a.keep[(size_t)row * pitch + entry_tile(e0)];
    // RAGGED: a score row starts anywhere in a Philox group of 8 when K is not a multiple of 8.  The bits of a tile are
    // then cut out of five groups, the first of which the tile before has drawn as its last (`carry`).
    const uint64_t e_row = (uint64_t)row * (unsigned)a.K;
    const uint32_t shift = (uint32_t)e_row & 7u;
    uint32_t carry = 0, carry_tile = ~0u;
    wait_loads();

    for (unsigned i = 0; i < longest; ++i) {
        const uint32_t e3 = live_entry<MASKED>(live, begin + i + 3);
        const unsigned t = entry_tile(e0);
        const bool from_mask = MASKED && entry_class(e0, piece + wave) != BLOCK_CLEAR;
        const bool fetch = i + 2 < n;
        const uint32_t word_ready = word_ahead;
        if (key.thr && i + 1 < n && entry_tile(e1) < a.keep_tiles_ready)
            word_ahead = a.keep[(size_t)row * pitch + entry_tile(e1)];
        if (fetch) {
            tiles_k.fetch(a.k, h, b, entry_tile(e2), a.K, tid, kr);
            tiles_v.fetch(a.v, h, b, entry_tile(e2), a.K, tid, vr);
        }
        if (working && (PARTS == 1 || i < n)) {
        f16v s;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.f;
        if (from_mask) start_from_mask(mk, s);
        if (MASKED && i + 1 < n && entry_class(e1, piece + wave) != BLOCK_CLEAR) load_mask<true, RAGGED>(a, j, entry_tile(e1) * 32, hi, mk);
#pragma unroll
        for (int ks = 0; ks < G::NKS; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(fk[ks], fq[ks], s, 0, 0, 0);
        // fragments for the second product of this tile and the first of the next
        h8 va[2][G::NPT];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt) va[st][pt] = tr_frag<P>(vt[cur], pt * 32, st, lane);
        row_frags_lds<P>(kt[nxt], l32, hi, fk);
        if (RAGGED && t * 32 + 32 > (unsigned)a.K) drop_past_end(s, t * 32, a.K, hi);

        // keep bits of the 32 scores (this query, keys of tile t): each half of the
        // wave draws two of the four groups of 8 and the halves trade them
        uint32_t word = 0xffffffffu;
        if (key.thr && t < a.keep_tiles_ready) {
            word = word_ready;                                       // drawn ahead of this launch
        } else if (RAGGED && key.thr) {
            const uint64_t g0 = (e_row >> 3) + 4 * t;
            if (carry_tile != t) carry = keep8(philox_group_dev(key, g0), key.thr);
            const uint32_t mine = keep8(philox_group_dev(key, g0 + 1 + 2 * hi), key.thr) |
                                  (keep8(philox_group_dev(key, g0 + 2 + 2 * hi), key.thr) << 8);
            const auto both = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
            word = __builtin_amdgcn_alignbit(both[1] >> 8, carry | (both[0] << 8) | (both[1] << 24), shift);
            carry = both[1] >> 8; carry_tile = t + 1;
        } else if (key.thr) {
            const uint64_t g0 = (uint64_t)row * (a.K / 8) + 4 * t + 2 * hi;
            const uint32_t mine = keep8(philox_group_dev(key, g0), key.thr) |
                                  (keep8(philox_group_dev(key, g0 + 1), key.thr) << 8);
            // v_permlane32_swap on two copies: [0] holds the lower half's value in both halves
            // of the wave, [1] the upper half's
            const auto both = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);
            word = both[0] | (both[1] << 16);
        }
        if (hi == 0 && mine_ && t >= a.keep_tiles_ready) a.keep[(size_t)row * pitch + t] = word;
        const uint32_t nib = word >> (hi * 4);                       // bit reg_pos(v, 0) of nib = keep of register v

        // Running softmax with a reference value per query that trails the running
        // maximum by up to RESCALE_SLACK (in log2 units): the accumulators are only
        // rescaled when some query of the wave outgrows its reference by more, which
        // after the first tiles is rare.  Scores and reference are in raw units.
        // The exponentials are taken against the reference as it stands, beside the search
        // for the tile's maximum rather than behind it (the chain maximum -> exchange between
        // the wave's halves -> vote -> exponentials left the wave with nothing to issue), and
        // again in the rare case that the reference moves.
        float ex[16];
        {
            const float mc0 = m_ref == -INFINITY ? 0.f : -m_ref * c;
#pragma unroll
            for (int v = 0; v < 16; ++v) ex[v] = __builtin_amdgcn_exp2f(fmaf(s[v], c, mc0));
        }
        float mt = s[0];
#pragma unroll
        for (int v = 1; v < 16; ++v) mt = fmaxf(mt, s[v]);
        {
            const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
            mt = fmaxf(__uint_as_float(both[0]), __uint_as_float(both[1]));
        }
        if (__builtin_amdgcn_ballot_w64(mt > m_ref + slack) != 0) {
            const float m_new = fmaxf(m_ref, mt);
            // (masked: a query that has seen no key yet has nothing to rescale; the
            // difference of its two infinities is not a number)
            const float corr = (MASKED && m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f((m_ref - m_new) * c);
            m_ref = m_new;
            l_run *= corr;
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[pt][v] *= corr;
            // (masked: a query whose keys so far are all masked out has no reference yet)
            const float mc = m_ref == -INFINITY ? 0.f : -m_ref * c;
#pragma unroll
            for (int v = 0; v < 16; ++v) ex[v] = __builtin_amdgcn_exp2f(fmaf(s[v], c, mc));
        }
        h8 pb[2];
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = ex[v];
        {   // four partial sums: a single one would be a chain of 16 dependent additions
            float l4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < 16; ++v) l4[v & 3] += s[v];
            l_run += (l4[0] + l4[1]) + (l4[2] + l4[3]);
        }
        each<16>([&](auto V) __attribute__((always_inline)) { constexpr int v = V; s[v] = keep_probability<reg_pos(v, 0)>(s[v], nib); });
#pragma unroll
        for (int v = 0; v < 16; ++v) pb[v >> 3][v & 7] = (half_t)s[v];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt)
                o[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[st][pt], pb[st], o[pt], 0, 0, 0);
        }
        if (fetch) {
            tile_put<P, PARTS>(kt[nn], tid, kr);
            tile_put<P, PARTS>(vt[nn], tid, vr);
        }
        __syncthreads();
        const int x = cur; cur = nxt; nxt = nn; nn = x;
        e0 = e1; e1 = e2; e2 = e3;
    }
    [[maybe_unused]] float* left = nullptr;
    if constexpr (PARTS > 1) {
        // (the tiles' places are free)
        static_assert(Place<PARTS>::WAVES * G::NPT * 16 * 64 * sizeof(float) <= sizeof(kt_), "two waves' accumulators");
        left = reinterpret_cast<float*>(kt_) + wave * (G::NPT * 16 * 64);
        float* const stats = reinterpret_cast<float*>(vt_) + wave * 128;
        if (at.half) {
            leave(left, lane, o);
            stats[lane] = m_ref;
            stats[64 + lane] = l_run;
        }
        __syncthreads();
        if (at.half) return;
        const float m1 = stats[lane], m_new = fmaxf(m_ref, m1);
        // (a half that has seen no key of this query has nothing, and no reference)
        const float mine = m_ref == -INFINITY ? (m_new == -INFINITY ? 1.f : 0.f) : __builtin_amdgcn_exp2f((m_ref - m_new) * c);
        const float theirs = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m1 - m_new) * c);
        l_run = l_run * mine + stats[64 + lane] * theirs;
        collect(left, lane, o, mine, theirs);
        m_ref = m_new;
    }
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const int w = __builtin_amdgcn_readfirstlane(wave);
    half_t* const out = PARTS > 1 ? reinterpret_cast<half_t*>(left) : w < 2 ? kt[w] : vt[w - 2];
    store_rows<P, RAGGED>(a.o, h, b, qb * QB + (piece + w) * 32, a.J, lane, o, 1.0f / l_tot, out, nullptr);
    if (mine_ && hi == 0) a.lse[row] = m_ref * c + __builtin_amdgcn_logf(l_tot);
}
template <int P, bool MASKED, bool RAGGED>
__global__ __launch_bounds__(256) void k_mha_fwd(AttnArgs a, PhiloxKey key_) {
    mha_fwd<P, MASKED, RAGGED, 1>(a, key_);
}
template <int P, bool MASKED, bool RAGGED>
__global__ __launch_bounds__(256) void k_mha_fwd_halves(AttnArgs a, PhiloxKey key_) {
    mha_fwd<P, MASKED, RAGGED, 2>(a, key_);
}

// ---------------------------------------------------------------------------
// backward, dQ.  grid = H * B * ceil(J / 128); wave = 32 queries.
// ---------------------------------------------------------------------------
template <int P, bool MASKED, bool RAGGED, int PARTS>
__device__ __forceinline__ void mha_bwd_dq(const AttnArgs& a) {
    using G = Geo<P>;
    // Head size 128: with the key and value fragments of a whole tile in registers a tile ahead the kernel
    // needs 300 registers per lane and runs one wave per SIMD; read two k-slices ahead of their use instead,
    // it fits 256 and two waves share a SIMD.
    constexpr bool JIT = !MASKED;
    __shared__ __attribute__((aligned(16))) half_t kt_[PARTS][RING][G::TILE];
    __shared__ __attribute__((aligned(16))) half_t vt_[PARTS][RING][G::TILE];
    const Place<PARTS> at;
    const int tid = at.tid, lane = at.lane, wave = at.wave, l32 = lane & 31, hi = lane >> 5;
    half_t (*const kt)[G::TILE] = kt_[at.half];
    half_t (*const vt)[G::TILE] = vt_[at.half];
    const unsigned qblocks = RAGGED ? (a.J + QB - 1) / QB : a.J / QB;
    const unsigned lb = logical_block() / PARTS;
    const unsigned nt = RAGGED ? (a.K + 31) / 32 : a.K / 32, pitch = RAGGED ? keep_pitch(a.K) : nt;
    unsigned qb = lb % qblocks, hb = lb / qblocks;
    if (MASKED) masked_order(a.qlist, qblocks, nt, a.H * a.B, lb, qb, hb);
    const unsigned b = hb % a.B, h = hb / a.B;
    const int piece = PARTS > 1 ? (int)(logical_block() % PARTS) * Place<PARTS>::WAVES : 0;      // its first wave's, of the block's four
    const unsigned j_ = qb * QB + (piece + wave) * 32 + l32;
    const bool mine_ = !RAGGED || j_ < (unsigned)a.J;
    const unsigned j = RAGGED ? min(j_, (unsigned)a.J - 1) : j_;
    const bool working = !RAGGED || __builtin_amdgcn_readfirstlane((int)(qb * QB + (piece + wave) * 32)) < a.J;
    const unsigned row = (h * a.B + b) * a.J + j;
    const float c = a.alpha * LOG2E;
    const uint32_t* live = (MASKED && a.qlist) ? a.qlist + (size_t)qb * (nt + kListPad) : nullptr;
    const unsigned all = live ? live[0] : nt, longest = (all + PARTS - 1) / PARTS;
    // (the second half's begin behind the first's; of an odd number it has one less)
    const unsigned begin = at.half ? longest : 0, n = at.half ? all - longest : longest;
    uint32_t e0 = live_entry<MASKED>(live, begin), e1 = live_entry<MASKED>(live, begin + 1), e2 = live_entry<MASKED>(live, begin + 2);

    h8 fq[G::NKS], fdo[G::NKS], fk[G::NKS], fv[G::NKS], kr[G::VL * PARTS], vr[G::VL * PARTS];
    float dsum, lse;
    uint32_t word;
    Tiles<P, !MASKED && !RAGGED, RAGGED, PARTS> tiles_k(a.k, h, b, begin, tid), tiles_v(a.v, h, b, begin, tid);
    {   // the first two tiles, the rows of this lane's query and its statistics: all
        // loads in flight together
        h8 kr1[G::VL * PARTS], vr1[G::VL * PARTS], fo[G::NKS];
        tiles_k.fetch(a.k, h, b, entry_tile(e0), a.K, tid, kr);
        tiles_v.fetch(a.v, h, b, entry_tile(e0), a.K, tid, vr);
        tiles_k.fetch(a.k, h, b, entry_tile(e1), a.K, tid, kr1);
        tiles_v.fetch(a.v, h, b, entry_tile(e1), a.K, tid, vr1);
        row_frags<P>(a.q, h, b, j, hi, fq);
        row_frags<P>(a.d_o, h, b, j, hi, fdo);
        row_frags<P>(a.o, h, b, j, hi, fo);
        lse = a.lse[row];
        word = a.keep[(size_t)row * pitch + entry_tile(e0)];
        tile_put<P, PARTS>(kt[0], tid, kr);
        tile_put<P, PARTS>(vt[0], tid, vr);
        tile_put<P, PARTS>(kt[1], tid, kr1);
        tile_put<P, PARTS>(vt[1], tid, vr1);
        float part = 0.f;
#pragma unroll
        for (int ks = 0; ks < G::NKS; ++ks)
#pragma unroll
            for (int i = 0; i < 8; ++i) part += (float)fdo[ks][i] * (float)fo[ks][i];
        dsum = part + __shfl_xor(part, 32);
        if (hi == 0 && mine_ && !at.half) a.dsum[row] = dsum;
    }
    __syncthreads();
    if constexpr (!JIT) {
        row_frags_lds<P>(kt[0], l32, hi, fk);
        row_frags_lds<P>(vt[0], l32, hi, fv);
    }

    f16v dq[G::NPT];
#pragma unroll
    for (int pt = 0; pt < G::NPT; ++pt)
#pragma unroll
        for (int v = 0; v < 16; ++v) dq[pt][v] = 0.f;
    int cur = 0, nxt = 1, nn = 2;
    MaskRegs mk = {};
    if (MASKED && n > 0 && entry_class(e0, piece + wave) != BLOCK_CLEAR) load_mask<true, RAGGED>(a, j, entry_tile(e0) * 32, hi, mk);
    wait_loads();

    for (unsigned i = 0; i < longest; ++i) {
        const uint32_t e3 = live_entry<MASKED>(live, begin + i + 3);
        const bool from_mask = MASKED && entry_class(e0, piece + wave) != BLOCK_CLEAR;
        const bool fetch = i + 2 < n;
        if (fetch) {
            tiles_k.fetch(a.k, h, b, entry_tile(e2), a.K, tid, kr);
            tiles_v.fetch(a.v, h, b, entry_tile(e2), a.K, tid, vr);
        }
        const uint32_t wordn = i + 1 < n ? a.keep[(size_t)row * pitch + entry_tile(e1)] : 0u;
        if (working && (PARTS == 1 || i < n)) {
        f16v s, dp;
#pragma unroll
        for (int v = 0; v < 16; ++v) { s[v] = 0.f; dp[v] = 0.f; }
        if (from_mask) start_from_mask(mk, s);
        if (MASKED && i + 1 < n && entry_class(e1, piece + wave) != BLOCK_CLEAR) load_mask<true, RAGGED>(a, j, entry_tile(e1) * 32, hi, mk);
        if constexpr (JIT) {
            h8 ck[2], cv[2];
            ck[0] = *reinterpret_cast<const h8*>(kt[cur] + G::at(l32, hi));
            cv[0] = *reinterpret_cast<const h8*>(vt[cur] + G::at(l32, hi));
#pragma unroll
            for (int ks = 0; ks < G::NKS; ++ks) {
                if (ks + 1 < G::NKS) {
                    ck[(ks + 1) & 1] = *reinterpret_cast<const h8*>(kt[cur] + G::at(l32, 2 * (ks + 1) + hi));
                    cv[(ks + 1) & 1] = *reinterpret_cast<const h8*>(vt[cur] + G::at(l32, 2 * (ks + 1) + hi));
                }
                s = __builtin_amdgcn_mfma_f32_32x32x16_f16(ck[ks & 1], fq[ks], s, 0, 0, 0);
                dp = __builtin_amdgcn_mfma_f32_32x32x16_f16(cv[ks & 1], fdo[ks], dp, 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int ks = 0; ks < G::NKS; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(fk[ks], fq[ks], s, 0, 0, 0);
#pragma unroll
            for (int ks = 0; ks < G::NKS; ++ks) dp = __builtin_amdgcn_mfma_f32_32x32x16_f16(fv[ks], fdo[ks], dp, 0, 0, 0);
        }
        h8 ka[2][G::NPT];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt) ka[st][pt] = tr_frag<P>(kt[cur], pt * 32, st, lane);
        if constexpr (!JIT) {
            row_frags_lds<P>(kt[nxt], l32, hi, fk);
            row_frags_lds<P>(vt[nxt], l32, hi, fv);
        }
        if (RAGGED && entry_tile(e0) * 32 + 32 > (unsigned)a.K) drop_past_end(s, entry_tile(e0) * 32, a.K, hi);
        const uint32_t nib = word >> (hi * 4);
        // stage by stage over the 16 scores of the lane, so that consecutive
        // instructions do not depend on one another
        h8 ds[2];
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = fmaf(s[v], c, -lse);
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = __builtin_amdgcn_exp2f(s[v]);
#pragma unroll
        for (int v = 0; v < 16; ++v) dp[v] = keep_if(dp[v], nib, reg_pos(v, 0));
#pragma unroll
        for (int v = 0; v < 16; ++v) dp[v] -= dsum;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] *= dp[v];
#pragma unroll
        for (int v = 0; v < 16; ++v) ds[v >> 3][v & 7] = (half_t)s[v];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt)
                dq[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[st][pt], ds[st], dq[pt], 0, 0, 0);
        }
        if (fetch) {
            tile_put<P, PARTS>(kt[nn], tid, kr);
            tile_put<P, PARTS>(vt[nn], tid, vr);
        }
        word = wordn;
        __syncthreads();
        const int x = cur; cur = nxt; nxt = nn; nn = x;
        e0 = e1; e1 = e2; e2 = e3;
    }
    const int w = __builtin_amdgcn_readfirstlane(wave);
    half_t* out = w < 2 ? kt[w] : vt[w - 2];
    float* const sums = a.bias_q ? reinterpret_cast<float*>(PARTS > 1 ? vt_[0][2] : kt_[0][2]) : nullptr;       // (of 4 waves 64 * P bytes, a tile's)
    if constexpr (PARTS > 1) {
        // (the tiles' places are free)
        static_assert(Place<PARTS>::WAVES * G::NPT * 16 * 64 * sizeof(float) <= sizeof(kt_), "two waves' accumulators");
        float* const left = reinterpret_cast<float*>(kt_) + w * (G::NPT * 16 * 64);
        if (at.half) leave(left, lane, dq);
        __syncthreads();
        if (!at.half) collect(left, lane, dq, 1.f, 1.f);
        out = reinterpret_cast<half_t*>(left);
    }
    if (!at.half)
        store_rows<P, RAGGED>(a.dq, h, b, qb * QB + (piece + w) * 32, a.J, lane, dq, a.alpha, out,
                              sums ? sums + w * 4 * P : nullptr);
    if (!sums) return;
    __syncthreads();
    const unsigned part = (b * qblocks + qb) * PARTS + piece / Place<PARTS>::WAVES;
    if (threadIdx.x < P) a.bias_q[((size_t)h * (a.B * qblocks * PARTS) + part) * P + threadIdx.x] = column_sum<P, Place<PARTS>::WAVES>(sums, threadIdx.x);
}
template <int P, bool MASKED, bool RAGGED>
__global__ __launch_bounds__(256, !MASKED ? (P == 128 ? 2 : 3) : 1) void k_mha_bwd_dq(AttnArgs a) {
    mha_bwd_dq<P, MASKED, RAGGED, 1>(a);
}
template <int P, bool MASKED, bool RAGGED>
__global__ __launch_bounds__(256) void k_mha_bwd_dq_halves(AttnArgs a) {
    mha_bwd_dq<P, MASKED, RAGGED, 2>(a);
}

// ---------------------------------------------------------------------------
// backward, dK and dV.  grid = H * B * ceil(K / 128); wave = 32 keys.
// Per tile of 32 queries the workgroup stages Q, dO, the two row statistics and
// the keep words of its four key tiles in LDS.
// ---------------------------------------------------------------------------
template <int P>
struct KvStage {
    half_t q[Geo<P>::TILE];
    half_t d_o[Geo<P>::TILE];
    float lse[32];
    float dsum[32];
    uint32_t keep[4][32];         // [wave's key tile][query]
};

// acc += a b with acc in the accumulation registers, where the 128 of dK and dV at head size 128 leave the ordinary ones
// to everything that vector instructions work on.  The compiler does not see what this is: the two wait states that an
// operand written by a vector instruction needs are spelled out, and settle() stands between the last product and the
// first read of acc.
__device__ __forceinline__ void add_product(f16v& acc, h8 a, h8 b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// acc = a b and acc += a b with b in the accumulation registers and acc in the ordinary ones; nothing may read acc within
// the 18 wait states that follow.
__device__ __forceinline__ void set_product(f16v& acc, h8 a, h8 b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "a"(b));
}
__device__ __forceinline__ void add_product_v(f16v& acc, h8 a, h8 b) {
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "a"(b));
}
template <int N>
__device__ __forceinline__ void settle(f16v (&acc)[N]) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+a"(acc[i]));
}

template <int P, bool MASKED, bool RAGGED, int PARTS>
__device__ __forceinline__ void mha_bwd_dkv(const AttnArgs& a) {
    using G = Geo<P>;
    // Head size 128 has one wave per SIMD, in which the vector work on a tile and the products around it wait for one another
    // (4400 cycles a tile, of which the matrix pipe works 1024).  There the scores of a tile are formed during the vector
    // work on the one before it, a product for each element, dV and dK behind them; the fragments come from LDS a few
    // products ahead of their use, the tiles of queries from memory four tiles ahead.  The registers allow it with dK,
    // dV and the wave's own K and V in the accumulation half.  H 32, P 128, 4 x 2048: 1048 -> 759 us, of which 145 us lie
    // before and behind the tiles.  (Fragments all read a tile ahead: 44 loads a tile from scratch.  Tiles fetched
    // five ahead: 787 us.  With a mask the tiles are taken from a list and begin from mask values: as for head size 64,
    // where two waves per SIMD fill each other's gaps.)
    constexpr bool AHEAD = P == 128 && !MASKED;
    static_assert(PARTS == 1 || P == 64, "head size 128 has the registers of a whole SIMD");
    __shared__ __attribute__((aligned(16))) KvStage<P> stage_[PARTS][AHEAD ? 4 : RING];
    const Place<PARTS> at;
    const int tid = at.tid, lane = at.lane, l32 = lane & 31, hi = lane >> 5;
    const int piece = PARTS > 1 ? (int)(logical_block() % PARTS) * Place<PARTS>::WAVES : 0;      // its first wave's, of the block's four
    const int wave = piece + at.wave;                                // (of the block)
    KvStage<P>* const stage = stage_[at.half];
    const unsigned kblocks = RAGGED ? (a.K + QB - 1) / QB : a.K / QB;
    const unsigned lb = logical_block() / PARTS;
    const unsigned nq = RAGGED ? (a.J + 31) / 32 : a.J / 32, nkt = RAGGED ? keep_pitch(a.K) : a.K / 32;
    unsigned kb = lb % kblocks, hb = lb / kblocks;
    if (MASKED) masked_order(a.klist, kblocks, nq, a.H * a.B, lb, kb, hb);
    const unsigned b = hb % a.B, h = hb / a.B;
    const unsigned kpos_ = kb * QB + wave * 32 + l32;                // this lane's key
    const unsigned kpos = RAGGED ? min(kpos_, (unsigned)a.K - 1) : kpos_;
    const bool working = !RAGGED || __builtin_amdgcn_readfirstlane((int)(kb * QB + wave * 32)) < a.K;
    const unsigned row0 = (h * a.B + b) * a.J;                       // score row of query 0
    const float c = a.alpha * LOG2E;
    // the query tiles to walk: all of them, or those a mask leaves for these 128 keys
    const uint32_t* live = (MASKED && a.klist) ? a.klist + (size_t)kb * (nq + kListPad) : nullptr;
    const unsigned all = live ? live[0] : nq, longest = (all + PARTS - 1) / PARTS;
    const unsigned begin = at.half ? longest : 0, n = at.half ? all - longest : longest;
    uint32_t e0 = live_entry<MASKED>(live, begin), e1 = live_entry<MASKED>(live, begin + 1), e2 = live_entry<MASKED>(live, begin + 2);

    h8 fk[G::NKS], fv[G::NKS], fq[G::NKS], fdo[G::NKS];
    struct InFlight {             // one tile of queries on its way from memory
        h8 q[G::VL * PARTS], d_o[G::VL * PARTS];
        float stat;
        uint4 kw;
    };
    Tiles<P, !MASKED && !RAGGED, RAGGED, PARTS> tiles_q(a.q, h, b, begin, tid), tiles_do(a.d_o, h, b, begin, tid);
    auto fetch = [&](unsigned qt, InFlight& f) {
        tiles_q.fetch(a.q, h, b, qt, a.J, tid, f.q);
        tiles_do.fetch(a.d_o, h, b, qt, a.J, tid, f.d_o);
        const unsigned q = qt * 32 + (tid & 31);
        const unsigned r = row0 + (RAGGED ? min(q, (unsigned)a.J - 1) : q);
        // (a log-sum-exp of +inf: the probabilities of a query past the end are zero)
        if (tid < 32) f.stat = !RAGGED || q < (unsigned)a.J ? a.lse[r] : INFINITY;
        else if (tid < 64) f.stat = a.dsum[r];
        else if (tid < 96) f.kw = *reinterpret_cast<const uint4*>(a.keep + (size_t)r * nkt + kb * 4);
    };
    auto put = [&](KvStage<P>& sg, const InFlight& f) {
        tile_put<P, PARTS>(sg.q, tid, f.q);
        tile_put<P, PARTS>(sg.d_o, tid, f.d_o);
        if (tid < 32) sg.lse[tid] = f.stat;
        else if (tid < 64) sg.dsum[tid - 32] = f.stat;
        else if (tid < 96) {
            sg.keep[0][tid - 64] = f.kw.x; sg.keep[1][tid - 64] = f.kw.y;
            sg.keep[2][tid - 64] = f.kw.z; sg.keep[3][tid - 64] = f.kw.w;
        }
    };
    InFlight fl;
    fl.stat = 0.f; fl.kw = make_uint4(0, 0, 0, 0);
    f16v dk[G::NPT], dv[G::NPT];
#pragma unroll
    for (int pt = 0; pt < G::NPT; ++pt)
#pragma unroll
        for (int v = 0; v < 16; ++v) { dk[pt][v] = 0.f; dv[pt][v] = 0.f; }
    if constexpr (AHEAD) {
        // The tiles in turn, by addresses that move along (worked out for each tile they are a dozen 64-bit products in the
        // open), the last one again behind it.  Each lane brings one word besides: the lower half of wave w the keep words of
        // its keys, the upper halves the statistics, so that no branch has a load on its way kept until its end.
        const half_t* pq = a.q.p + (long)h * a.q.sh + (long)b * a.q.sb + (long)(tid / (P / 8)) * a.q.sr + tid % (P / 8) * 8;
        const half_t* pd_o = a.d_o.p + (long)h * a.d_o.sh + (long)b * a.d_o.sb + (long)(tid / (P / 8)) * a.d_o.sr + tid % (P / 8) * 8;
        const uint32_t* small = hi ? reinterpret_cast<const uint32_t*>(wave & 1 ? a.dsum : a.lse) + row0
                                   : a.keep + (size_t)row0 * nkt + kb * 4 + wave;
        const long small_row = hi ? 1 : nkt;
        if (!RAGGED) small += l32 * small_row;
        uint32_t* const small_to = hi ? reinterpret_cast<uint32_t*>(wave & 1 ? stage[0].dsum : stage[0].lse) + l32 : stage[0].keep[wave] + l32;
        unsigned upto = 0;
        struct Tile { h8 q[2], d_o[2]; uint32_t w; };
        auto bring = [&](Tile& f) __attribute__((always_inline)) {
            if (RAGGED) {
                const unsigned q = upto * 32 + l32, last = (unsigned)a.J - 1;
                tile_fetch<P, RAGGED>(a.q, h, b, upto * 32, a.J, tid, f.q);
                tile_fetch<P, RAGGED>(a.d_o, h, b, upto * 32, a.J, tid, f.d_o);
                f.w = small[min(q, last) * small_row];
                ++upto;
            } else {
                f.q[0] = *reinterpret_cast<const h8*>(pq);
                f.q[1] = *reinterpret_cast<const h8*>(pq + 16 * a.q.sr);
                f.d_o[0] = *reinterpret_cast<const h8*>(pd_o);
                f.d_o[1] = *reinterpret_cast<const h8*>(pd_o + 16 * a.d_o.sr);
                f.w = *small;
                const long on = ++upto < n ? 32 : 0;
                pq += on * a.q.sr;
                pd_o += on * a.d_o.sr;
                small += on * small_row;
            }
        };
        // Tile t into its stage.
        auto lay = [&](unsigned t, const Tile& f) __attribute__((always_inline)) {
            KvStage<P>& sg = stage[t & 3];
            tile_put<P>(sg.q, tid, f.q);
            tile_put<P>(sg.d_o, tid, f.d_o);
            // (a log-sum-exp of +inf: the probabilities of a query past the end are zero)
            const bool beyond = RAGGED && hi && !(wave & 1) && t * 32 + l32 >= (unsigned)a.J;
            small_to[(t & 3) * (sizeof(KvStage<P>) / 4)] = beyond ? 0x7F800000u : f.w;
        };
        Tile way;
        {
            Tile f1, f2;
            bring(way);
            bring(f1);
            bring(f2);
            row_frags<P>(a.k, h, b, kpos, hi, fk);
            row_frags<P>(a.v, h, b, kpos, hi, fv);
            lay(0, way);
            lay(1, f1);
            lay(2, f2);
        }
        __syncthreads();
        wait_loads();
#pragma unroll
        for (int ks = 0; ks < G::NKS; ++ks) asm volatile("" : "+a"(fk[ks]), "+a"(fv[ks]));
        bring(way);
        constexpr int NS = 4, NT = 5;
        h8 rq[NS], rd[NS], tr[8];       // fragments on their way: NS slices of the features, NT transposed ones
        auto slice = [&](const KvStage<P>& sg, int ks) __attribute__((always_inline)) {
            rq[ks % NS] = *reinterpret_cast<const h8*>(sg.q + Geo<P>::at(l32, 2 * ks + hi));
            rd[ks % NS] = *reinterpret_cast<const h8*>(sg.d_o + Geo<P>::at(l32, 2 * ks + hi));
        };
        // fragment f of the sixteen that dV and dK take: dO and Q in turn, feature tile f / 2 % NPT, half f / 8 of the queries
        auto turned = [&](const KvStage<P>& sg, int f) __attribute__((always_inline)) {
            tr[f & 7] = tr_frag<P>(f & 1 ? sg.q : sg.d_o, (f / 2 % G::NPT) * 32, f / (2 * G::NPT), lane);
        };
        f16v s0, dp0, s1, dp1;
        auto scores = [&](const KvStage<P>& next, auto V, f16v& sn, f16v& dpn) __attribute__((always_inline)) {      // product V
            constexpr int ks = V / 2;
            if constexpr (V == 0) set_product(sn, rq[0], fk[0]);
            else if constexpr (V == 1) set_product(dpn, rd[0], fv[0]);
            else if constexpr (V % 2 == 0) add_product_v(sn, rq[ks % NS], fk[ks]);
            else add_product_v(dpn, rd[ks % NS], fv[ks]);
            if constexpr (V % 2 == 1 && ks + NS < G::NKS) slice(next, ks + NS);
        };
        each<NS>([&](auto S) __attribute__((always_inline)) { slice(stage[0], S); });
        each<2 * G::NKS>([&](auto V) __attribute__((always_inline)) { scores(stage[0], V, s0, dp0); });
        each<NS>([&](auto S) __attribute__((always_inline)) { slice(stage[1], S); });
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(s0), "+v"(dp0));
        // Tile i, whose scores are (s, dp); those of tile i + 1 into (sn, dpn) (behind the last tile: of what lies there, unused).
        auto tile = [&](unsigned i, const f16v& s, const f16v& dp, f16v& sn, f16v& dpn) __attribute__((always_inline)) {
            const KvStage<P>&sg = stage[i & 3], &next = stage[(i + 1) & 3], &after = stage[(i + 2) & 3];
            if (working) {
                h8 pd[2], ds[2];
                float4 ls[2], dd[2];
                uint4 w[2];
                auto stats = [&](int q) __attribute__((always_inline)) {
                    ls[q & 1] = *reinterpret_cast<const float4*>(sg.lse + q * 8 + hi * 4);
                    dd[q & 1] = *reinterpret_cast<const float4*>(sg.dsum + q * 8 + hi * 4);
                    w[q & 1] = *reinterpret_cast<const uint4*>(sg.keep[wave] + q * 8 + hi * 4);
                };
                stats(0);
                float p[2];
                int keep[2];
                auto second = [&](auto V) __attribute__((always_inline)) {       // of element V: what follows its exponential
                    constexpr int v = V, q = v / 4, e = v % 4;
                    const float ddv = e == 0 ? dd[q & 1].x : e == 1 ? dd[q & 1].y : e == 2 ? dd[q & 1].z : dd[q & 1].w;
                    pd[v >> 3][v & 7] = (half_t)__int_as_float(__float_as_int(p[v & 1]) & keep[v & 1]);
                    ds[v >> 3][v & 7] = (half_t)(p[v & 1] * (__int_as_float(__float_as_int(dp[v]) & keep[v & 1]) - ddv));
                };
                each<16>([&](auto V) __attribute__((always_inline)) {
                    constexpr int v = V, q = v / 4, e = v % 4;
                    scores(next, V, sn, dpn);
                    if constexpr (e == 1 && q < 3) stats(q + 1);
                    if constexpr (v >= 16 - NT) turned(sg, v - 16 + NT);
                    if constexpr (v > 0) second(std::integral_constant<int, v - 1>{});
                    const float lsv = e == 0 ? ls[q & 1].x : e == 1 ? ls[q & 1].y : e == 2 ? ls[q & 1].z : ls[q & 1].w;
                    const uint32_t wv = e == 0 ? w[q & 1].x : e == 1 ? w[q & 1].y : e == 2 ? w[q & 1].z : w[q & 1].w;
                    p[v & 1] = __builtin_amdgcn_exp2f(fmaf(s[v], c, -lsv));
                    keep[v & 1] = __builtin_amdgcn_sbfe((int)wv, l32, 1);
                    __builtin_amdgcn_sched_barrier(0);
                });
                second(std::integral_constant<int, 15>{});
                each<4 * G::NPT>([&](auto F) __attribute__((always_inline)) {
                    constexpr int f = F, st = f / (2 * G::NPT), pt = f / 2 % G::NPT;
                    if constexpr (f + NT < 4 * G::NPT) turned(sg, f + NT);
                    if constexpr (f >= 2 && f % 2 == 0 && f / 2 <= NS) slice(after, f / 2 - 1);
                    if constexpr (f == 7) lay(i + 3, way);
                    if constexpr (f == 9) bring(way);
                    if constexpr (f & 1) add_product(dk[pt], tr[f & 7], ds[st]);
                    else add_product(dv[pt], tr[f & 7], pd[st]);
                    __builtin_amdgcn_sched_barrier(0);
                });
                asm volatile("" : "+v"(sn), "+v"(dpn));      // (theirs until the products have arrived, also where unused)
            }
            if (!working) {
                lay(i + 3, way);
                bring(way);
            }
            __syncthreads();
        };
        unsigned i = 0;
        do {
            tile(i, s0, dp0, s1, dp1);
            if (i + 1 < n) tile(i + 1, s1, dp1, s0, dp0);
            i += 2;
        } while (i < n);
        settle(dk);
        settle(dv);
    } else {
    {
        InFlight f1;
        f1.stat = 0.f; f1.kw = make_uint4(0, 0, 0, 0);
        fetch(entry_tile(e0), fl);
        fetch(entry_tile(e1), f1);
        row_frags<P>(a.k, h, b, kpos, hi, fk);
        row_frags<P>(a.v, h, b, kpos, hi, fv);
        put(stage[0], fl);
        put(stage[1], f1);
    }
    __syncthreads();
    row_frags_lds<P>(stage[0].q, l32, hi, fq);
    row_frags_lds<P>(stage[0].d_o, l32, hi, fdo);

    int cur = 0, nxt = 1, nn = 2;
    MaskRegs mk = {};
    if (MASKED && n > 0 && entry_class(e0, wave) != BLOCK_CLEAR) load_mask<false, RAGGED>(a, kpos, entry_tile(e0) * 32, hi, mk);
    wait_loads();

    for (unsigned i = 0; i < longest; ++i) {
        const uint32_t e3 = live_entry<MASKED>(live, begin + i + 3);
        const bool from_mask = MASKED && entry_class(e0, wave) != BLOCK_CLEAR;
        const bool more = i + 2 < n;
        if (more) fetch(entry_tile(e2), fl);
        const KvStage<P>& sg = stage[cur];
        if (working && (PARTS == 1 || i < n)) {
        f16v s, dp;
#pragma unroll
        for (int v = 0; v < 16; ++v) { s[v] = 0.f; dp[v] = 0.f; }
        if (from_mask) start_from_mask(mk, s);
        if (MASKED && i + 1 < n && entry_class(e1, wave) != BLOCK_CLEAR) load_mask<false, RAGGED>(a, kpos, entry_tile(e1) * 32, hi, mk);
#pragma unroll
        for (int ks = 0; ks < G::NKS; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(fq[ks], fk[ks], s, 0, 0, 0);
#pragma unroll
        for (int ks = 0; ks < G::NKS; ++ks) dp = __builtin_amdgcn_mfma_f32_32x32x16_f16(fdo[ks], fv[ks], dp, 0, 0, 0);
        h8 qa[2][G::NPT], da[2][G::NPT];
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt) {
                da[st][pt] = tr_frag<P>(sg.d_o, pt * 32, st, lane);
                qa[st][pt] = tr_frag<P>(sg.q, pt * 32, st, lane);
            }
        row_frags_lds<P>(stage[nxt].q, l32, hi, fq);
        row_frags_lds<P>(stage[nxt].d_o, l32, hi, fdo);
        // D[query, key]: lane = key, register v = query reg_pos(v, hi)
        h8 pd[2], ds[2];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 ls = *reinterpret_cast<const float4*>(sg.lse + q * 8 + hi * 4);
            const float4 dd = *reinterpret_cast<const float4*>(sg.dsum + q * 8 + hi * 4);
            const uint4 w = *reinterpret_cast<const uint4*>(sg.keep[wave] + q * 8 + hi * 4);
            const float lsv[4] = {ls.x, ls.y, ls.z, ls.w}, ddv[4] = {dd.x, dd.y, dd.z, dd.w};
            const uint32_t wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int v = q * 4 + e;
                const float p = __builtin_amdgcn_exp2f(fmaf(s[v], c, -lsv[e]));
                const int keep = __builtin_amdgcn_sbfe((int)wv[e], l32, 1);
                pd[v >> 3][v & 7] = (half_t)__int_as_float(__float_as_int(p) & keep);
                ds[v >> 3][v & 7] = (half_t)(p * (__int_as_float(__float_as_int(dp[v]) & keep) - ddv[e]));
            }
        }
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int pt = 0; pt < G::NPT; ++pt) {
                dv[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(da[st][pt], pd[st], dv[pt], 0, 0, 0);
                dk[pt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(qa[st][pt], ds[st], dk[pt], 0, 0, 0);
            }
        }
        if (more) put(stage[nn], fl);
        __syncthreads();
        const int x = cur; cur = nxt; nxt = nn; nn = x;
        e0 = e1; e1 = e2; e2 = e3;
    }
    }
    const int w = __builtin_amdgcn_readfirstlane(at.wave);
    half_t* tile = w < 2 ? stage[w].q : stage[w - 2].d_o;
    float *sums_k = reinterpret_cast<float*>(stage_[0][2].q), *sums_v = reinterpret_cast<float*>(stage_[0][2].d_o);   // (of 4 waves 64 * P bytes, a tile's)
    if constexpr (PARTS > 1) {
        // (all stages are free: what the second half leaves lies from the first on, a wave's rows go out by way of its own place
        // there, and the sums lie behind)
        constexpr int LEFT = 2 * G::NPT * 16 * 64;
        static_assert((2 * LEFT + 2 * 16 * P) * sizeof(float) <= sizeof(stage_), "two waves' accumulators and sums");
        float* const first = reinterpret_cast<float*>(&stage_[0][0]);
        float* const left = first + w * LEFT;
        if (at.half) { leave(left, lane, dk); leave(left + LEFT / 2, lane, dv); }
        __syncthreads();
        if (!at.half) { collect(left, lane, dk, 1.f, 1.f); collect(left + LEFT / 2, lane, dv, 1.f, 1.f); }
        tile = reinterpret_cast<half_t*>(left);
        sums_k = first + 2 * LEFT;
        sums_v = sums_k + 16 * P;
    }
    if (!at.half) {
        store_rows<P, RAGGED>(a.dk, h, b, kb * QB + (piece + w) * 32, a.K, lane, dk, a.alpha, tile, a.bias_kv ? sums_k + w * 4 * P : nullptr);
        store_rows<P, RAGGED>(a.dv, h, b, kb * QB + (piece + w) * 32, a.K, lane, dv, 1.0f, tile, a.bias_kv ? sums_v + w * 4 * P : nullptr);
    }
    if (!a.bias_kv) return;
    __syncthreads();
    const size_t ntc = (size_t)a.B * kblocks * PARTS, part = (size_t)h * ntc + (b * kblocks + kb) * PARTS + piece / Place<PARTS>::WAVES;
    const int to = threadIdx.x;
    if (to < 2 * P) a.bias_kv[((to < P ? 0 : (size_t)a.H * ntc) + part) * P + to % P] = column_sum<P, Place<PARTS>::WAVES>(to < P ? sums_k : sums_v, to % P);
}
template <int P, bool MASKED, bool RAGGED>
__global__ __launch_bounds__(256, (P == 64 && MASKED) ? 2 : 1) void k_mha_bwd_dkv(AttnArgs a) {
    mha_bwd_dkv<P, MASKED, RAGGED, 1>(a);
}
template <int P, bool MASKED, bool RAGGED>
__global__ __launch_bounds__(256, MASKED && RAGGED ? 2 : 1) void k_mha_bwd_dkv_halves(AttnArgs a) {
    mha_bwd_dkv<P, MASKED, RAGGED, 2>(a);
}

// Whether the kernels have to watch the ends of the sequences.
bool ragged(const AttnArgs& a) { return a.J % QB != 0 || a.K % QB != 0; }

// 8-byte loads of four mask values along whichever dim is contiguous; the ragged kernels look at the strides themselves
bool mask_ok(const AttnArgs& a) {
    if (!a.amask) return true;
    if (ragged(a)) return (reinterpret_cast<uintptr_t>(a.amask) & (a.am_sk % 4 == 0 || a.am_sj % 4 == 0 ? 7 : 1)) == 0;
    if ((reinterpret_cast<uintptr_t>(a.amask) & 7) != 0) return false;
    if (a.am_sk == 1) return a.am_sj % 4 == 0;
    if (a.am_sj == 1) return a.am_sk % 4 == 0;
    return true;
}

bool side_ok(const AttnSide& s) {
    return s.p && (reinterpret_cast<uintptr_t>(s.p) & 15) == 0 && s.sh % 8 == 0 && s.sb % 8 == 0 && s.sr % 8 == 0;
}

}  // namespace

bool mha_shape_ok(long H, long B, long J, long K, long P) {
    if (P != 64 && P != 128) return false;
    return J > 0 && K > 0 && J < (1L << 21) && K < (1L << 21) && H * B * J <= 0x7fffffffL && H * B * K <= 0x7fffffffL;
}

size_t mha_stat_bytes(long H, long B, long J) { return (size_t)(H * B * J) * 2 * sizeof(float); }
size_t mha_keep_bytes(long H, long B, long J, long K) { return (size_t)(H * B * J) * mha_keep_pitch((unsigned)K) * 4; }

bool mha_forward_ok(const AttnArgs& a, int P) {
    return mha_shape_ok(a.H, a.B, a.J, a.K, P) && a.alpha > 0.f && side_ok(a.q) && side_ok(a.k) && side_ok(a.v) && side_ok(a.o) &&
           a.lse && a.keep && (reinterpret_cast<uintptr_t>(a.lse) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(a.keep) & 15) == 0 && mask_ok(a);
}

namespace {
size_t up16(size_t x) { return (x + 15) & ~(size_t)15; }
long tiles(long n) { return (n + 31) / 32; }
long blocks(long n) { return (n + QB - 1) / QB; }
size_t qlist_bytes(long J, long K) { return up16((size_t)blocks(J) * (size_t)(tiles(K) + kListPad) * 4); }
size_t klist_bytes(long J, long K) { return up16((size_t)blocks(K) * (size_t)(tiles(J) + kListPad) * 4); }
}  // namespace

size_t mha_mask_plan_bytes(long J, long K) {
    return qlist_bytes(J, K) + klist_bytes(J, K) + up16((size_t)tiles(J) * (size_t)tiles(K));
}

void launch_mha_mask_plan(AttnArgs& a, void* plan, bool rebuild, hipStream_t st) {
    uint32_t* qlist = (uint32_t*)plan;
    uint32_t* klist = (uint32_t*)((char*)plan + qlist_bytes(a.J, a.K));
    uint8_t* cls = (uint8_t*)plan + qlist_bytes(a.J, a.K) + klist_bytes(a.J, a.K);
    if (rebuild) {
        hipLaunchKernelGGL(k_mha_mask_classes, dim3((unsigned)(tiles(a.J) * tiles(a.K))), dim3(64), 0, st, a.amask,
                           a.am_sj, a.am_sk, a.J, a.K, cls);
        hipLaunchKernelGGL(k_mha_mask_lists, dim3((unsigned)(blocks(a.J) + blocks(a.K))), dim3(64), 0, st, cls, a.J, a.K, qlist,
                           klist);
    }
    a.qlist = qlist; a.klist = klist;
}

namespace {
// Calls fn with (head size, has a mask, ragged) as compile-time constants.
template <class Fn>
void for_variant(int P, const AttnArgs& a, Fn&& fn) {
    auto rag = [&](auto p, auto masked) {
        if (ragged(a)) fn(p, masked, std::true_type{});
        else fn(p, masked, std::false_type{});
    };
    auto msk = [&](auto p) {
        if (a.amask) rag(p, std::true_type{});
        else rag(p, std::false_type{});
    };
    if (P == 64) msk(std::integral_constant<int, 64>{});
    else msk(std::integral_constant<int, 128>{});
}

// A lone wave already keeps its SIMD issuing (1400 cycles a tile, 284 vector instructions), so that the halves give nothing where
// every CU has a workgroup: they are for launches that leave half of the CUs without one.  us of forward, dQ, and dK and dV with whole
// blocks and with halves, H 12, P 64: 1 x 1024 (96 blocks) 30.9, 24.0, 31.2 and 21.2, 17.4, 21.6, causal 36.6, 30.6, 41.0 and 24.7, 19.8,
// 25.1; 4 x 256 causal (96) 13.3, 12.4, 15.1 and 10.3, 9.7, 11.7; 3 x 300 (108) 13.6, 11.8, 15.9 and 10.3, 9.7, 11.8; 8 x 128 (96) 7.0, 7.4,
// 8.2 and 6.5, 7.1, 7.4.  Beyond: 8 x 256 on 512, H 16 (256) no difference, 13 x 201 (312) 15.0, 14.4, 16.4 and 17.4, 15.5, 20.2.
// With a mask a tile has more to wait for (its mask values, a list's next entry), and the second wave that the halves put on a SIMD fills that,
// whatever the mask leaves to do, as long as whole blocks are no more than one to a CU and there are tiles enough: then every kernel gains
// under every mask that was timed, with lists of tiles (a layer's) and without (an operator's).  us of whole blocks and of halves, 256 blocks of
// 32 tiles, H 4: causal 37.9, 31.8, 42.0 and 24.6, 22.1, 29.9; all zeros 39.7, 33.4, 42.6 and 33.5, 28.7, 36.2; a quarter of the keys gone 31.2,
// 26.6, 41.2 and 27.2, 24.0, 34.7; a window of a quarter 19.8, 18.0, 22.5 and 17.7, 16.9, 21.0; a slope 43.8, 42.4, 59.9 and 36.6, 33.2, 46.3; causal without
// lists 37.1, 38.0, 56.8 and 31.4, 31.8, 44.4.  192 blocks of 12 tiles: causal 17.8, 16.2, 20.1 and 14.9, 14.6, 17.7, a quarter gone 15.2, 13.2, 24.4 and
// 14.5, 14.2, 19.9.  With fewer tiles some lose: 256 blocks of 8, a window 12.8, 12.8, 13.9 and 13.2, 13.5, 14.8.
// Up to one and a half to a CU dK and dV lose too (320 blocks of 32 tiles, zeros 52.1 and 53.9, a window 26.7 and 31.0), forward and dQ of 32 tiles
// and more do not, but for masks that leave a block a few tiles.  us of forward and dQ in ten layers of 288 to 384 blocks, each timed alone by
// events: 3 x 1024, H 12, causal 60.1, 46.4 and 42.7, 33.2; zeros 60.7, 47.6 and 56.4, 43.7; a quarter gone 48.3, 37.8 and 46.2, 35.8; windows of a
// half, a quarter and an eighth 43.9, 33.9 and 36.9, 28.6; 33.1, 25.6 and 30.0, 23.4; 27.8, 21.9 and 26.4, 20.8; documents of 256 25.9, 19.9 and 26.5,
// 20.5; all of them between 0.65 and 1.07 (3 x 1000, H 12, documents, dQ 19.8 and 21.0), in the middle 0.93 and 0.92.
int parts(const AttnArgs& a, int P, long rows, long others, bool kv) {
    const long few = !a.amask || tiles(others) < 12 ? kFewBlocks : kv || tiles(others) < 32 ? 2 * kFewBlocks : 3 * kFewBlocks;
    return P == 64 && a.H * (long)a.B * blocks(rows) <= few && tiles(others) >= 4 ? 2 : 1;
}
}  // namespace

long mha_bias_rows_q(const AttnArgs& a, int P) { return a.B * blocks(a.J) * parts(a, P, a.J, a.K, false); }
long mha_bias_rows_kv(const AttnArgs& a, int P) { return a.B * blocks(a.K) * parts(a, P, a.K, a.J, true); }
size_t mha_bias_floats(long H, long B, long J, long K, long P) { return (size_t)(2 * H * P * B * (blocks(J) + 2 * blocks(K))); }

void launch_mha_forward(const AttnArgs& a, int P, PhiloxKey key, bool same_order, hipStream_t st) {
    if (!mha_forward_ok(a, P)) fail("attention forward: shape, strides or alignment not supported");
    const int n = same_order ? 1 : parts(a, P, a.J, a.K, false);
    dim3 grid((unsigned)(a.H * a.B * blocks(a.J) * n));
    for_variant(P, a, [&](auto p, auto masked, auto rag) {
        if constexpr (p() == 64) {
            if (n == 2) { hipLaunchKernelGGL((k_mha_fwd_halves<p(), masked(), rag()>), grid, dim3(256), 0, st, a, key); return; }
        }
        hipLaunchKernelGGL((k_mha_fwd<p(), masked(), rag()>), grid, dim3(256), 0, st, a, key);
    });
    check_launch("attention forward");
}

bool mha_backward_ok(const AttnArgs& a, int P) {
    return mha_forward_ok(a, P) && a.dsum && side_ok(a.d_o) && side_ok(a.dq) && side_ok(a.dk) && side_ok(a.dv);
}

void launch_mha_backward_dq(const AttnArgs& a, int P, hipStream_t st) {
    if (!mha_backward_ok(a, P)) fail("attention backward: shape, strides or alignment not supported");
    const int n = parts(a, P, a.J, a.K, false);
    dim3 grid((unsigned)(a.H * a.B * blocks(a.J) * n));
    for_variant(P, a, [&](auto p, auto masked, auto rag) {
        if constexpr (p() == 64) {
            if (n == 2) { hipLaunchKernelGGL((k_mha_bwd_dq_halves<p(), masked(), rag()>), grid, dim3(256), 0, st, a); return; }
        }
        hipLaunchKernelGGL((k_mha_bwd_dq<p(), masked(), rag()>), grid, dim3(256), 0, st, a);
    });
    check_launch("attention backward (dQ)");
}

void launch_mha_backward_dkv(const AttnArgs& a, int P, hipStream_t st) {
    if (!mha_backward_ok(a, P)) fail("attention backward: shape, strides or alignment not supported");
    const int n = parts(a, P, a.K, a.J, true);
    dim3 grid((unsigned)(a.H * a.B * blocks(a.K) * n));
    for_variant(P, a, [&](auto p, auto masked, auto rag) {
        if constexpr (p() == 64) {
            // (behind a mask and with two workgroups on a CU the kernel for any length at every length: without the end checks it takes 284
            // registers, one wave per SIMD, where this one takes 249; held to 256 it spills around the mask values.  us at 256 blocks of 32
            // tiles, all zeros, H 16: whole blocks 40.8, halves 49.1 with 284 registers, 36.2 now.  Alone on a CU the one without is the faster:
            // dQ, dK and dV of 1 x 2048 on 128, H 16, 60.6 and 67.1; 1 x 2048, H 8, 101 and 108; 2 x 512, H 16, 33.4 and 35.4)
            if constexpr (masked()) {
                if (n == 2 && a.H * (long)a.B * blocks(a.K) > kFewBlocks) {
                    hipLaunchKernelGGL((k_mha_bwd_dkv_halves<p(), true, true>), grid, dim3(256), 0, st, a);
                    return;
                }
            }
            if (n == 2) { hipLaunchKernelGGL((k_mha_bwd_dkv_halves<p(), masked(), rag()>), grid, dim3(256), 0, st, a); return; }
        }
        hipLaunchKernelGGL((k_mha_bwd_dkv<p(), masked(), rag()>), grid, dim3(256), 0, st, a);
    });
    check_launch("attention backward (dK, dV)");
}

}  // namespace sub
