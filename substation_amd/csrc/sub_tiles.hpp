// What the kernels that walk a launch's list of tiles share: the list, the way from a workgroup to its tiles, loads that
// go to LDS.
#pragma once

#include <algorithm>
#include <type_traits>

#include "sub_finish.hpp"
#include "sub_gemm.hpp"

namespace sub {

namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned lds_addr(const void* p) {
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// What lies behind `at` in LDS may have changed.
__device__ __forceinline__ void lds_fence(unsigned at) { asm volatile("" ::"v"(at) : "memory"); }

// 16 bytes per lane from buffer `r` into LDS at `lds` + 16 * lane; zeros from beyond the buffer's end.  Spelled out
// because of what the compiler makes of its own form of it: a transposing read from LDS, which it cannot tell from
// a read of bytes on their way, then waits for every load in flight, so that a step takes a round trip to memory
// (1100 cycles for 64 k of a 64 x 64 tile, where 500 do).  The waits that are needed stand in the loops.
// (All but voff are the same in every lane; m0 holds nothing else in these kernels.  In two parts, with an instruction
// of another kind between, where one is at hand: the second may not follow the first at once.)
__device__ __forceinline__ void load_to_lds_at(unsigned lds) {
    asm volatile("s_mov_b32 m0, %0" ::"s"((uint32_t)__builtin_amdgcn_readfirstlane((int)lds)));
}
__device__ __forceinline__ void load_to_lds_from(unsigned voff, u4v r, unsigned soff) {
    auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
    const u4v ru = {u(r[0]), u(r[1]), u(r[2]), u(r[3])};
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(ru), "s"(soff));
}
__device__ __forceinline__ void load_to_lds(unsigned lds, unsigned voff, u4v r) {
    auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
    const u4v ru = {u(r[0]), u(r[1]), u(r[2]), u(r[3])};
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 ::"s"(u(lds)), "v"(voff), "s"(ru));
}

// What the epilogue does after the scaling and the optional addend.
// EPI_RELU_DROPOUT_PRE: EPI_RELU_DROPOUT with the keep bits drawn ahead of the launch (GemmEpilogue::keep_words)
// EPI_GELU_DROPOUT: as EPI_RELU_DROPOUT with GELU; also stores the rounded sum before the activation
// (GemmArgs::pre_out, which the backward pass needs) and leaves the keep bits where the ReLU form leaves its gate bits.
// EPI_GELU_ALONE: without either, where no backward pass follows.
// EPI_GELU_GATE_COLSUM: the backward counterpart: out = keep bit ? gelu'(pre-activation) * product : 0, and column sums.
enum { EPI_PLAIN = 0, EPI_RELU_DROPOUT = 1, EPI_GATE_COLSUM = 2, EPI_RELU_DROPOUT_PRE = 3, EPI_GELU_DROPOUT = 4,
       EPI_GELU_GATE_COLSUM = 5, EPI_GELU_ALONE = 6 };

template <typename Key>
__device__ __forceinline__ PhiloxKey key_of(Key& from) {
    PhiloxKey k;
    k.k0 = from.k0; k.k1 = from.k1; k.site = from.site; k.step = from.step; k.thr = from.thr; k.step_dev = from.step_dev;
    return resolved(k);
}

// Eight halves (non-negative, or zero) where the bits of w's low byte are set, else zero; and the bits of those that are not zero.
__device__ __forceinline__ h8 keep8_of(h8 v, uint32_t w) {
    // bits 2 p and 2 p + 1 side by side, 16 apart, for every pair p; 0 - bit is a half's mask
    const uint32_t x = (w & 0xffu) | (w << 15);
    u4v r = __builtin_bit_cast(u4v, v);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const uint32_t b = (x >> (2 * p)) & 0x10001u;
        uint32_t m;
        asm("v_pk_sub_u16 %0, 0, %1" : "=v"(m) : "v"(b));
        r[p] &= m;
    }
    return __builtin_bit_cast(h8, r);
}
__device__ __forceinline__ uint32_t nonzero8(h8 v) {
    const u4v r = __builtin_bit_cast(u4v, v);
    uint32_t d = 0;
#pragma unroll
    for (int p = 3; p >= 0; --p) {
        uint32_t b;
        asm("v_pk_min_u16 %0, %1, %2" : "=v"(b) : "v"(r[p]), "v"(0x10001u));
        d = (d << 2) | b;
    }
    return (d | (d >> 15)) & 0xffu;
}

// One bit per output travels in canonical order (bit m N + n), N a multiple of 32.  Four lanes next to one another hold the 32
// columns of a word, each the byte of its 8 (a pack); of four packs, lane j of the four writes and reads the word of pack j.
__device__ __forceinline__ uint32_t quad_word(uint32_t byte, int lane) {
    uint32_t x = (byte & 0xffu) << (8 * (lane & 3));
    x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, true);      // the lane next to this one
    x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, true);      // the other two
    return x;
}
// Byte of pack j (its word is in lane j of the four).
template <int j>
__device__ __forceinline__ uint32_t quad_byte(uint32_t word, int lane) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)word, j * 0x55, 0xF, 0xF, true) >> (8 * (lane & 3));
}

// A pack of rounded sums through the activation; `keep`: its keep bits, on return the bits to leave for the backward pass.
// GELU: the keep bits themselves; ReLU: set where the result is positive.
template <int EPI>
__device__ __forceinline__ h8 act_forward(h8 v, uint32_t& keep) {
    if constexpr (EPI == EPI_GELU_DROPOUT || EPI == EPI_GELU_ALONE) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (half_t)gelu_fwd((float)v[e]);       // for every element, then selected: no branches
        return keep8_of(v, keep);
    } else {
        // what the bias-activation-dropout operator does to the rounded sum
        v = keep8_of(__builtin_elementwise_max(v, (h8)(half_t)0.0f), keep);     // ReLU, packed
        keep = nonzero8(v);
        return v;
    }
}
// A pack of the incoming gradient through the activation's backward pass, added to the column sums.  saved: GELU's
// pre-activation values; ReLU without bits: its output.
template <int EPI, bool BITS>
__device__ __forceinline__ h8 act_backward(h8 v, h8 saved, uint32_t bits, float (&colsum)[8]) {
    if constexpr (EPI == EPI_GELU_GATE_COLSUM) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (half_t)gelu_bwd((float)saved[e], (float)v[e]);
    }
    if constexpr (BITS) {
        v = keep8_of(v, bits);
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)saved[e] > 0.f ? v[e] : (half_t)0.0f;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) colsum[e] += (float)v[e];
    return v;
}

// Logical index of workgroup b of n such that the ones that the eight XCDs get in turn are consecutive on one XCD.
__device__ __forceinline__ unsigned xcd_order(unsigned b, unsigned n) {
    const unsigned q = n >> 3, r = n & 7u, x = b & 7u;
    return x * q + (x < r ? x : r) + (b >> 3);
}

template <typename T>
__device__ __forceinline__ T* uniform(T* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t up = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return reinterpret_cast<T*>(((uint64_t)up << 32) | lo);
}

struct NoJobs { int n = 0; };
template <int NP>
struct TileGroup {
    GemmArgs g[NP];
    unsigned end[NP];                 // products' tiles in the launch's list: those of product p end at end[p]
    unsigned second[NP];              // operands read the way of K2 (see k_gemm_ring)
    unsigned n = 0, workers = 0;      // products; workgroups that take tiles
    Schedule when;                    // (of several products)
    unsigned tail_groups = 0;
    // column sums of earlier launches, finished by the workgroups behind those
    typename std::conditional<NP == 1, NoJobs, FinishJobs>::type tail;
};
static_assert(sizeof(TileGroup<kMaxProducts>) <= 4096, "a kernel's arguments");

// (the launch's arguments where they lie: an index into them that is not a constant would otherwise have them copied
// into scratch memory)
typedef const __attribute__((address_space(4))) GemmArgs Args;

// The tiles of BM x BN outputs of a launch's products.
template <int BM, int BN, int NP>
struct TileList {
    typedef const __attribute__((address_space(4))) TileGroup<NP> Group;
    // One tile of the list.
    struct Tile {
        int p;                        // product
        int m0, n0, kt_begin, nkt;
        unsigned split, bz;
        long b0, b1, b2;
    };
    static __device__ __forceinline__ void locate(Group& G, unsigned id, Tile& t) {
        t.p = 0;
        unsigned first = 0;
        if constexpr (NP > 1) {
#pragma unroll
            for (unsigned i = 1; i < NP; ++i)
                if (G.n > i && id >= G.end[i - 1]) { t.p = (int)i; first = G.end[i - 1]; }
        }
        Args& g = G.g[t.p];
        id -= first;
        // (a division is some 30 instructions in front of a workgroup's first load: those of the common product are left out)
        const unsigned tiles_m = (unsigned)(g.M + BM - 1) / BM, tiles_n = (unsigned)(g.N + BN - 1) / BN;
        t.split = 0; t.kt_begin = 0;
        t.nkt = g.K0 * ((g.K1 + BK - 1) / BK);
        if (g.splits > 1) {
            const unsigned ns = (unsigned)g.splits, nkt = (unsigned)t.nkt, rest = id / ns;       // k-splits of one tile sit next to each other
            t.split = id - rest * ns; id = rest;
            t.kt_begin = (int)(nkt * t.split / ns);
            t.nkt = (int)(nkt * (t.split + 1) / ns) - t.kt_begin;
        }
        t.bz = 0; t.b0 = t.b1 = t.b2 = 0;
        if (g.nbatch > 1) {
            const unsigned per_batch = tiles_m * tiles_n;
            t.bz = id / per_batch;
            id -= t.bz * per_batch;
            const unsigned tq = t.bz / (unsigned)g.nb2;
            t.b2 = t.bz - tq * (unsigned)g.nb2; t.b0 = tq / (unsigned)g.nb1; t.b1 = tq - (unsigned)t.b0 * (unsigned)g.nb1;
        }
        // tiles that run together on an XCD share operand panels: groups of GM tile rows
        constexpr unsigned GM = BM > BN ? 4 : 8;
        const unsigned grp = tiles_m <= GM ? 0 : id / (GM * tiles_n), first_m = grp * GM, gsz = min(tiles_m - first_m, GM);
        const unsigned rr = id - grp * GM * tiles_n, col = gsz == GM ? rr / GM : rr / gsz;
        t.m0 = (int)((first_m + rr - col * gsz) * BM); t.n0 = (int)(col * BN);
    }
    // The tile of logical workgroup l of n in entry r of the launch's schedule, or in the next one that has any for it (r is moved
    // there).  One product: rounds of n, what is left of the last one goes to the workgroups from the other end.
    static __device__ __forceinline__ bool tile_of(Group& G, unsigned l, unsigned n, unsigned& r, Tile& t) {
        unsigned id;
        if constexpr (NP == 1) {
            const unsigned total = G.end[0];
            id = r * n + ((r + 1) * n <= total ? l : n - 1 - l);
            if (id >= total) return false;
        } else if (r < G.when.rounds) {
            id = r * n + l;
        } else {
            for (;; ++r) {
                const unsigned s = r - G.when.rounds;
                if (s >= G.when.n) return false;
                const unsigned j = l - G.when.part[s].worker;         // (wraps around below the first)
                if (j < G.when.part[s].count) { id = G.when.part[s].tile + j; break; }
            }
        }
        locate(G, id, t);
        return true;
    }
};

// ---- host --------------------------------------------------------------------------------------------------------------
inline long tiles_of(const GemmArgs& a, int splits, int bm, int bn) {
    return ((a.M + bm - 1) / bm) * (long)((a.N + bn - 1) / bn) * a.nbatch * splits;
}
inline long steps_of(const GemmArgs& a, int splits) { return ((long)a.K0 * ((a.K1 + BK - 1) / BK) + splits - 1) / splits; }

// The indices of n products, longest contraction first.
inline void longest_first(const TileProduct* p, int n, int (&order)[kMaxProducts]) {
    for (int i = 0; i < n; ++i) order[i] = i;
    std::stable_sort(order, order + n, [&](int x, int y) { return steps_of(p[x].a, p[x].a.splits) > steps_of(p[y].a, p[y].a.splits); });
}

// The list of a launch in tiles of form `form`, longest contractions first; `tail`: see launch_tiles.
template <int NP>
void list_tiles(TileGroup<NP>& G, const TileProduct* p, int n, int form, FinishJobs* tail, int& k1, int& k2) {
    const TileForm f = tile_form(form);
    const int bm = f.bm, bn = f.bn;
    const long places = 256L * f.per_cu;
    int order[kMaxProducts];
    if (n < 1 || n > NP || !orientations(p, n, k1, k2)) fail("gemm: these products do not share a launch");
    longest_first(p, n, order);
    long total = 0, len[NP], cnt[NP];
    for (int i = 0; i < n; ++i) {
        const TileProduct& q = p[order[i]];
        G.g[i] = q.a;
        G.second[i] = ((q.akc ? 1 : 0) | (q.bkc ? 2 : 0)) != k1;
        len[i] = steps_of(q.a, q.a.splits);
        total += cnt[i] = tiles_of(q.a, q.a.splits, bm, bn);
        if (total > 0x7fffffffL) fail("gemm: too many tiles");
        G.end[i] = (unsigned)total;
    }
    G.n = (unsigned)n;
    G.workers = (unsigned)std::min(total, places);
    if constexpr (NP > 1) schedule_tiles(len, cnt, n, G.workers, f.out_steps, G.when);
    if constexpr (NP > 1)
        if (tail && tail->n > 0) {
            const long groups = finish_groups(*tail);
            if (groups * tail->n <= 4096) { G.tail = *tail; G.tail_groups = (unsigned)groups; tail->n = 0; }
        }
}

}  // namespace

// One product with activation EPI in its epilogue, in tiles of form `form` (k_gemm_act.hip, compiled once for each EPI).
template <int EPI>
void launch_act(const TileProduct& p, int form, hipStream_t st);

}  // namespace sub
