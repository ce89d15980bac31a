// Contractions in tiles of 256 x 256 outputs: four waves, one per SIMD, each of which fetches, multiplies and stores.
//
// What bounds a large product here is power: a bare loop of v_mfma_f32_32x32x16_f16 on normally distributed operands runs
// at 1594 TFLOP/s, one of v_mfma_f32_16x16x32_f16 at 1847 (both at 2440 on zeros), so the smaller instruction is what this
// kernel is built on; and a wave that owns 128 x 128 outputs reads a third less from LDS than two of 128 x 64.  A wave's
// accumulators are the 256 accumulation registers of its lane.
//
// A step is 64 k of both operands, each of them in two halves of 128 rows, in two sets of buffers (128 KiB).  It goes by in
// four quarters of 32 matrix instructions (512 cycles), the products of one half of A and one of B:
//     quarter       0            1            2            3
//     multiplies    A0 B0        A0 B1        A1 B1        A1 B0
//     reads         B1 (and the  A1           A0 of the    B0 of the next step, as far as
//                   rest of B0)               next step    its registers are free
//     fetches       A0           B0           B1           A1       of the step after the next
// so that reads and fetches are spread evenly, the buffer that a fetch goes into was read a quarter or two before, and
// what is read was asked for five quarters before (2500 cycles).  One barrier per quarter.  A workgroup stays on its CU:
// the first two steps of its next tile are on their way while it stores a tile.
//
// us of products of normally distributed operands behind one another, before (eight waves of 128 x 64, v_mfma_f32_32x32x16_f16,
// two stages of LDS with every load of the next step in flight at a step's end) and now: 8192 x 16384 x 4096 (m x n x k) 903 ->
// 760 (1450 TFLOP/s; the power limit of the bare loop is 1594 and 1847), 4096 x 4096 x 1024 35.5 -> 31.5, 12288 x 4096 x 1024
// 99 -> 86.  A step takes 1.0 us on one CU (2400 of 2048 cycles) and 1.42 on all 256, the way into and out of a tile 10, of which
// 4 per further tile of a workgroup.  Three things were in the way at first, each worth a tenth of a step: addresses
// computed between the matrix instructions (a burst of twenty scalar instructions keeps them waiting for 60 cycles; now a
// half's resource is fixed for a tile and a step is one scalar offset), a branch around the wait at each quarter, and the
// epilogue's slab written and read in turn (now four of them, two ahead).
// 256 x 128 tiles in this manner take 60 us for 4096 x 2048 x 4096, as those of k_gemm_ring do: the operand fetch bounds them.
// Registers: 163 to 191 and the 256 accumulation registers, 188 to 206 with an activation, none of them spilled.  The instances of one
// product hold its arguments in scalar registers and spill 84 to 96 of those (to lanes of vector registers), with an activation
// 105 to 217, on the way into and out of a tile; those of several products 0, of two orientations 65 or 66.
#pragma once

#include "sub_tiles.hpp"

namespace sub {

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

// acc += b^T a, 16 x 16 outputs, 32 k.  Spelled out so that the accumulators stay in the accumulation registers (left to
// itself the compiler moves a quarter of them back and forth every step).  What it then does not know of: the wait between
// the last of these and the first read of an accumulator (Wide::settle).
__device__ __forceinline__ void mul(f4v& acc, h8 b, h8 a) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
}

// One of them, read where it is used: left to itself the compiler reads all 256 ahead, and spills them.
__device__ __forceinline__ float accumulator(float a) {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(a));
    return x;
}
__device__ __forceinline__ void mul_first(f4v& acc, h8 b, h8 a) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(b), "v"(a));
}

// A workgroup that multiplies nothing (see GemmSideJob): workgroup sb of nsb.
__device__ __forceinline__ void side_block(Args& g, unsigned sb, unsigned nsb) {
    const PhiloxKey key = key_of(g.side_key);
    const uint32_t nt = g.side_nk / 32, td = g.side_tiles_done, rows = g.side_rows;
    uint32_t* const keep = g.side_keep;
    // word w of rows * td is (row w / td, tile w % td); a thread walks w in steps of `stride`, carrying row
    // and tile along instead of dividing (a 64-bit division is as long as one of the word's four draws)
    const uint32_t stride = nsb * 256u, first = sb * 256u + threadIdx.x;
    const uint32_t srow = stride / td, st = stride - srow * td;
    uint32_t row = first / td, t = first - row * td;
    for (; row < rows; row += srow) {
        keep[(size_t)row * nt + t] = attention_keep_word(key, row, g.side_nk, t);
        t += st;
        if (t >= td) { t -= td; ++row; }
    }
}

// The fragments of an operand: 16 rows x 32 k, 8 consecutive k per lane, out of a half of ROWS rows, in the layout of DTile.
// ALONG_K: [row][64 k], else [64 k][row].
template <int ROWS, int ALONG_K>
struct Fragments {
    typedef __attribute__((address_space(3))) const h8* lds_h8;
    typedef s4v __attribute__((address_space(3))) * lds_s4;
    // ALONG_K: the order within a row is the same 16 rows further, and a slice of 32 k further the slot differs in bit 2: two
    // addresses, everything else is a constant behind one of them.  Else: rows 16 i further the address differs in bits 5 and 6.
    using Along = DTile<ROWS, true, 4, 16>;
    using Across = DTile<ROWS, false, 4, 16>;
    unsigned at[4];
    __device__ __forceinline__ void open(unsigned lds, int row0, int lane) {
        const int l = lane & 15, k = 8 * (lane >> 4) + (l >> 2), m = row0 + 4 * (l & 3);
        const unsigned b = 2u * (unsigned)(ALONG_K ? Along::kc_off(row0 + l, lane >> 4)
                                                   : k * ROWS + (((m >> 3) ^ Across::mc_swz(k)) << 3) + (m & 7));
#pragma unroll
        for (int x = 0; x < 4; ++x) at[x] = lds + (b ^ (unsigned)(x * (ALONG_K ? 64 : 32)));
    }
    __device__ __forceinline__ void move(unsigned by) {
#pragma unroll
        for (int x = 0; x < 4; ++x) at[x] += by;
    }
    // rows 16 i .. of the wave's, k-slice ks (0, 1), of the half `half` bytes behind the first
    __device__ __forceinline__ void read(h8& f, int i, int ks, unsigned half) const {
        if (ALONG_K) {
            f = *(lds_h8)(uintptr_t)(at[ks] + half + (unsigned)(i * 16 * BK * 2));
        } else {
            typedef short s8 __attribute__((ext_vector_type(8)));
            const unsigned p = at[i] + half + (unsigned)(ks * 32 * ROWS * 2);
            const s4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(uintptr_t)p);
            const s4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(uintptr_t)(p + 4 * ROWS * 2));
            const s8 r = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            f = __builtin_bit_cast(h8, r);
        }
    }
};

// 4 QM x 4 QN outputs per tile; a wave multiplies QM x QN of them in a quarter.
// K1, K2: as in k_gemm_ring.
template <int QM, int QN, int NP, int K1, int K2, int EPI>
struct Wide : TileList<4 * QM, 4 * QN, NP> {
    static constexpr int BM = 4 * QM, BN = 4 * QN, NW = 4;
    typedef TileList<BM, BN, NP> List;
    typedef typename List::Group Group;
    typedef typename List::Tile Tile;
    using List::tile_of;
    static constexpr int HM = 2 * QM, HN = 2 * QN;                     // rows of a half of A, of B
    static constexpr unsigned HA = HM * BK * 2, HB = HN * BK * 2;      // its bytes
    static constexpr unsigned AT_B = 4 * HA, AT_SLAB = AT_B + 4 * HB;
    static constexpr int SLAB = 16 * QN, SLABS = 4;                    // a wave's slabs of 16 output rows (elements)
    static constexpr unsigned BYTES = AT_SLAB + NW * SLABS * SLAB * 2;
    static constexpr int TA = QM / 16, TB = QN / 16, NM = TA * TB * 2; // fragments of a half, matrix instructions of a quarter
    static constexpr int LA = HM / (8 * NW), LB = HN / (8 * NW);       // a wave's loads of a half
    static constexpr int LATE = TB / 2;                                // fragments of B0 read in the quarter that uses them
    static constexpr int LPR = QN / 8, RPI = 64 / LPR, NI = 16 / RPI;  // lanes per output row, rows per store, stores per slab
    static constexpr int PACKS = 4 * TA * NI;                          // packs of 8 outputs that a lane stores
    static constexpr bool DRAWS = EPI == EPI_RELU_DROPOUT || EPI == EPI_GELU_DROPOUT || EPI == EPI_GELU_ALONE;
    static constexpr bool GATED = EPI == EPI_GATE_COLSUM || EPI == EPI_GELU_GATE_COLSUM;
    static constexpr bool READS = GATED || EPI == EPI_RELU_DROPOUT_PRE;          // bits of the outputs, as another launch left them
    static_assert(EPI == EPI_PLAIN || (PACKS == 32 && LPR == 8 && TA == 4), "32 packs of keep bits per lane, in the order of Epilogue::bits_part");

    // ---- what is fetched: the tiles' steps one after the other -----------------------------------------------------
    // (All of it in scalar registers but the offsets, and next to nothing to be computed from step to step: with one wave
    // per SIMD every instruction between two matrix instructions is one that these may wait for.)
    struct Stream {
        u4v ra[2], rb[2];             // the halves of A and of B, from an outer k's first element to the tile's last
        unsigned ka = 0, kb = 0;      // bytes from there to the next step
        unsigned step_a = 0, step_b = 0;
        unsigned to_a = 0, to_b = 0;  // where in LDS this wave's words go
        int left = 0, in_k1 = 0, p = 0;                     // steps of the tile, of those up to the end of an outer k
        unsigned round = 0;
        unsigned oa[LA], ob[LB];      // bytes from a half's first element to the lane's words
    };
    // (The range check takes a load's scalar offset, the place in k, from the half's size: that offset is never larger than it.  So
    // a second half that lies past the operand's last row is not one of no bytes: its rows are read as those of the first, and
    // multiplied into outputs that there are none of.)
    static __device__ __forceinline__ void aim(u4v (&r)[2], const half_t* first, long bytes, long half, bool second) {
        auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const long at = h && second ? half : 0;
            const uint64_t p = reinterpret_cast<uint64_t>(first) + (uint64_t)at;
            r[h] = u4v{u((uint32_t)p), u((uint32_t)(p >> 32)), u((uint32_t)(bytes - at)), 0x00020000u};
        }
    }
    static __device__ __forceinline__ void open(Group& G, Stream& s, unsigned l, unsigned n, int wave, int lane) {
        Tile t;
        s.ka = s.kb = 0;
        const bool more = tile_of(G, l, n, s.round, t);
        ++s.round;
        if (!more) {
            // nothing more: loads out of range, so that the count of loads in flight goes on
            s.ra[0][2] = s.ra[1][2] = s.rb[0][2] = s.rb[1][2] = 0u;
            s.step_a = s.step_b = 0;
            s.left = s.in_k1 = 0x7fffffff;
            return;
        }
        Args& g = G.g[t.p];
        s.p = t.p;
        const int per_k1 = (g.K1 + BK - 1) / BK, outer = g.K0 > 1 ? t.kt_begin / per_k1 : 0, kin = t.kt_begin - outer * per_k1;
        const int kc = K1 == K2 || !G.second[t.p] ? K1 : K2;
        s.step_a = (unsigned)(2 * BK * g.sAK1); s.step_b = (unsigned)(2 * BK * g.sBK1);
        s.ka = s.step_a * (unsigned)kin; s.kb = s.step_b * (unsigned)kin;
        const int rows = min(g.M - t.m0, BM), cols = min(g.N - t.n0, BN);
        aim(s.ra, g.A + t.b0 * g.sAb[0] + t.b1 * g.sAb[1] + t.b2 * g.sAb[2] + (long)t.m0 * g.sAM + outer * g.sAK0,
            2 * ((long)(rows - 1) * g.sAM + (long)(g.K1 - 1) * g.sAK1 + 1), 2 * HM * g.sAM, rows > HM);
        aim(s.rb, g.B + t.b0 * g.sBb[0] + t.b1 * g.sBb[1] + t.b2 * g.sBb[2] + (long)t.n0 * g.sBN + outer * g.sBK0,
            2 * ((long)(cols - 1) * g.sBN + (long)(g.K1 - 1) * g.sBK1 + 1), 2 * HN * g.sBN, cols > HN);
        if (kc & 1) DTile<HM, true, NW, 16>::offsets(s.oa, g.sAM, g.sAK1, wave, lane);
        else DTile<HM, false, NW, 16>::offsets(s.oa, g.sAM, g.sAK1, wave, lane);
        if (kc & 2) DTile<HN, true, NW, 16>::offsets(s.ob, g.sBN, g.sBK1, wave, lane);
        else DTile<HN, false, NW, 16>::offsets(s.ob, g.sBN, g.sBK1, wave, lane);
#pragma unroll
        for (int i = 0; i < LA; ++i) s.oa[i] *= 2;
#pragma unroll
        for (int i = 0; i < LB; ++i) s.ob[i] *= 2;
        s.left = t.nkt;
        s.in_k1 = per_k1 - kin;
    }
    // The next outer k of the tile.
    static __device__ __forceinline__ void next_outer(Group& G, Stream& s) {
        Args& g = G.g[s.p];
        auto ahead = [](u4v& r, long by) {
            const uint64_t p = (((uint64_t)r[1] << 32) | r[0]) + (uint64_t)by;
            r[0] = (uint32_t)p; r[1] = (uint32_t)(p >> 32);
        };
#pragma unroll
        for (int h = 0; h < 2; ++h) { ahead(s.ra[h], 2 * g.sAK0); ahead(s.rb[h], 2 * g.sBK0); }
        s.ka = s.kb = 0;
        s.in_k1 = (g.K1 + BK - 1) / BK;
    }
    // Load i of quarter q's half (in the order of the table above), of LA or LB, in two parts.
    template <int q, int i>
    static __device__ __forceinline__ void load_at(Group& G, Stream& s, unsigned l, unsigned n, int wave, int lane) {
        constexpr bool A = q == 0 || q == 3;
        constexpr int h = q >> 1;
        if constexpr (q == 0 && i == 0) if (s.left == 0) open(G, s, l, n, wave, lane);
        load_to_lds_at(A ? s.to_a + (unsigned)(h * HA + i * 1024) : s.to_b + (unsigned)(h * HB + i * 1024));
    }
    template <int q, int i>
    static __device__ __forceinline__ void load(Group& G, Stream& s) {
        constexpr bool A = q == 0 || q == 3;
        constexpr int h = q >> 1;
        // (the sum of a load's offsets is what is checked against the half's end)
        if constexpr (A) load_to_lds_from(s.oa[i], s.ra[h], s.ka);
        else load_to_lds_from(s.ob[i], s.rb[h], s.kb);
        if constexpr (q == 3 && i == LA - 1) {
            s.ka += s.step_a; s.kb += s.step_b;
            s.to_a ^= 2 * HA; s.to_b ^= 2 * HB;
            --s.left;
            if (--s.in_k1 == 0 && s.left > 0) next_outer(G, s);
        }
    }
    template <int q>
    static __device__ __forceinline__ void load_half(Group& G, Stream& s, unsigned l, unsigned n, int wave, int lane) {
        each<(q == 0 || q == 3 ? LA : LB)>([&](auto i) __attribute__((always_inline)) {
            load_at<q, decltype(i)::value>(G, s, l, n, wave, lane);
            asm volatile("s_nop 0");
            load<q, decltype(i)::value>(G, s);
        });
    }
    static __device__ __forceinline__ void whole_step(Group& G, Stream& s, unsigned l, unsigned n, int wave, int lane) {
        load_half<0>(G, s, l, n, wave, lane);
        load_half<1>(G, s, l, n, wave, lane);
        load_half<2>(G, s, l, n, wave, lane);
        load_half<3>(G, s, l, n, wave, lane);
    }

    // ---- between two quarters ---------------------------------------------------------------------------------------
    // This wave's reads are done and its loads of the half that is read next have landed (all but the VM latest ones;
    // landed: they have anyway); then, of all waves.
    template <int VM>
    static __device__ __forceinline__ void next_quarter(unsigned lds, bool landed) {
        lds_fence(lds);
        if (!landed) __builtin_amdgcn_s_waitcnt(waitcnt_vm(VM) & ~0x0F00);      // and lgkmcnt(0)
        else __builtin_amdgcn_s_waitcnt(0xC07F);      // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        lds_fence(lds);
        __builtin_amdgcn_sched_barrier(0);
    }

    // Keep bits of the packs that this lane stores, drawn while the matrix cores work: pack c in byte c of 32.
    struct Draw {
        PhiloxKey key;
        uint64_t group0 = 0;          // of pack 0
        long stride = 0;              // groups from a row to the next
        uint32_t word = 0, kb[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
        int c = 0;
        U4 v;
        uint32_t k0 = 0, k1 = 0;
        uint32_t tz = 0, tw = 0;
        // The draw of one pack in 22 parts, to be dealt out between the matrix instructions: the two multiplications of a
        // round take a quarter of the rate each, and as one part (five parts behind one another) they kept these waiting.
        static constexpr int PARTS = 22;
        __device__ __forceinline__ void part(int i) {
            if (i == 0) {
                // pack c: half of A, half of B, slab of 16 rows, 8 rows
                const int hb = (c >> 3) & 1, row = (c >> 4) * HM + ((c >> 1) & 3) * 16 + (c & 1) * RPI;
                const uint64_t g = group0 + (uint64_t)(row * stride) + (uint64_t)(hb * (HN / 8));
                v.x = (uint32_t)g; v.y = (uint32_t)(g >> 32); v.z = key.site; v.w = key.step;
                k0 = key.k0; k1 = key.k1;
            } else if (i == PARTS - 1) {
                word = (word >> 8) | (keep8(v, key.thr) << 24);
                if ((++c & 3) == 0) {
#pragma unroll
                    for (int w = 0; w < 7; ++w) kb[w] = kb[w + 1];
                    kb[7] = word;
                }
            } else if (i & 1) {
                uint32_t hi0;
                mulhilo(0xD2511F53u, v.x, hi0, tw);
                tz = xor3(hi0, v.w, k1);
            } else {
                uint32_t hi1, lo1;
                mulhilo(0xCD9E8D57u, v.z, hi1, lo1);
                v = U4{xor3(hi1, v.y, k0), lo1, tz, tw};
                k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
            }
        }
        __device__ __forceinline__ void one() {
#pragma unroll
            for (int i = 0; i < PARTS; ++i) part(i);
        }
    };

    // ---- a tile ------------------------------------------------------------------------------------------------------
    // Tiles from `t` on, the r-th, as long as they are of one product.  set: which buffers the next step is in.
    // landed: both halves of the first two steps have landed, of every wave.
    template <int AK, int BKC>
    static __device__ __forceinline__ bool consume(Group& G, Stream& s, unsigned l, unsigned n, unsigned& r, Tile& t, unsigned& set,
                                                   bool& landed, unsigned lds, half_t* slab, int wave, int lane) {
        const int wm = wave >> 1, wn = wave & 1, p = t.p;
        Fragments<HM, AK> FA;
        Fragments<HN, BKC> FB;
        FA.open(lds + set * 2 * HA, wm * QM, lane);
        FB.open(lds + AT_B + set * 2 * HB, wn * QN, lane);
        h8 a0[TA][2], a1[TA][2], b0[TB][2], b1[TB][2];
        f4v acc[2][2][TA][TB];
        Args& g = G.g[p];
        bool any;
        do {
            Epilogue e;
            e.open(g, t, wm, wn, wave, lane);
            lds_fence(lds);
#pragma unroll
            for (int i = 0; i < 2 * TA; ++i) FA.read(a0[i >> 1][i & 1], i >> 1, i & 1, 0);
#pragma unroll
            for (int j = 0; j < 2 * (TB - LATE); ++j) FB.read(b0[j >> 1][j & 1], j >> 1, j & 1, 0);
            // Quarter q: b by a into c, with the reads, loads and (draw) half of a pack's draw between.
            // Matrix instruction m: columns m / (2 TA), k-slice, rows m % TA.
            auto quarter = [&](auto q_, f4v (&c)[TA][TB], const h8 (&a)[TA][2], const h8 (&b)[TB][2], auto read, auto first, auto draw) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value;
                constexpr int VM = q == 0 || q == 1 ? 3 * LA + 2 * LB : 2 * LA + 3 * LB;
                constexpr int NL = q == 0 || q == 3 ? LA : LB;
                next_quarter<VM>(lds, decltype(first)::value && landed);
                each<NM>([&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value, col = m / (2 * TA), ks = (m / TA) & 1, row = m % TA;
                    constexpr bool loads = m % 4 == 3 && m / 4 < NL;
                    if constexpr (loads) load_at<q, m / 4>(G, s, l, n, wave, lane);
                    if constexpr (decltype(first)::value && ks == 0) mul_first(c[row][col], b[col][ks], a[row][ks]);
                    else mul(c[row][col], b[col][ks], a[row][ks]);
                    // three reads and a load in turn
                    if constexpr (m % 4 != 3) read(std::integral_constant<int, m / 4 * 3 + m % 4>{});
                    else if constexpr (loads) load<q, m / 4>(G, s);
                    if constexpr (decltype(draw)::value && m % 3 == 1) e.draw.part(q % 2 * 11 + m / 3);       // two packs a step
                    __builtin_amdgcn_sched_barrier(0);
                });
            };
            auto step = [&](auto first, auto draw) __attribute__((always_inline)) {
                quarter(std::integral_constant<int, 0>{}, acc[0][0], a0, b0, [&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value, F = 2 * LATE, f = m - F;
                    if constexpr (m < F) FB.read(b0[TB - LATE + m / 2][m & 1], TB - LATE + m / 2, m & 1, 0);
                    else if constexpr (f < 2 * TB) FB.read(b1[f / 2][f & 1], f / 2, f & 1, HB);
                }, first, draw);
                quarter(std::integral_constant<int, 1>{}, acc[0][1], a0, b1, [&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value;
                    if constexpr (m < 2 * TA) FA.read(a1[m / 2][m & 1], m / 2, m & 1, HA);
                }, first, draw);
                FA.move(set ? 0u - 2 * HA : 2 * HA);
                quarter(std::integral_constant<int, 2>{}, acc[1][1], a1, b1, [&](auto m_) __attribute__((always_inline)) {
                    constexpr int m = decltype(m_)::value;
                    if constexpr (m < 2 * TA) FA.read(a0[m / 2][m & 1], m / 2, m & 1, 0);
                }, first, draw);
                FB.move(set ? 0u - 2 * HB : 2 * HB);
                quarter(std::integral_constant<int, 3>{}, acc[1][0], a1, b0, [&](auto m_) __attribute__((always_inline)) {
                    // (a fragment's registers are free behind the TA instructions that use it)
                    constexpr int m = decltype(m_)::value, at = m / 3 * 4 + m % 3, f = (at + 1) / TA - 1;
                    if constexpr (m % 3 == 2 && f >= 0 && f < 2 * (TB - LATE)) FB.read(b0[f / 2][f & 1], f / 2, f & 1, 0);
                }, first, draw);
                set ^= 1u;
            };
            step(std::true_type{}, std::false_type{});
            int kt = 1;
            if constexpr (DRAWS) {
                const int from = e.draw.c ? t.nkt : t.nkt - PACKS / 2;
                for (; kt < from; ++kt) step(std::false_type{}, std::false_type{});
                for (; kt < t.nkt; ++kt) step(std::false_type{}, std::true_type{});
                while (e.draw.c < PACKS) e.draw.one();        // a contraction shorter than that
            } else {
                for (; kt < t.nkt; ++kt) step(std::false_type{}, std::false_type{});
            }
            // every load so far has landed before the first store: the count of what is in flight does not tell them apart
            lds_fence(lds);
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");          // (the last accumulators are written)
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
            __builtin_amdgcn_sched_barrier(0);
            landed = true;
            e.store(g, t, acc, slab, wm, wn, wave, lane);
            any = tile_of(G, l, n, ++r, t);
        } while (any && t.p == p);
        return any;
    }

    // ---- accumulators -> a slab of 16 rows in LDS -> 16-byte row segments -> memory ----------------------------------
    struct Epilogue {
        Draw draw;
        h8 bias8[2];                  // a bias row's 8 columns of this lane, in both halves of B
        uint32_t bits[READS ? 8 : 1];          // words of 4 packs each (quad_word)

        // The bits of a tile's outputs from the wave's first row and column on, and the lane's place in them: of 4 packs,
        // pack lane % 4 (two slabs of 16 rows, 8 rows at a time), the word of its columns.
        static __device__ __forceinline__ __amdgpu_buffer_rsrc_t bits_of(Args& g, const Tile& t, const uint32_t* p, int wm, int wn, int lane,
                                                                         unsigned (&at)[2]) {
            const int m_wave = t.m0 + wm * QM, n_wave = t.n0 + wn * QN, rows = g.M - m_wave, cols = g.N - n_wave, q = lane & 3;
            const uint64_t first = reinterpret_cast<uint64_t>(uniform(p)) + (uint64_t)(((long)m_wave * g.N + n_wave) >> 3);
            const long bytes = p && rows > 0 && cols > 0 ? ((long)(rows - 1) * g.N + cols) >> 3 : 0;
            auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
                at[hb] = (unsigned)(((q >> 1) * 16 + (q & 1) * RPI + lane / LPR) * (g.N >> 3) + (lane % LPR >> 2) * 4) |
                         ((lane % LPR >> 2) * 32 + hb * HN < cols ? 0u : 1u << 31);
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(first), 0, (int)u((uint32_t)(bytes < 0x7fffffffL ? bytes : 0x7fffffffL)), 0x00020000);
        }
        // word k: packs 4 k .. 4 k + 3
        static __device__ __forceinline__ unsigned bits_part(Args& g, int k) {
            return (unsigned)((k >> 2) * HM + (k & 1) * 32) * (unsigned)(g.N >> 3) + (unsigned)((k >> 1 & 1) * (HN >> 3));
        }

        // What it reads besides the accumulators, asked for ahead of the contraction.
        __device__ __forceinline__ void open(Args& g, const Tile& t, int wm, int wn, int wave, int lane) {
            if constexpr (EPI != EPI_PLAIN) {
                if (READS && (EPI != EPI_GATE_COLSUM || g.gate_bits)) {
                    unsigned at[2];
                    const __amdgpu_buffer_rsrc_t r = bits_of(g, t, GATED ? g.gate_bits : g.keep_words, wm, wn, lane, at);
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        bits[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)(at[k >> 1 & 1] + bits_part(g, k)), 0, 0);
                }
                if constexpr (DRAWS) {
                    draw.key = key_of(g.key);
                    const uint64_t row = (uint64_t)(t.m0 + wm * QM + lane / LPR);
                    draw.group0 = (row * (uint64_t)g.sCM + (uint64_t)(t.n0 + wn * QN + (lane % LPR) * 8)) >> 3;
                    draw.stride = g.sCM >> 3;
                    if (!draw.key.thr) {
                        // nothing is dropped
                        draw.c = PACKS;
#pragma unroll
                        for (int k = 0; k < 8; ++k) draw.kb[k] = ~0u;
                    }
                }
            }
        }

        __device__ __forceinline__ void store(Args& g, const Tile& t, f4v (&acc)[2][2][TA][TB], half_t* slab, int wm, int wn, int wave,
                                              int lane) {
            const int m_wave = t.m0 + wm * QM, n_wave = t.n0 + wn * QN;
            const float alpha = g.alpha;
            // (buffer accesses: what lies outside of the output is dropped by the range check instead of a branch per row)
            const int nl = (lane % LPR) * 8, row = lane / LPR, rows = g.M - m_wave, cols = g.N - n_wave;
            auto buffer = [&](const half_t* p, long s_row) __attribute__((always_inline)) {
                const uint64_t at = reinterpret_cast<uint64_t>(uniform(p + (long)m_wave * s_row + n_wave));
                const long bytes = rows > 0 && cols > 0 ? 2 * ((long)(rows - 1) * s_row + cols) : 0;
                auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
                return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at), 0, (int)u((uint32_t)(bytes < 0x7fffffffL ? bytes : 0x7fffffffL)), 0x00020000);
            };
            // (at: the lane's part of a word's place, `uni` the wave's.  Their sum is the vector offset, which alone is certain to
            // be checked: `uni` may lie beyond the buffer's size, and as a scalar offset would be taken from that.)
            auto get = [](__amdgpu_buffer_rsrc_t r, unsigned at, unsigned uni) __attribute__((always_inline)) {
                return __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(at + uni), 0, 0));
            };
            auto put = [](__amdgpu_buffer_rsrc_t r, unsigned at, unsigned uni, h8 v) __attribute__((always_inline)) {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, v), r, (int)(at + uni), 0, 0);
            };
            const long c_first = t.b0 * g.sCb[0] + t.b1 * g.sCb[1] + t.b2 * g.sCb[2];
            const __amdgpu_buffer_rsrc_t rc = buffer(g.C + c_first, g.sCM);
            // byte offset of pack (h, hb, i, it) in a tensor of rows s_row apart
            auto lane_part = [&](long s_row, int hb) __attribute__((always_inline)) {
                return (unsigned)(2 * (row * s_row + nl)) | (nl + hb * HN + 8 <= cols ? 0u : 1u << 31);
            };
            auto wave_part = [](long s_row, int h, int hb, int i, int it) __attribute__((always_inline)) {
                return (unsigned)(2 * (h * HM + i * 16 + it * RPI)) * (unsigned)s_row + (unsigned)(2 * hb * HN);
            };
            const unsigned at_c[2] = {lane_part(g.sCM, 0), lane_part(g.sCM, 1)};
            // in a slab: row lane % 16, 4 columns from 4 (lane / 16) on; row lane / LPR, the 8 columns from nl on
            const int to = (lane & 15) * QN + ((lane >> 4) & 1) * 4, to_swz = (((lane >> 5) ^ ((lane & 15) >> 1)) & (LPR - 1)) * 8;
            const int from = row * QN + (((lane % LPR) ^ (row >> 1)) & (LPR - 1)) * 8;
            float colsum[2][8];
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                for (int e = 0; e < 8; ++e) colsum[hb][e] = 0.f;
            uint32_t out_word = 0;
            unsigned at_o[2] = {0, 0};
            __amdgpu_buffer_rsrc_t ro = rc;
            if constexpr (EPI != EPI_PLAIN && !GATED) ro = bits_of(g, t, g.gate_bits_out, wm, wn, lane, at_o);     // (null: none)
            auto tile = [&](auto kind) __attribute__((always_inline)) {
                constexpr int ADD = decltype(kind)::value;          // 0 no addend, 1 a row, 2 a tensor, 3 the gate's values
                __amdgpu_buffer_rsrc_t rb = rc, rl = rc;
                h8 one[2], ad[4][NI];           // (addends are asked for four slabs ahead)
                if (ADD == 1 || ADD == 2) rb = buffer(g.bias + t.b0 * g.sbb[0] + t.b1 * g.sbb[1] + t.b2 * g.sbb[2], g.sbM);
                if (ADD == 3) rb = buffer(g.gate, g.sbM);
                if (EPI == EPI_GELU_DROPOUT) rl = buffer(g.pre_out, g.sCM);
                const unsigned at_b[2] = {lane_part(g.sbM, 0), lane_part(g.sbM, 1)};
                if (ADD == 1) {
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb) one[hb] = get(rb, at_b[hb], wave_part(0, 0, hb, 0, 0));
                }
                auto addends = [&](auto sl_) __attribute__((always_inline)) {
                    constexpr int sl = decltype(sl_)::value, h = sl / (2 * TA), hb = sl / TA % 2, i = sl % TA;
#pragma unroll
                    for (int it = 0; it < NI; ++it) ad[sl % 4][it] = get(rb, at_b[hb], wave_part(g.sbM, h, hb, i, it));
                };
                // Slab sl (16 rows of a quadrant) into one of four places; a 16-byte word's place in its row is xor-ed with half
                // the row's index, so that neither the writes (16 rows of 8 bytes) nor the reads (8 rows of 128) meet in a bank.
                auto fill = [&](auto sl_) __attribute__((always_inline)) {
                    constexpr int sl = decltype(sl_)::value, h = sl / (2 * TA), hb = sl / TA % 2, i = sl % TA;
                    float x[TB][4];
#pragma unroll
                    for (int j = 0; j < TB; ++j)
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[j][e] = accumulator(acc[h][hb][i][j][e]);
                    if (EPI == EPI_PLAIN && alpha != 1.0f) {
#pragma unroll
                        for (int j = 0; j < TB; ++j)
#pragma unroll
                            for (int e = 0; e < 4; ++e) x[j][e] *= alpha;
                    }
                    lds_fence(lds_addr(slab));
#pragma unroll
                    for (int j = 0; j < TB; ++j) {
                        h4 w;
#pragma unroll
                        for (int e = 0; e < 4; ++e) w[e] = (half_t)x[j][e];
                        *reinterpret_cast<h4*>(slab + (sl % SLABS) * SLAB + to + ((j * 16) ^ to_swz)) = w;
                    }
                    // (LDS operations of one wave execute in order: what other lanes wrote here is seen by the reads behind)
                    lds_fence(lds_addr(slab));
                };
                if constexpr (ADD >= 2) each<4>(addends);
                fill(std::integral_constant<int, 0>{});
                fill(std::integral_constant<int, 1>{});
                each<4 * TA>([&](auto sl_) __attribute__((always_inline)) {
                    constexpr int sl = decltype(sl_)::value, qd = sl / TA, h = qd >> 1, hb = qd & 1, i = sl % TA;
                    h8 vals[NI];
#pragma unroll
                    for (int it = 0; it < NI; ++it) vals[it] = *reinterpret_cast<const h8*>(slab + (sl % SLABS) * SLAB + it * RPI * QN + (from ^ (it * RPI / 2 * 8)));
                    if constexpr (sl + 2 < 4 * TA) fill(std::integral_constant<int, sl + 2>{});
                    {
                        each<NI>([&](auto it_) __attribute__((always_inline)) {
                            constexpr int it = decltype(it_)::value, c = sl * NI + it;
                            const unsigned at = at_c[hb], uni = wave_part(g.sCM, h, hb, i, it);
                            h8 val = vals[it];
                            // (packed half add: the same single rounding as through fp32)
                            if (ADD == 1) val = val + one[hb];
                            if (ADD == 2) val = val + ad[sl % 4][it];
                            if constexpr (GATED) {
                                uint32_t w = 0;
                                if constexpr (ADD == 0 || EPI == EPI_GELU_GATE_COLSUM) w = quad_byte<c & 3>(bits[c >> 2], lane);
                                // (rows beyond the last: nothing in the column sums; without bits, what is read there is zero)
                                w = h * HM + i * 16 + it * RPI + row < rows ? w : 0u;
                                val = act_backward<EPI, ADD == 0 || EPI == EPI_GELU_GATE_COLSUM>(val, ad[sl % 4][it], w, colsum[hb]);
                            }
                            if constexpr (EPI == EPI_GELU_DROPOUT) put(rl, at, uni, val);          // the pre-activation, for the backward pass
                            if constexpr (DRAWS || EPI == EPI_RELU_DROPOUT_PRE) {
                                uint32_t keep;
                                if constexpr (DRAWS) keep = draw.kb[c >> 2] >> (8 * (c & 3));
                                else keep = quad_byte<c & 3>(bits[c >> 2], lane);
                                val = act_forward<EPI>(val, keep);
                                if constexpr (EPI != EPI_GELU_ALONE) {
                                    const uint32_t word = quad_word(keep, lane);
                                    out_word = (lane & 3) == (c & 3) ? word : out_word;
                                }
                                if constexpr (EPI != EPI_GELU_ALONE && (c & 3) == 3)
                                    __builtin_amdgcn_raw_buffer_store_b32(out_word, ro, (int)(at_o[c >> 3 & 1] + bits_part(g, c >> 2)), 0, 0);
                            }
                            put(rc, at, uni, val);
                        });
                    }
                    if constexpr (ADD >= 2 && sl + 4 < 4 * TA) addends(std::integral_constant<int, sl + 4>{});
                });
            };
            if constexpr (GATED) {
                if (EPI == EPI_GELU_GATE_COLSUM || !g.gate_bits) tile(std::integral_constant<int, 3>{});
                else tile(std::integral_constant<int, 0>{});        // (a gated product has no addend)
            } else {
                if (!g.bias) tile(std::integral_constant<int, 0>{});
                else if (g.sbM == 0) tile(std::integral_constant<int, 1>{});
                else tile(std::integral_constant<int, 2>{});
            }
            if constexpr (GATED) {
                // lanes LPR apart hold the same 8 columns for other rows: add them up, then one fp32 row of partial sums
                // per wave (a finishing launch adds them up)
#pragma unroll
                for (int o = LPR; o < 64; o <<= 1)
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                        for (int e = 0; e < 8; ++e) colsum[hb][e] += __shfl_xor(colsum[hb][e], o);
                if (lane < LPR) {
#pragma unroll
                    for (int hb = 0; hb < 2; ++hb) {
                        if (hb * HN + nl >= cols) continue;
                        float* dst = g.colsum + ((long)(t.m0 / BM) * 2 + wm) * g.N + n_wave + hb * HN + lane * 8;
#pragma unroll
                        for (int e = 0; e < 8; ++e) dst[e] = colsum[hb][e];
                    }
                }
            }
        }
    };

    static __device__ __forceinline__ void run(Group& G, unsigned char* lds_) {
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const unsigned n = G.workers;
        if constexpr (NP > 1) if (blockIdx.x >= n) {
            // (behind the tiles: dispatched last, into places that they leave free or vacate first)
            const unsigned b = blockIdx.x - n;
            finish_block(G.tail.j[b / G.tail_groups], b % G.tail_groups, reinterpret_cast<float (*)[33]>(lds_));
            return;
        }
        if constexpr (NP == 1 && EPI == EPI_PLAIN) if (blockIdx.x >= n) {
            side_block(G.g[0], blockIdx.x - n, gridDim.x - n);
            return;
        }
        const unsigned l = xcd_order(blockIdx.x, n), lds = lds_addr(lds_);
        half_t* const slab = reinterpret_cast<half_t*>(lds_ + AT_SLAB) + wave * SLABS * SLAB;
        fetch_gemm_args(G.g[0]);
        Stream s;
        s.to_a = lds + (unsigned)(wave * LA * 1024); s.to_b = lds + AT_B + (unsigned)(wave * LB * 1024);
        open(G, s, l, n, wave, lane);
        whole_step(G, s, l, n, wave, lane);
        whole_step(G, s, l, n, wave, lane);
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(3 * LA + 3 * LB));      // A0 and B0 of the first step
        __builtin_amdgcn_s_barrier();
        Tile t;
        unsigned r = 0, set = 0;
        bool landed = false, any = tile_of(G, l, n, r, t);
        while (any) {
            if (K1 == K2 || !G.second[t.p]) any = consume<K1 & 1, (K1 >> 1)>(G, s, l, n, r, t, set, landed, lds, slab, wave, lane);
            else any = consume<K2 & 1, (K2 >> 1)>(G, s, l, n, r, t, set, landed, lds, slab, wave, lane);
        }
    }
};

template <int QM, int QN, int NP, int K1, int K2, int EPI>
__global__ __launch_bounds__(256, 1) void k_gemm_wide(TileGroup<NP>) {
    using W = Wide<QM, QN, NP, K1, K2, EPI>;
    __shared__ __attribute__((aligned(131072))) unsigned char lds[W::BYTES];
    W::run(*(typename W::Group*)__builtin_amdgcn_kernarg_segment_ptr(), lds);
}

// The kernel for the orientations of G's products (k1, k2: see list_tiles).
template <int NP, int EPI>
void launch_wide_as(const TileGroup<NP>& G, int k1, int k2, unsigned blocks, hipStream_t st) {
    const dim3 grid(blocks), block(256);
    if constexpr (NP > 1) if (k1 == 1 && k2 == 0) { hipLaunchKernelGGL((k_gemm_wide<64, 64, NP, 1, 0, EPI>), grid, block, 0, st, G); return; }
    if constexpr (NP > 1) if (k1 == 3 && k2 == 0) { hipLaunchKernelGGL((k_gemm_wide<64, 64, NP, 3, 0, EPI>), grid, block, 0, st, G); return; }
    if (k1 == 3) hipLaunchKernelGGL((k_gemm_wide<64, 64, NP, 3, 3, EPI>), grid, block, 0, st, G);
    else if (k1 == 2) hipLaunchKernelGGL((k_gemm_wide<64, 64, NP, 2, 2, EPI>), grid, block, 0, st, G);
    else if (k1 == 1) hipLaunchKernelGGL((k_gemm_wide<64, 64, NP, 1, 1, EPI>), grid, block, 0, st, G);
    else hipLaunchKernelGGL((k_gemm_wide<64, 64, NP, 0, 0, EPI>), grid, block, 0, st, G);
}

}  // namespace

}  // namespace sub
