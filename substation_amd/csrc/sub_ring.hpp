// Contractions in a ring of LDS stages with waves of their own for the fetching; one launch takes up to kMaxProducts products.
//
// What bounds a product here is how fast a CU draws its operands: 51 bytes a cycle of lines that its L2 has, 12 of lines
// that it has not, so about 31 where a fifth is missing (4096 x 1024 x 4096: 512 MiB drawn, 104 of them from beyond the L2s;
// its 36 us are what the fetch alone takes at those two rates).  A wave that issues an asynchronous load waits until the
// memory path has taken it, so when the multiplying waves fetched as well, a step of 64 k of a 128 x 128 tile took the
// cycles that its 32 KiB take (640 at best) plus the 512 of its matrix instructions.  Here four waves only fetch and the others
// only multiply, and a workgroup stays on its CU: while it writes one tile, the first stages of its next one are on their way.
// Tiles with remainders are read and written through range-checked buffers, so a 128 x 128 tile at the edge costs what
// one inside does (the kernel before predicated every load of such a product).  M = 2613 rows, us before and now:
// 768 x 3072 (n x k) 35 -> 21, 3072 x 768 21 -> 18.5, its weight gradient 42 -> 20.5; 64 rows x 768 x 768: 14 -> 6.4; 4096 x 1024 x
// 4096: 43 -> 35-37 (930 to 990 TFLOP/s, box to box).  4096 x 1024 x 1024, one tile of 16 steps per CU, takes 15 to 17 us.
// Registers without an activation: 72 to 168 a lane up to 128 x 128 tiles, 242 to 256 at 256 x 128, where the instance of data and weight
// gradients (two loop bodies) spills two of them (12 bytes of scratch) and that of one product with both operands across k one;
// the instances of one product hold its arguments in scalar registers and spill 26 to 36 of those, the ones of several
// products none.  With one: 85 to 212 up to 128 x 128 (128 x 64 with GELU, and 64 x 64 with GELU where no gradient is wanted: 20 bytes of
// scratch), 251 to 256 at 256 x 128, where GELU spills 2 to 7 (12 to 32 bytes; none where no gradient is wanted), ReLU's gate 44 to 50
// (180 to 204), GELU's backward form 56 to 61 (228 to 248), all in the epilogue; 27 to 39 scalar registers backward, 76 to 125 forward
// (the keys and constants of the draws).
#pragma once

#include "sub_tiles.hpp"

namespace sub {

namespace {

// NM matrix instructions with NR reads from LDS dealt out evenly in front of them (and NV vector instructions behind each).
template <int m, int NM, int NR, int NV = 0>
__device__ __forceinline__ void deal_reads() {
    if constexpr (m < NM) {
        constexpr int r = (NR * (m + 1)) / NM - (NR * m) / NM;
        if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if constexpr (NV > 0) __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
        deal_reads<m + 1, NM, NR, NV>();
    }
}

// 32 TM WM x 32 TN WN outputs per tile, WM x WN waves that multiply, NL that fetch, S stages of 64 k.
// K1, K2: which operands are contiguous along k (bit 0: A, bit 1: B), of products with `second` clear and set.
template <int TM, int TN, int WM, int WN, int NL, int S, int NP, int K1, int K2, int EPI = EPI_PLAIN>
struct Ring : TileList<32 * TM * WM, 32 * TN * WN, NP> {
    static constexpr int NC = WM * WN, BM = 32 * TM * WM, BN = 32 * TN * WN;
    typedef TileList<BM, BN, NP> List;
    typedef typename List::Group Group;
    typedef typename List::Tile Tile;
    using List::tile_of;
    static constexpr int STAGE = (BM + BN) * BK;
    static constexpr int PITCH = 32 * TN + 8, SLAB = 16 * PITCH;      // a wave's slab of 16 output rows
    static constexpr int HALVES = S * STAGE + NC * SLAB;
    static constexpr int LPR = 4 * TN, RPI = 64 / LPR;                // lanes per output row, rows per store
    using TAK = DTile<BM, true, NL>;
    using TAF = DTile<BM, false, NL>;
    using TBK = DTile<BN, true, NL>;
    using TBF = DTile<BN, false, NL>;
    static constexpr int LA = TAK::NV, LB = TBK::NV, L = LA + LB;     // loads per fetching wave and stage

    // ---- the fetching waves ---------------------------------------------------------------------------------------
    // One operand of the product at hand.
    template <int N>
    struct Operand {
        const half_t* p = nullptr;    // the next k-tile, within one outer k
        unsigned off[N];              // bytes from there to the lane's words
        unsigned past = 0;            // bit i: word i of the last k-tile of an outer k lies beyond K1
        long left = 0;                // bytes from p to the operand's last element within this outer k
        long step = 0, outer = 0;     // (in bytes)

        template <typename TK, typename TF>
        __device__ __forceinline__ void open(const half_t* first, bool kc, int rows, long s_row, int K1_, long s_k, long s_k0, int kin,
                                             int wave, int lane) {
            step = 2 * BK * s_k;
            outer = 2 * s_k0 - (long)((K1_ - 1) / BK) * step;
            left = 2 * ((long)(rows - 1) * s_row + (long)(K1_ - 1) * s_k + 1) - kin * step;
            p = uniform(first + (long)kin * BK * s_k);
            past = 0;
            if (kc) {
                TK::offsets(off, s_row, s_k, wave, lane);
                const int k_last = K1_ - (K1_ - 1) / BK * BK;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const int row = (wave * N + i) * 8 + (lane >> 3);
                    past |= ((((lane & 7) ^ (row ^ (row >> 3))) & 7) * 8 >= k_last ? 1u : 0u) << i;
                }
            } else {
                TF::offsets(off, s_row, s_k, wave, lane);       // (k beyond K1 lies beyond `left`)
            }
#pragma unroll
            for (int i = 0; i < N; ++i) off[i] *= 2;
        }
        __device__ __forceinline__ void issue(unsigned at, bool last_of_k1) {
            const uint64_t a = reinterpret_cast<uint64_t>(p);
            // (offsets stay below 2^31, see tiles_take: a word with that bit set is out of range)
            const u4v r = {(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)(left < 0x7fffffffL ? left : 0x7fffffffL), 0x00020000u};
            const unsigned none = last_of_k1 ? past : 0u;
#pragma unroll
            for (int i = 0; i < N; ++i) load_to_lds(at + (unsigned)(i * 1024), off[i] | (((none >> i) & 1u) << 31), r);
            const long by = last_of_k1 ? outer : step;
            p = reinterpret_cast<const half_t*>(a + by);
            left -= step;
        }
    };
    static __device__ __forceinline__ void fetch(Group& G, unsigned l, unsigned n, unsigned ring_at, int wave, int lane) {
        Operand<LA> oa;
        Operand<LB> ob;
        int left = 0, kin = 0, per_k1 = 1, stage = 0;
        bool more = true;
        long full_a = 0, full_b = 0;  // `left` at the start of an outer k
        unsigned round = 0, steps = 0;
        auto next_tile = [&]() {
            Tile t;
            more = tile_of(G, l, n, round, t);
            ++round;
            if (!more) { oa.left = oa.step = ob.left = ob.step = full_a = full_b = 0; left = 0x7fffffff; return; }
            Args& g = G.g[t.p];
            per_k1 = (g.K1 + BK - 1) / BK;
            const int outer = g.K0 > 1 ? t.kt_begin / per_k1 : 0;
            const long k0 = outer;
            kin = t.kt_begin - outer * per_k1;
            const int kc = K1 == K2 || !G.second[t.p] ? K1 : K2;
            oa.template open<TAK, TAF>(g.A + t.b0 * g.sAb[0] + t.b1 * g.sAb[1] + t.b2 * g.sAb[2] + (long)t.m0 * g.sAM + k0 * g.sAK0,
                                       kc & 1, g.M - t.m0, g.sAM, g.K1, g.sAK1, g.sAK0, kin, wave, lane);
            ob.template open<TBK, TBF>(g.B + t.b0 * g.sBb[0] + t.b1 * g.sBb[1] + t.b2 * g.sBb[2] + (long)t.n0 * g.sBN + k0 * g.sBK0,
                                       kc & 2, g.N - t.n0, g.sBN, g.K1, g.sBK1, g.sBK0, kin, wave, lane);
            full_a = oa.left + kin * oa.step;
            full_b = ob.left + kin * ob.step;
            left = t.nkt;
            steps += (unsigned)t.nkt;
        };
        // The next k-tile into the next stage.  Past the last one the loads are out of range: nothing is read, and the
        // count of loads in flight stays the same.
        auto issue = [&]() {
            if (left == 0) next_tile();
            const unsigned at = ring_at + (unsigned)(stage * STAGE * 2);
            const bool wrap = kin + 1 == per_k1;
            oa.issue(at + (unsigned)(wave * LA * 1024), wrap);
            ob.issue(at + (unsigned)(BM * BK * 2 + wave * LB * 1024), wrap);
            if (wrap) { oa.left = full_a; ob.left = full_b; }
            kin = wrap ? 0 : kin + 1;
            --left;
            stage = stage + 1 == S ? 0 : stage + 1;
        };
        // (the first step starts as soon as its stage has landed: the last stages are asked for behind that)
        constexpr int FIRST = S > 2 ? 2 : 1;
        for (int i = 0; i < FIRST; ++i) {
            if (left == 0) next_tile();
            if (more) issue();
        }
        if (more) __builtin_amdgcn_s_waitcnt(waitcnt_vm((FIRST - 1) * L));
        else __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
        __builtin_amdgcn_s_barrier();                 // step 0 has landed
        for (int i = FIRST; i < S && more; ++i) {
            if (left == 0) next_tile();
            if (more) issue();
        }
        if (!more) {
            // fewer steps than stages: all of them are on their way
            __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
            for (unsigned i = 0; i < steps; ++i) __builtin_amdgcn_s_barrier();
            return;
        }
        // (steps grows while tiles are found, which is ahead of this count)
        for (unsigned i = 0; i < steps; ++i) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm((S - 2) * L));
            __builtin_amdgcn_s_barrier();             // step i + 1 has landed, the fragments of step i are in registers
            issue();
        }
        __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    }

    // ---- the multiplying waves ------------------------------------------------------------------------------------
    // Tiles from `r` on as long as they are of product `p`; on entry step 0 of the first has landed, on return the barrier
    // behind the last one's last step has been passed.
    template <bool AKC, bool BKC>
    static __device__ __forceinline__ void consume(Group& G, unsigned l, unsigned n, unsigned& r, Tile& t, bool& any,
                                                   half_t* ring, unsigned ring_at, int& stage, int wave, int lane) {
        using TA = DTile<BM, AKC, NL>;
        using TB = DTile<BN, BKC, NL>;
        const int wm = wave / WN, wn = wave % WN;
        const int p = t.p;
        struct Slice { h8 a[TM], b[TN]; };            // the fragments of one k-slice of 16
        const int base_a = DTile<BM, true, NL>::kc_off(wm * TM * 32 + (lane & 31), lane >> 5);
        const int base_b = DTile<BN, true, NL>::kc_off(wn * TN * 32 + (lane & 31), lane >> 5);
        f16v acc[TM][TN];
        auto clear = [&]() {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
        };
        auto read = [&](Slice& f, int ks) {
            const half_t* sA = ring + stage * STAGE;
            const half_t* sB = sA + BM * BK;
            // (fragment addresses of an operand contiguous along k are formed from one register where they are used: left
            // alone the compiler keeps all of them, 24 registers of a 256 x 128 tile, across the loop)
            int ba = base_a, bb = base_b;
            asm volatile("" : "+v"(ba), "+v"(bb));
#pragma unroll
            for (int i = 0; i < TM; ++i) f.a[i] = AKC ? TA::frag_at(sA, ba, i, ks) : TA::frag(sA, (wm * TM + i) * 32, ks, lane);
#pragma unroll
            for (int j = 0; j < TN; ++j) f.b[j] = BKC ? TB::frag_at(sB, bb, j, ks) : TB::frag(sB, (wn * TN + j) * 32, ks, lane);
        };
        auto multiply = [&](const Slice& f) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
        };
        auto pass = [&]() {
            lds_fence(ring_at);
            __builtin_amdgcn_s_waitcnt(0xC07F);       // lgkmcnt(0): every fragment of this step is in registers
            __builtin_amdgcn_s_barrier();
            lds_fence(ring_at);
            stage = stage + 1 == S ? 0 : stage + 1;
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr int NM = TM * TN, NR = TM * (AKC ? 1 : 2) + TN * (BKC ? 1 : 2);

        // Two k-slices are read ahead of the one that is multiplied.  The barrier of a step stands between its two halves:
        // there the fragments of slices 2 and 3 of a k-tile are in registers and its stage is free.
        Slice f0, f1, f2, f3;
        clear();
        read(f0, 0); read(f1, 1); read(f2, 2);
        multiply(f0);
        read(f3, 3);
        multiply(f1);
        for (;;) {
            for (int kt = 1; kt < t.nkt; ++kt) {
                pass();
                read(f0, 0);
                multiply(f2);
                read(f1, 1);
                multiply(f3);
                read(f2, 2);
                multiply(f0);
                read(f3, 3);
                multiply(f1);
                deal_reads<0, 4 * NM, 4 * NR>();
                __builtin_amdgcn_sched_barrier(0);
            }
            pass();
            // the next tile's first fragments are on their way while this one is finished (behind the last one: zeros, or
            // what an earlier tile left, multiplied by nobody)
            read(f0, 0);
            multiply(f2);
            read(f1, 1);
            multiply(f3);
            deal_reads<0, 2 * NM, 2 * NR>();
            __builtin_amdgcn_sched_barrier(0);
            store(G.g[p], t, acc, ring + S * STAGE + wave * SLAB, wm, wn, lane);
            any = tile_of(G, l, n, ++r, t);
            if (!any || t.p != p) return;
            clear();
            read(f2, 2);
            multiply(f0);
            read(f3, 3);
            multiply(f1);
            deal_reads<0, 2 * NM, 2 * NR>();
        }
    }

    // Accumulators -> a slab of 16 rows in LDS -> 16-byte row segments -> memory.
    static __device__ __forceinline__ void store(Args& g, const Tile& t, f16v (&acc)[TM][TN], half_t* slab, int wm, int wn,
                                                 int lane) {
        const int l32 = lane & 31, hi = lane >> 5;
        const int m_wave = t.m0 + wm * 32 * TM, n_wave = t.n0 + wn * 32 * TN;
        if (g.splits > 1) {
            // fp32 partial tile, [split][batch][M][N]; a reduction adds them up
            float* P = g.partial + ((long)t.split * g.nbatch + t.bz) * (long)g.M * g.N;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int mm = m_wave + i * 32 + l32, nn = n_wave + j * 32 + q * 8 + hi * 4;
                        if (mm < g.M && nn + 4 <= g.N)
                            *reinterpret_cast<float4*>(P + (long)mm * g.N + nn) = make_float4(
                                acc[i][j][q * 4 + 0], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]);
                    }
            return;
        }
        const float alpha = g.alpha;
        // (buffer accesses: what lies outside of the output is dropped by the range check instead of a branch per row)
        const int nl = (lane % LPR) * 8, row = lane / LPR, rows = g.M - m_wave, cols = g.N - n_wave;
        const unsigned outside = nl + 8 <= cols ? 0u : 1u << 31;
        auto uniform_rsrc = [&](uint64_t at, long bytes) {
            auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(at), 0,
                                                     (int)u((uint32_t)(rows > 0 && cols > 0 ? bytes < 0x7fffffffL ? bytes : 0x7fffffffL : 0L)), 0x00020000);
        };
        auto buffer = [&](const half_t* p, long s_row) {
            return uniform_rsrc(reinterpret_cast<uint64_t>(uniform(p + (long)m_wave * s_row + n_wave)), 2 * ((long)(rows - 1) * s_row + cols));
        };
        const __amdgpu_buffer_rsrc_t rc = buffer(g.C + t.b0 * g.sCb[0] + t.b1 * g.sCb[1] + t.b2 * g.sCb[2], g.sCM);
        const unsigned c_step = (unsigned)(2 * RPI * g.sCM);
        unsigned c_at = (unsigned)(2 * (row * g.sCM + nl)) | outside;
        constexpr int NI = 16 / RPI;                                       // stores per lane and slab
        // ---- the activation's part (see quad_word): a word of four packs, of which lane j of four has pack j's
        constexpr int PACKS = 2 * TM * NI, WORDS = (PACKS + 3) / 4;
        constexpr bool GATED = EPI == EPI_GATE_COLSUM || EPI == EPI_GELU_GATE_COLSUM, FORWARD = EPI != EPI_PLAIN && !GATED;
        const int q = lane & 3;
        auto bits_rsrc = [&](const uint32_t* p) {
            if (!p) return uniform_rsrc(0, 0);
            return uniform_rsrc(reinterpret_cast<uint64_t>(uniform(p)) + (uint64_t)(((long)m_wave * g.N + n_wave) >> 3), ((long)(rows - 1) * g.N + cols) >> 3);
        };
        const unsigned bits_at = (unsigned)((q / NI * 16 + q % NI * RPI + row) * (g.N >> 3) + (lane % LPR >> 2) * 4) |
                                 ((lane % LPR >> 2) * 32 < cols && q < PACKS ? 0u : 1u << 31);
        const unsigned bits_step = (unsigned)(64 / NI * (g.N >> 3));       // four packs further
        uint32_t bits[WORDS];
        bool from_bits = false;
        if constexpr (EPI != EPI_PLAIN) {
            const uint32_t* p = GATED ? g.gate_bits : g.keep_words;
            from_bits = p != nullptr;
            if (from_bits) {
                const __amdgpu_buffer_rsrc_t r = bits_rsrc(p);
#pragma unroll
                for (int k = 0; k < WORDS; ++k) bits[k] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)(bits_at + k * bits_step), 0, 0);
            }
        }
        uint32_t kb[WORDS];                                                // FORWARD: keep bits of the lane's packs, a byte each
        if constexpr (FORWARD) {
            const PhiloxKey key = key_of(g.key);
#pragma unroll
            for (int k = 0; k < WORDS; ++k) kb[k] = ~0u;
            if (key.thr && !from_bits) {
                const uint64_t group0 = ((uint64_t)(m_wave + row) * (uint64_t)g.sCM + (uint64_t)(n_wave + nl)) >> 3;
                const uint64_t stride = (uint64_t)(g.sCM >> 3);
#pragma unroll
                for (int c = 0; c < PACKS; ++c) {
                    const uint32_t b = keep8(philox_group_dev(key, group0 + (uint64_t)(c / NI * 16 + c % NI * RPI) * stride), key.thr) << (8 * (c & 3));
                    kb[c >> 2] = (c & 3) ? kb[c >> 2] | b : b;
                }
            }
        }
        float colsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        auto tile = [&](auto kind) __attribute__((always_inline)) {
            constexpr int ADD = decltype(kind)::value;                    // 0 no addend, 1 a row, 2 a tensor, 3 the gate's values
            __amdgpu_buffer_rsrc_t rb = rc, rl = rc, ro = rc;
            unsigned b_at = 0, b_step = 0;
            if (ADD) {
                rb = ADD == 3 ? buffer(g.gate, g.sbM) : buffer(g.bias + t.b0 * g.sbb[0] + t.b1 * g.sbb[1] + t.b2 * g.sbb[2], g.sbM);
                b_at = (unsigned)(2 * (row * g.sbM + nl)) | outside;
                b_step = (unsigned)(2 * RPI * g.sbM);
            }
            if constexpr (EPI == EPI_GELU_DROPOUT) rl = buffer(g.pre_out, g.sCM);
            if constexpr (FORWARD) ro = bits_rsrc(g.gate_bits_out);       // (null: none)
            auto addend = [&]() {
                const h8 v = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)b_at, 0, 0));
                b_at += b_step;
                return v;
            };
            h8 one, next[NI];
            uint32_t out_word = 0;
            if (ADD == 1) one = addend();
            if (ADD >= 2)
#pragma unroll
                for (int it = 0; it < NI; ++it) next[it] = addend();      // (a slab ahead of its use)
            auto each_slab = [&](auto sl_) __attribute__((always_inline)) {
                constexpr int sl = decltype(sl_)::value, i = sl >> 1;
                h8 ad[NI];
#pragma unroll
                for (int it = 0; it < NI; ++it) ad[it] = ADD == 1 ? one : next[it];
                if (ADD >= 2 && sl + 1 < 2 * TM)
#pragma unroll
                    for (int it = 0; it < NI; ++it) next[it] = addend();
                // (the fences: the reads are of what other lanes wrote, which a single thread's rules do not show)
                lds_fence(lds_addr(slab));
                if ((l32 >> 4) == (sl & 1)) {
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            h4 w;
#pragma unroll
                            for (int e = 0; e < 4; ++e) w[e] = (half_t)(acc[i][j][q * 4 + e] * alpha);
                            *reinterpret_cast<h4*>(slab + (l32 & 15) * PITCH + j * 32 + q * 8 + hi * 4) = w;
                        }
                }
                // (LDS operations of one wave execute in order: the reads below see the writes above)
                lds_fence(lds_addr(slab));
                each<NI>([&](auto it_) __attribute__((always_inline)) {
                    constexpr int it = decltype(it_)::value, c = sl * NI + it;
                    h8 val = *reinterpret_cast<const h8*>(slab + (it * RPI + row) * PITCH + nl);
                    // (packed half add: the same single rounding as through fp32)
                    if (ADD == 1 || ADD == 2) val = val + ad[it];
                    if constexpr (GATED) {
                        uint32_t w = 0;
                        if constexpr (ADD == 0 || EPI == EPI_GELU_GATE_COLSUM) w = quad_byte<c & 3>(bits[c >> 2], lane);
                        // (rows beyond the last: nothing in the column sums; without bits, what is read there is zero)
                        w = sl * 16 + it * RPI + row < rows ? w : 0u;
                        val = act_backward<EPI, ADD == 0 || EPI == EPI_GELU_GATE_COLSUM>(val, ad[it], w, colsum);
                    }
                    if constexpr (EPI == EPI_GELU_DROPOUT)                 // the pre-activation, for the backward pass
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, val), rl, (int)c_at, 0, 0);
                    if constexpr (FORWARD) {
                        uint32_t keep = kb[c >> 2] >> (8 * (c & 3));
                        if (from_bits) keep = quad_byte<c & 3>(bits[c >> 2], lane);
                        val = act_forward<EPI>(val, keep);
                        if constexpr (EPI != EPI_GELU_ALONE) {
                            const uint32_t word = quad_word(keep, lane);
                            out_word = q == (c & 3) ? word : out_word;
                        }
                        if constexpr (EPI != EPI_GELU_ALONE && ((c & 3) == 3 || c == PACKS - 1))
                            __builtin_amdgcn_raw_buffer_store_b32(out_word, ro, (int)(bits_at + (c >> 2) * bits_step), 0, 0);
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, val), rc, (int)c_at, 0, 0);
                    c_at += c_step;
                });
                // (a slab's arithmetic is not spread over the next ones': registers)
                if (EPI == EPI_GELU_GATE_COLSUM) __builtin_amdgcn_sched_barrier(0);
            };
            each<2 * TM>(each_slab);
        };
        if constexpr (GATED) {
            if (EPI == EPI_GELU_GATE_COLSUM || !from_bits) tile(std::integral_constant<int, 3>{});
            else tile(std::integral_constant<int, 0>{});                  // (a gated product has no addend)
            // lanes LPR apart hold the same 8 columns for other rows: add them up, then one fp32 row of partial sums per
            // wave (a finishing launch adds them up)
#pragma unroll
            for (int o = LPR; o < 64; o <<= 1)
#pragma unroll
                for (int e = 0; e < 8; ++e) colsum[e] += __shfl_xor(colsum[e], o);
            if (lane < LPR && nl < cols) {
                float* dst = g.colsum + ((long)(t.m0 / BM) * WM + wm) * g.N + n_wave + lane * 8;
#pragma unroll
                for (int e = 0; e < 8; ++e) dst[e] = colsum[e];
            }
        } else {
            if (!g.bias) tile(std::integral_constant<int, 0>{});
            else if (g.sbM == 0) tile(std::integral_constant<int, 1>{});
            else tile(std::integral_constant<int, 2>{});
        }
    }

    static __device__ __forceinline__ void run(Group& G, half_t* lds) {
        const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const unsigned n = G.workers;
        if constexpr (NP > 1) if (blockIdx.x >= n) {
            // (behind the tiles: dispatched last, into places that they leave free or vacate first)
            if (tid >= kFinishThreads) return;
            const unsigned b = blockIdx.x - n;
            finish_block(G.tail.j[b / G.tail_groups], b % G.tail_groups, reinterpret_cast<float (*)[33]>(lds));
            return;
        }
        const unsigned l = xcd_order(blockIdx.x, n), ring_at = lds_addr(lds);
        fetch_gemm_args(G.g[0]);
        if (wave >= NC) {
            fetch(G, l, n, ring_at, wave - NC, lane);
            return;
        }
        unsigned r = 0;
        int stage = 0;
        Tile t;
        bool any = tile_of(G, l, n, r, t);
        lds_fence(ring_at);
        __builtin_amdgcn_s_barrier();
        lds_fence(ring_at);
        while (any) {
            if (K1 == K2 || !G.second[t.p]) consume<(K1 & 1) != 0, (K1 & 2) != 0>(G, l, n, r, t, any, lds, ring_at, stage, wave, lane);
            else consume<(K2 & 1) != 0, (K2 & 2) != 0>(G, l, n, r, t, any, lds, ring_at, stage, wave, lane);
        }
    }
};

template <int TM, int TN, int WM, int WN, int NL, int S, int NP, int K1, int K2, int EPI = EPI_PLAIN>
__global__ __launch_bounds__((WM * WN + NL) * 64) void k_gemm_ring(TileGroup<NP>) {
    using R = Ring<TM, TN, WM, WN, NL, S, NP, K1, K2, EPI>;
    __shared__ __attribute__((aligned(128))) half_t lds[R::HALVES];
    R::run(*(typename R::Group*)__builtin_amdgcn_kernarg_segment_ptr(), lds);
}

// The kernels of tile form `form` for the orientations of G's products (k1, k2: see list_tiles).
#define SUB_RING(...)                                                                                                        \
    do {                                                                                                                     \
        if constexpr (NP > 1) if (k1 == 1 && k2 == 0) { hipLaunchKernelGGL((k_gemm_ring<__VA_ARGS__, NP, 1, 0, EPI>), grid, block, 0, st, G); break; } \
        if constexpr (NP > 1) if (k1 == 3 && k2 == 0) { hipLaunchKernelGGL((k_gemm_ring<__VA_ARGS__, NP, 3, 0, EPI>), grid, block, 0, st, G); break; } \
        if (k1 == 3) hipLaunchKernelGGL((k_gemm_ring<__VA_ARGS__, NP, 3, 3, EPI>), grid, block, 0, st, G);                    \
        else if (k1 == 1) hipLaunchKernelGGL((k_gemm_ring<__VA_ARGS__, NP, 1, 1, EPI>), grid, block, 0, st, G);               \
        else if constexpr (EPI == EPI_PLAIN) {                                                                               \
            if (k1 == 2) hipLaunchKernelGGL((k_gemm_ring<__VA_ARGS__, NP, 2, 2, EPI>), grid, block, 0, st, G);                \
            else hipLaunchKernelGGL((k_gemm_ring<__VA_ARGS__, NP, 0, 0, EPI>), grid, block, 0, st, G);                        \
        } else fail("gemm: with an activation the first operand lies along k");                                              \
    } while (0)
template <int NP, int EPI>
void launch_ring_as(const TileGroup<NP>& G, int form, int k1, int k2, unsigned blocks, hipStream_t st) {
    const dim3 grid(blocks), block(512);
    switch (form) {
        case TILE_64x64: SUB_RING(1, 1, 2, 2, 4, 4); break;
        case TILE_128x64: SUB_RING(2, 1, 2, 2, 4, 3); break;
        case TILE_128x128: SUB_RING(2, 2, 2, 2, 4, 3); break;
        case TILE_256x128: SUB_RING(4, 2, 2, 2, 4, 3); break;
        default: fail("gemm: unknown tile");
    }
}
#undef SUB_RING

}  // namespace

}  // namespace sub
