// Tensor contractions: strided, batched fp16 GEMM with fp32 accumulation on the
// gfx950 matrix cores (v_mfma_f32_32x32x16_f16), honouring each operand's
// stride layout.  Takes the place of the cuBLAS calls behind
// pytorch_module/gemm.cuh:52-147.
//
//   C[b, m, n] = alpha * sum_k A[b, m, k] * B[b, k, n]  (+ bias)
//
// Operands may be contiguous along the contraction (K) or along their free
// dimension (M resp. N); an operand that is contiguous along its free dimension
// lies in LDS as in memory and is gathered with the transposing LDS read, so the
// matrix-core fragments are always 8 consecutive k per lane.  (Turning such tiles
// around in registers on the way into LDS instead, to read them at the full rate of
// ds_read_b128, was measured: 1 to 3 us slower per product of 34 GFLOP.)
// The output is produced transposed in the
// accumulators (4 consecutive n per lane), staged through LDS and written as
// full 128-bit rows.
#include <type_traits>
#include <cstring>

#include "sub_gemm.hpp"
#include "sub_finish.hpp"

namespace sub {

namespace {

// A workgroup that multiplies nothing (see GemmSideJob): workgroup sb of nsb.
__device__ __forceinline__ void side_block(const GemmArgs& g, unsigned sb, unsigned nsb) {
    const PhiloxKey key = resolved(g.side_key);
    const uint32_t nt = g.side_nk / 32, td = g.side_tiles_done;
    // word w of rows * td is (row w / td, tile w % td); a thread walks w in steps of `stride`, carrying row
    // and tile along instead of dividing (a 64-bit division is as long as one of the word's four draws)
    const uint32_t stride = nsb * blockDim.x, first = sb * blockDim.x + threadIdx.x;
    const uint32_t srow = stride / td, st = stride - srow * td;
    uint32_t row = first / td, t = first - row * td;
    for (; row < g.side_rows; row += srow) {
        g.side_keep[(size_t)row * nt + t] = attention_keep_word(key, row, g.side_nk, t);
        t += st;
        if (t >= td) { t -= td; ++row; }
    }
}

// ---------------------------------------------------------------------------
// Any strides, any sizes: what the matrix-core kernels do not take (mostly rows that are not whole 16-byte words: the
// score-sized products of sequence lengths that are not multiples of 8).  64 x 64 outputs per workgroup, 4 x 4 per
// thread, operands converted into LDS 32 k at a time; every output is one fp32 chain of fused multiply-adds in the
// order of k.  (One thread per output, straight from memory, before: 750 us for the scores of B=8 L=197 H=12, 0.5 GFLOP,
// bound by the latency of that chain's single-element loads.)
// ---------------------------------------------------------------------------
constexpr int FB = 64, FK = 32, FPITCH = FB + 4;

// One operand's 64 x 32 elements into LDS as [k][row].  vec: whole 16-byte words along k.
__device__ __forceinline__ void fma_tile(float (*dst)[FPITCH], const half_t* p, long s_row, long s_k, int rows, int ks, bool vec,
                                         int tid) {
    if (vec) {
        const int row = tid >> 2, k = (tid & 3) * 8;
        h8 v = (h8)(half_t)0.0f;
        if (row < rows && k < ks) v = *reinterpret_cast<const h8*>(p + (long)row * s_row + k);
#pragma unroll
        for (int i = 0; i < 8; ++i) dst[k + i][row] = (float)v[i];
        return;
    }
    half_t v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = tid + i * 256, row = s_k == 1 ? e / FK : e % FB, k = s_k == 1 ? e % FK : e / FB;
        v[i] = row < rows && k < ks ? p[(long)row * s_row + (long)k * s_k] : (half_t)0.0f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int e = tid + i * 256, row = s_k == 1 ? e / FK : e % FB, k = s_k == 1 ? e % FK : e / FB;
        dst[k][row] = (float)v[i];
    }
}

__global__ __launch_bounds__(256) void k_gemm_fma(GemmArgs g, bool vec_a, bool vec_b) {
    __shared__ __attribute__((aligned(16))) float ta[FK][FPITCH], tb[FK][FPITCH];
    const int tid = threadIdx.x, tm = (tid >> 4) * 4, tn = (tid & 15) * 4;
    const unsigned tiles_m = (g.M + FB - 1) / FB, tiles_n = (g.N + FB - 1) / FB;
    unsigned id = blockIdx.x;
    const unsigned n0 = id % tiles_n * FB; id /= tiles_n;
    const unsigned m0 = id % tiles_m * FB; id /= tiles_m;
    const long b2 = id % g.nb2; id /= g.nb2;
    const long b1 = id % g.nb1, b0 = id / g.nb1;
    const half_t* a = g.A + b0 * g.sAb[0] + b1 * g.sAb[1] + b2 * g.sAb[2] + (long)m0 * g.sAM;
    const half_t* b = g.B + b0 * g.sBb[0] + b1 * g.sBb[1] + b2 * g.sBb[2] + (long)n0 * g.sBN;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < g.K0; ++k0)
        for (int k = 0; k < g.K1; k += FK) {
            const int ks = min(FK, g.K1 - k);
            __syncthreads();
            fma_tile(ta, a + (long)k0 * g.sAK0 + (long)k * g.sAK1, g.sAM, g.sAK1, g.M - (int)m0, ks, vec_a, tid);
            fma_tile(tb, b + (long)k0 * g.sBK0 + (long)k * g.sBK1, g.sBN, g.sBK1, g.N - (int)n0, ks, vec_b, tid);
            __syncthreads();
#pragma unroll 8
            for (int i = 0; i < ks; ++i) {
                const float4 x = *reinterpret_cast<const float4*>(&ta[i][tm]), y = *reinterpret_cast<const float4*>(&tb[i][tn]);
                const float xv[4] = {x.x, x.y, x.z, x.w}, yv[4] = {y.x, y.y, y.z, y.w};
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[r][c] = __builtin_fmaf(xv[r], yv[c], acc[r][c]);
            }
        }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int m = (int)m0 + tm + r, n = (int)n0 + tn + c;
            if (m >= g.M || n >= g.N) continue;
            half_t out = (half_t)(acc[r][c] * g.alpha);
            if (g.bias)     // same two roundings as the product followed by a separate add
                out = (half_t)((float)out + (float)g.bias[b0 * g.sbb[0] + b1 * g.sbb[1] + b2 * g.sbb[2] +
                                                          (long)m * g.sbM + (long)n * g.sbN]);
            g.C[b0 * g.sCb[0] + b1 * g.sCb[1] + b2 * g.sCb[2] + (long)m * g.sCM + (long)n * g.sCN] = out;
        }
}

// ---------------------------------------------------------------------------
// Asynchronous variant for full tiles: global memory -> LDS directly
// (global_load_lds_dwordx4), a ring of S stages, no staging registers and no
// ds_write.  Each wave instruction deposits 64 x 16 bytes at consecutive LDS
// addresses, so the lane -> global-chunk map is chosen such that the bytes land
// in the (bank-swizzled) tile layout the fragment reads expect.  The stages are
// separate __shared__ arrays and the k loop is unrolled over them, which lets
// the compiler see that the fragment reads of one stage do not depend on the
// loads in flight to another; completion is tracked by hand with s_waitcnt
// vmcnt(n) followed by a plain s_barrier.
// ---------------------------------------------------------------------------
// Issue order of half a step of the eight-wave kernel: NM matrix instructions with NR
// fragment reads dealt out evenly between them (after FIRST reads in front).
template <int m, int NM, int NR>
__device__ __forceinline__ void sched_mfma_reads_from() {
    if constexpr (m < NM) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        constexpr int r = (NR * (m + 1)) / NM - (NR * m) / NM;
        if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
        sched_mfma_reads_from<m + 1, NM, NR>();
    }
}
// NM matrix instructions, each followed by NV vector instructions.
template <int NM, int NV, int m = 0>
__device__ __forceinline__ void sched_mfma_valu() {
    if constexpr (m < NM) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
        sched_mfma_valu<NM, NV, m + 1>();
    }
}
template <int FIRST, int NM, int NR>
__device__ __forceinline__ void sched_half_step() {
    if constexpr (FIRST > 0) __builtin_amdgcn_sched_group_barrier(0x100, FIRST, 0);
    sched_mfma_reads_from<0, NM, NR>();
}

// NW waves as 2 x (NW / 2); each wave owns TM x TN accumulator tiles of 32 x 32.
// Eight waves (two per SIMD) on a 256 x 256 tile: a wave cannot issue past an
// asynchronous load that the memory path has not accepted yet, and with all 256 CUs
// drawing on L2 that takes long (measured: the loads of a step alone cost about as
// much time as its multiplications, and with one wave per SIMD the two add up);
// while one wave of a SIMD sits in the issue of its loads the other multiplies.
// EPI: what the epilogue does after the scaling and the optional addend.  A template
// parameter so that the plain kernel does not carry the registers of the others.
// EPI_RELU_DROPOUT_PRE: EPI_RELU_DROPOUT with the keep bits drawn ahead of the launch (GemmEpilogue::keep_words)
// EPI_GELU_DROPOUT: as EPI_RELU_DROPOUT with GELU; also stores the rounded sum before the activation
// (GemmArgs::pre_out, which the backward pass needs) and leaves the keep bits where the ReLU form leaves its gate bits.
// EPI_GELU_GATE_COLSUM: the backward counterpart: out = keep bit ? gelu'(pre-activation) * product : 0, and column sums.
enum { EPI_PLAIN = 0, EPI_RELU_DROPOUT = 1, EPI_GATE_COLSUM = 2, EPI_RELU_DROPOUT_PRE = 3, EPI_GELU_DROPOUT = 4,
       EPI_GELU_GATE_COLSUM = 5 };

template <int TM, int TN, bool AKC, bool BKC, int S, int NW, int EPI = EPI_PLAIN>
__global__ __launch_bounds__(NW * 64) void k_gemm_dma(GemmArgs g) {
    static_assert(S == 2 || S == 3, "two or three LDS stages");
    static_assert(NW == 4 || NW == 8, "four or eight waves");
    constexpr int WN = NW / 2;
    constexpr int BM = 64 * TM, BN = 32 * TN * WN;
    using TA = DTile<BM, AKC, NW>;
    using TB = DTile<BN, BKC, NW>;
    constexpr int STAGE = TA::HALVES + TB::HALVES;
    constexpr int STAGE_PITCH = 32 * TN + 8;
    constexpr int STAGE_WAVE = 32 * STAGE_PITCH;
    static_assert(NW * STAGE_WAVE <= STAGE, "epilogue staging must fit one stage");
    // one array per stage: the compiler then sees that an asynchronous load into one
    // stage does not alias the fragment reads from another, and adds no waits of its own
    __shared__ __attribute__((aligned(16))) half_t st0[STAGE];
    __shared__ __attribute__((aligned(16))) half_t st1[STAGE];
    __shared__ __attribute__((aligned(16))) half_t st2[S > 2 ? STAGE : 8];
    constexpr int L = TA::NV + TB::NV;               // loads per thread per tile

    // (the wave index as a scalar: LDS destinations of the asynchronous loads are then scalar arithmetic)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int l32 = lane & 31, hi = lane >> 5;

    fetch_gemm_args(g);
    const int tiles_m = g.M / BM, tiles_n = g.N / BN;
    unsigned lid = blockIdx.x;
    {
        unsigned nblocks = gridDim.x;
        if constexpr (NW == 8 && EPI == EPI_PLAIN) {
            if (g.side_blocks) {
                if (blockIdx.x >= g.side_first) { side_block(g, blockIdx.x - g.side_first, g.side_blocks); return; }
                nblocks = g.side_first;
            }
        }
        if ((nblocks & 7) == 0) lid = (lid & 7u) * (nblocks >> 3) + (lid >> 3);
    }
    // (32-bit arithmetic)
    const unsigned per_batch = (unsigned)(tiles_m * tiles_n);
    const unsigned bz = lid / per_batch;
    int r = (int)(lid - bz * per_batch);
    constexpr int GM = 8;
    const int grp = r / (GM * tiles_n), first_m = grp * GM;
    const int gsz = tiles_m - first_m < GM ? tiles_m - first_m : GM;
    const int rr = r - grp * GM * tiles_n;
    const int tile_m = first_m + rr % gsz, tile_n = rr / gsz;
    const unsigned tq = bz / (unsigned)g.nb2;
    const long b2 = bz - tq * (unsigned)g.nb2, b0 = tq / (unsigned)g.nb1, b1 = tq - (unsigned)b0 * (unsigned)g.nb1;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    // (the tile pointers are the same for every lane: kept in scalar registers, a load's address is
    // scalar base + 32-bit lane offset instead of a 64-bit vector addition per load)
    auto uniform = [](const half_t* p) {
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
        const uint32_t hi2 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
        return reinterpret_cast<const half_t*>(((uint64_t)hi2 << 32) | lo);
    };
    const half_t* pa = uniform(g.A + b0 * g.sAb[0] + b1 * g.sAb[1] + b2 * g.sAb[2] + (long)m0 * g.sAM);
    const half_t* pb = uniform(g.B + b0 * g.sBb[0] + b1 * g.sBb[1] + b2 * g.sBb[2] + (long)n0 * g.sBN);

    const int tiles_per_k1 = g.K1 / BK;
    const int nkt = g.K0 * tiles_per_k1;

    f16v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    unsigned offa[TA::NV], offb[TB::NV];
    TA::offsets(offa, g.sAM, g.sAK1, wave, lane);
    TB::offsets(offb, g.sBN, g.sBK1, wave, lane);

    int kin = 0, fetched = 0;
    const long stepA = (long)BK * g.sAK1, stepB = (long)BK * g.sBK1;
    const long wrapA = g.sAK0 - (long)(tiles_per_k1 - 1) * stepA;
    const long wrapB = g.sBK0 - (long)(tiles_per_k1 - 1) * stepB;

    // Fetch the next k-tile into `stage`; past the last tile the pointers stay put
    // (surplus fetches re-read valid memory and keep the vmcnt bookkeeping uniform).
#define SUB_DMA_ISSUE(stage_)                                                                     \
    do {                                                                                          \
        TA::issue(stage_, pa, offa, wave);                                                        \
        TB::issue(stage_ + TA::HALVES, pb, offb, wave);                                           \
        const bool more_ = fetched + 1 < nkt;                                                     \
        const bool wrap_ = kin + 1 == tiles_per_k1;                                               \
        pa += more_ ? (wrap_ ? wrapA : stepA) : 0;                                                \
        pb += more_ ? (wrap_ ? wrapB : stepB) : 0;                                                \
        kin = more_ ? (wrap_ ? 0 : kin + 1) : kin;                                                \
        fetched += more_ ? 1 : 0;                                                                 \
    } while (0)

    // ReLU-dropout epilogue: the keep bits of the 16 packs of 8 outputs this lane stores are
    // drawn during the multiplication, one Philox call per step, where the vector unit is
    // otherwise idle; the epilogue only picks its byte.  Pack c (0..15) covers output row
    // (first row of the wave) + 8 c + lane / 8, so its group of 8 canonical elements is
    // kb_group0 + c * sCM.  Every step shifts the 128 bits up by a byte and draws pack
    // (kb_next & 15); the start is chosen so that the last 16 steps draw packs 0..15 in order.
    constexpr int LPR = 4 * TN;                      // lanes per output row of the wave's slab
    constexpr int RPI = 64 / LPR;                    // rows per store instruction
    constexpr bool DRAWS = EPI == EPI_RELU_DROPOUT || EPI == EPI_GELU_DROPOUT;    // keep bits drawn in the main loop
    static_assert(!DRAWS || TM * (32 / RPI) == 16, "16 packs of keep bits per lane");
    PhiloxKey rd_key = g.key;
    uint32_t kb[4] = {0u, 0u, 0u, 0u};
    uint64_t kb_group0 = 0;
    int kb_next = 0;
    if (DRAWS) {
        rd_key = resolved(g.key);
        const uint64_t row = (uint64_t)(m0 + wm * 32 * TM + lane / LPR);
        kb_group0 = (row * (uint64_t)g.sCM + (uint64_t)(n0 + wn * 32 * TN + (lane % LPR) * 8)) >> 3;
        kb_next = nkt >= 16 ? (16 - (nkt & 15)) & 15 : 0;
    }
#define SUB_DMA_KEEP()                                                                            \
    do {                                                                                          \
        const U4 r_ = philox_group(rd_key, kb_group0 + (uint64_t)(kb_next & 15) * (uint64_t)g.sCM); \
        const uint32_t b_ = keep8(r_, rd_key.thr);                                                \
        kb[3] = (kb[3] << 8) | (kb[2] >> 24);                                                     \
        kb[2] = (kb[2] << 8) | (kb[1] >> 24);                                                     \
        kb[1] = (kb[1] << 8) | (kb[0] >> 24);                                                     \
        kb[0] = (kb[0] << 8) | b_;                                                                \
        ++kb_next;                                                                                \
    } while (0)

    // What the epilogue reads besides the accumulators is requested here, ahead of the contraction: behind it the
    // round trip to memory would stand in the open (the loads complete in order, ahead of the tiles').
    half_t* Cb = g.C + b0 * g.sCb[0] + b1 * g.sCb[1] + b2 * g.sCb[2];
    const half_t* biasb = g.bias ? g.bias + b0 * g.sbb[0] + b1 * g.sbb[1] + b2 * g.sbb[2] : nullptr;
    // a bias row (the same for every row of the output): a lane's 8 columns are the same in all of its
    // packs, so it loads them once instead of before every store
    const bool bias_row = biasb && g.sbM == 0;
    h8 bias8 = (h8)(half_t)0.0f;
    if (bias_row) bias8 = *reinterpret_cast<const h8*>(biasb + n0 + wn * 32 * TN + (lane % LPR) * 8);
    // One bit per output of the ReLU-dropout epilogue (set = positive), a dword per lane and 32-row
    // slab in the order this epilogue walks the tile: the gate epilogue of a product with the same
    // output shape reads 1/16 of what the outputs themselves would cost it.
    constexpr bool RELU_DROP = EPI == EPI_RELU_DROPOUT || EPI == EPI_RELU_DROPOUT_PRE;
    constexpr bool GELU_DROP = EPI == EPI_GELU_DROPOUT;
    constexpr bool GATED = EPI == EPI_GATE_COLSUM || EPI == EPI_GELU_GATE_COLSUM;
    static_assert(EPI == EPI_PLAIN || 32 / RPI == 4, "four packs of 8 outputs per lane and slab");
    const long bits_at = (((long)tile_m * tiles_n + tile_n) * NW + wave) * (TM * 64) + lane;
    uint32_t gbits[TM];
    if (GATED && g.gate_bits) {
#pragma unroll
        for (int i = 0; i < TM; ++i) gbits[i] = g.gate_bits[bits_at + i * 64];
    }

    constexpr int RA_ = AKC ? 1 : 2, RB_ = BKC ? 1 : 2;      // LDS reads per fragment
    const int fbase_a = TA::frag_base(wm * TM * 32, lane), fbase_b = TB::frag_base(wn * TN * 32, lane);
#define SUB_DMA_FRAG_A(i_, ks_) (AKC && NW == 8 ? TA::frag_at(sA, ba_, i_, ks_) : TA::frag(sA, (wm * TM + (i_)) * 32, ks_, lane))
#define SUB_DMA_FRAG_B(j_, ks_) (BKC && NW == 8 ? TB::frag_at(sB, bb_, j_, ks_) : TB::frag(sB, (wn * TN + (j_)) * 32, ks_, lane))
#define SUB_DMA_COMPUTE(stage_, nx_)                                                              \
    do {                                                                                          \
        const half_t* sA = stage_;                                                                \
        const half_t* sB = stage_ + TA::HALVES;                                                   \
        h8 fa[2][TM], fb[2][TN];                                                                  \
        int ba_ = fbase_a, bb_ = fbase_b;                                                         \
        if constexpr (NW == 8) asm volatile("" : "+v"(ba_), "+v"(bb_));                           \
        _Pragma("unroll") for (int i = 0; i < TM; ++i)                                            \
            fa[0][i] = SUB_DMA_FRAG_A(i, 0);                                                      \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                            \
            fb[0][j] = SUB_DMA_FRAG_B(j, 0);                                                      \
        _Pragma("unroll") for (int ks = 0; ks < BK / 16; ++ks) {                                  \
            if (NW == 8 && ks == BK / 32) {                                                       \
                /* first half: the reads of k-slices 1 and 2 between the products of 0 and 1 */   \
                sched_half_step<TM * RA_ + TN * RB_, 2 * TM * TN, 2 * (TM * RA_ + TN * RB_)>();   \
                if (late) SUB_DMA_ISSUE(nx_);                                                     \
                __builtin_amdgcn_sched_barrier(0);                                                \
            }                                                                                     \
            if (NW == 8 && DRAWS && ks == BK / 16 - 1) {                                          \
                /* the last k-slice shares its issue slots with the keep bits: the fragments of  \
                   the slice before are dead by now, so the draw costs no registers */           \
                sched_half_step<0, TM * TN, TM * RA_ + TN * RB_>();                               \
                __builtin_amdgcn_sched_barrier(0);                                                \
                SUB_DMA_KEEP();                                                                   \
            }                                                                                     \
            if (ks + 1 < BK / 16) {                                                               \
                _Pragma("unroll") for (int i = 0; i < TM; ++i)                                    \
                    fa[(ks + 1) & 1][i] = SUB_DMA_FRAG_A(i, ks + 1);                              \
                _Pragma("unroll") for (int j = 0; j < TN; ++j)                                    \
                    fb[(ks + 1) & 1][j] = SUB_DMA_FRAG_B(j, ks + 1);                              \
            }                                                                                     \
            _Pragma("unroll") for (int i = 0; i < TM; ++i)                                        \
                _Pragma("unroll") for (int j = 0; j < TN; ++j)                                    \
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[ks & 1][j], fa[ks & 1][i], \
                                                                       acc[i][j], 0, 0, 0);       \
        }                                                                                         \
        /* second half: the reads of k-slice 3 between the products of k-slice 2 */               \
        if constexpr (NW == 8 && !DRAWS)                                                          \
            sched_half_step<0, 2 * TM * TN, TM * RA_ + TN * RB_>();                               \
        if constexpr (NW == 8 && DRAWS) sched_mfma_valu<TM * TN, 12>();                           \
    } while (0)

    // One step: tile kt is complete once at most the L loads of tile kt+1 are
    // outstanding; the barrier also says every wave is done reading the stage
    // that the fetch below overwrites (it was computed on one step earlier).
#define SUB_DMA_STEP(cur_, nxt2_)                                                                 \
    do {                                                                                          \
        __builtin_amdgcn_s_waitcnt(waitcnt_vm((S - 2) * L));                                      \
        __builtin_amdgcn_s_barrier();                                                             \
        if (!late) SUB_DMA_ISSUE(nxt2_);                                                          \
        /* keep the fetches ahead of the multiply phase: the scheduler must not sink them */      \
        __builtin_amdgcn_sched_barrier(0);                                                        \
        SUB_DMA_COMPUTE(cur_, nxt2_);                                                            \
    } while (0)

    // Eight waves: the second wave of each SIMD issues its loads half a step after
    // the first, so that the two are not held up in the issue at the same time.
    const bool late = NW == 8 && __builtin_amdgcn_readfirstlane(wave) >= 4;
    // S stages: while tile kt is multiplied, tiles kt+1 .. kt+S-2 are landed or on
    // their way and the fetch of tile kt+S-1 goes into the stage of tile kt-1.
    // (One array per stage and each round of S steps as straight-line code: with one
    // array for the ring, or the steps behind conditions of their own, the compiler
    // no longer sees which stage a fragment read touches and waits for every load
    // in flight before it.  More than three stages of 128 x 128 tiles gained nothing.)
    if (S == 2) {
        SUB_DMA_ISSUE(st0);
        const int nr = nkt / 2;
        for (int p = 0; p < nr; ++p) {
            SUB_DMA_STEP(st0, st1);
            SUB_DMA_STEP(st1, st0);
        }
        if (nkt & 1) SUB_DMA_STEP(st0, st1);
    } else if (S == 3) {
        SUB_DMA_ISSUE(st0);
        SUB_DMA_ISSUE(st1);
        const int nr = nkt / 3, rem = nkt - 3 * nr;
        for (int p = 0; p < nr; ++p) {
            SUB_DMA_STEP(st0, st2);
            SUB_DMA_STEP(st1, st0);
            SUB_DMA_STEP(st2, st1);
        }
        if (rem >= 1) SUB_DMA_STEP(st0, st2);
        if (rem >= 2) SUB_DMA_STEP(st1, st0);
    }
    if (DRAWS)
        for (int c = nkt; c < 16; ++c) SUB_DMA_KEEP();        // a contraction shorter than 16 steps
#undef SUB_DMA_STEP
#undef SUB_DMA_COMPUTE
#undef SUB_DMA_FRAG_A
#undef SUB_DMA_FRAG_B
#undef SUB_DMA_KEEP
#undef SUB_DMA_ISSUE
    // surplus fetches may still be landing: drain them before LDS is reused
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    __syncthreads();

    half_t* stage = st0 + wave * STAGE_WAVE;
    float colsum[8];              // gate mode: this lane's 8 columns summed over its rows of the wave's slab
#pragma unroll
    for (int e = 0; e < 8; ++e) colsum[e] = 0.f;
    if (EPI == EPI_RELU_DROPOUT_PRE) {
        const uint4 w = reinterpret_cast<const uint4*>(g.keep_words)[(((long)tile_m * tiles_n + tile_n) * NW + wave) * 64 + lane];
        kb[0] = w.x; kb[1] = w.y; kb[2] = w.z; kb[3] = w.w;
    }
    // The lane's stores walk down the tile RPI rows at a time: running pointers (a 64-bit product
    // per store otherwise), and one copy of the loop per kind of addend (none, a bias row, a tensor:
    // chosen per store, the branches joined in a wait for every store issued so far).  Most products
    // have alpha = 1: no multiplication then.
    const bool alpha_one = g.alpha == 1.0f;
    const long c_step = (long)RPI * g.sCM, b_step = (long)RPI * g.sbM;
    const int row_first = m0 + wm * 32 * TM + lane / LPR, col_first = n0 + wn * 32 * TN + (lane % LPR) * 8;
    half_t* const c_first = Cb + (long)row_first * g.sCM + col_first;
    const long b_first = (long)row_first * g.sbM + col_first;        // addend and gate share their strides
    auto store_tile = [&](auto addend_kind) {
        constexpr int ADD = decltype(addend_kind)::value;           // 0 none, 1 a bias row, 2 a tensor
        half_t* cp = c_first;
        const half_t* bp = ADD == 2 ? biasb + b_first : nullptr;
        // (the GELU form reads the pre-activation values there, and the keep bits besides)
        const half_t* gp = (EPI == EPI_GELU_GATE_COLSUM || (EPI == EPI_GATE_COLSUM && !g.gate_bits)) ? g.gate + b_first : nullptr;
        half_t* lp = GELU_DROP ? g.pre_out + (c_first - Cb) : nullptr;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            uint32_t positive = 0;
            if (alpha_one) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        h4 w;
#pragma unroll
                        for (int e = 0; e < 4; ++e) w[e] = (half_t)acc[i][j][q * 4 + e];
                        *reinterpret_cast<h4*>(stage + l32 * STAGE_PITCH + j * 32 + q * 8 + hi * 4) = w;
                    }
            } else {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        h4 w;
#pragma unroll
                        for (int e = 0; e < 4; ++e) w[e] = (half_t)(acc[i][j][q * 4 + e] * g.alpha);
                        *reinterpret_cast<h4*>(stage + l32 * STAGE_PITCH + j * 32 + q * 8 + hi * 4) = w;
                    }
            }
#pragma unroll
            for (int it = 0; it < 32 / RPI; ++it) {
                const int rr2 = it * RPI + lane / LPR, c8 = (lane % LPR) * 8;
                h8 val = *reinterpret_cast<const h8*>(stage + rr2 * STAGE_PITCH + c8);
                // packed half add: the same single rounding as through fp32
                if (ADD == 1) val = val + bias8;
                if (ADD == 2) val = val + *reinterpret_cast<const h8*>(bp);
                if (EPI == EPI_GATE_COLSUM) {
                    // the ReLU layer's backward-dropout-activation: zero where the forward output was not positive
                    if (g.gate_bits) {
                        const uint32_t bits = gbits[i] >> (8 * it);
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            val[e] = ((bits >> e) & 1u) ? val[e] : (half_t)0.0f;
                            colsum[e] += (float)val[e];
                        }
                    } else {
                        const h8 gt = *reinterpret_cast<const h8*>(gp);
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            val[e] = (float)gt[e] > 0.f ? val[e] : (half_t)0.0f;
                            colsum[e] += (float)val[e];
                        }
                    }
                }
                if (EPI == EPI_GELU_GATE_COLSUM) {
                    // the GELU layer's backward-dropout-activation, as the operator computes it
                    const uint32_t bits = gbits[i] >> (8 * it);
                    const h8 lin = *reinterpret_cast<const h8*>(gp);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        // (computed for every element and then selected: no branch per element)
                        const float gv = gelu_bwd((float)lin[e], (float)val[e]);
                        val[e] = ((bits >> e) & 1u) ? (half_t)gv : (half_t)0.0f;
                        colsum[e] += (float)val[e];
                    }
                }
                if (GELU_DROP) {
                    *reinterpret_cast<h8*>(lp) = val;              // the pre-activation, for the backward pass
                    lp += c_step;
                    const int c = i * (32 / RPI) + it, byte = 15 - c;
                    const uint32_t bits = kb[byte >> 2] >> ((byte & 3) * 8);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float gv = gelu_fwd((float)val[e]);       // for every element, then selected: no branches
                        val[e] = ((bits >> e) & 1u) ? (half_t)gv : (half_t)0.0f;
                    }
                    positive |= (bits & 0xffu) << (8 * it);        // here: the keep bits
                }
                if (RELU_DROP) {
                    // what the bias-activation-dropout operator does to the rounded sum, with the
                    // same keep bits (the element index is the offset into the dense output):
                    // pack c sits in byte 15 - c of the bits drawn in the main loop
                    const int c = i * (32 / RPI) + it, byte = 15 - c;
                    const uint32_t bits = kb[byte >> 2] >> ((byte & 3) * 8);
                    val = __builtin_elementwise_max(val, (h8)(half_t)0.0f);       // ReLU, packed
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        val[e] = ((bits >> e) & 1u) ? val[e] : (half_t)0.0f;
                        positive |= (val[e] > (half_t)0.0f ? 1u : 0u) << (8 * it + e);
                    }
                }
                *reinterpret_cast<h8*>(cp) = val;
                cp += c_step;
                if (ADD == 2) bp += b_step;
                if (GATED) gp += b_step;
            }
            if ((RELU_DROP || GELU_DROP) && g.gate_bits_out) g.gate_bits_out[bits_at + i * 64] = positive;
        }
    };
    if (GATED || !biasb) store_tile(std::integral_constant<int, 0>{});     // (a gated product has no addend)
    else if (bias_row) store_tile(std::integral_constant<int, 1>{});
    else store_tile(std::integral_constant<int, 2>{});
    if (GATED) {
        // lanes LPR apart hold the same 8 columns for other rows: add them up, then one fp32
        // row of partial sums per 128-row slab of the output (a finishing launch adds the slabs)
#pragma unroll
        for (int o = LPR; o < 64; o <<= 1)
#pragma unroll
            for (int e = 0; e < 8; ++e) colsum[e] += __shfl_xor(colsum[e], o);
        if (lane < LPR) {
            float* dst = g.colsum + ((long)tile_m * 2 + wm) * g.N + n0 + wn * 32 * TN + lane * 8;
#pragma unroll
            for (int e = 0; e < 8; ++e) dst[e] = colsum[e];
        }
    }
}

// Adds the k-split partials: C[b,m,n] = fp16(alpha * sum_s P[s][b][m][n]) (+ addend).
__device__ __forceinline__ void splitk_sum_block(const GemmArgs& g, long nb_total, long block) {
    const long quads = (long)g.N / 4;
    long idx = block * 256 + threadIdx.x;
    if (idx >= nb_total * g.M * quads) return;
    int nq = (int)(idx % quads); long rr = idx / quads;
    int m = (int)(rr % g.M); long bz = rr / g.M;
    const long slab = nb_total * (long)g.M * g.N;
    const float* p = g.partial + (bz * g.M + m) * (long)g.N + nq * 4;
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[8];                  // at most 8 splits: all loads in flight at once
#pragma unroll
    for (int s = 0; s < 8; ++s)
        v[s] = s < g.splits ? *reinterpret_cast<const float4*>(p + (long)s * slab) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < 8; ++s) { t.x += v[s].x; t.y += v[s].y; t.z += v[s].z; t.w += v[s].w; }
    long b2 = bz % g.nb2; long tt = bz / g.nb2;
    long b1 = tt % g.nb1; long b0 = tt / g.nb1;
    half_t* c = g.C + b0 * g.sCb[0] + b1 * g.sCb[1] + b2 * g.sCb[2] + (long)m * g.sCM + nq * 4;
    h4 o;
    o[0] = (half_t)(t.x * g.alpha); o[1] = (half_t)(t.y * g.alpha);
    o[2] = (half_t)(t.z * g.alpha); o[3] = (half_t)(t.w * g.alpha);
    if (g.bias) {
        const half_t* ad = g.bias + b0 * g.sbb[0] + b1 * g.sbb[1] + b2 * g.sbb[2] + (long)m * g.sbM + nq * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (half_t)((float)o[e] + (float)ad[e]);
    }
    *reinterpret_cast<h4*>(c) = o;
}

__global__ __launch_bounds__(256) void k_gemm_splitk_reduce(GemmArgs g, long nb_total) {
    splitk_sum_block(g, nb_total, blockIdx.x);
}

inline bool mult8(long x) { return (x & 7) == 0; }
inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Canonical form: C contiguous along N (swap the operands otherwise).
struct Canon {
    GemmArgs a;
    bool ok_c;       // C has a unit stride along N after canonicalisation
};

Canon canonicalise(const GemmShape& s, const half_t* A, const half_t* B, half_t* C, float alpha,
                   const GemmEpilogue& ep) {
    Canon c;
    GemmArgs& a = c.a;
    const bool swap = s.sCN != 1 && s.sCM == 1;
    if (!swap) {
        a.A = A; a.B = B; a.M = (int)s.M; a.N = (int)s.N;
        a.sAM = s.sAM; a.sAK1 = s.sAK1; a.sAK0 = s.sAK0;
        a.sBN = s.sBN; a.sBK1 = s.sBK1; a.sBK0 = s.sBK0;
        a.sCM = s.sCM; a.sCN = s.sCN;
        for (int i = 0; i < 3; ++i) { a.sAb[i] = s.sAb[i]; a.sBb[i] = s.sBb[i]; }
        a.sbM = ep.sbM; a.sbN = ep.sbN;
    } else {
        a.A = B; a.B = A; a.M = (int)s.N; a.N = (int)s.M;
        a.sAM = s.sBN; a.sAK1 = s.sBK1; a.sAK0 = s.sBK0;
        a.sBN = s.sAM; a.sBK1 = s.sAK1; a.sBK0 = s.sAK0;
        a.sCM = s.sCN; a.sCN = s.sCM;
        for (int i = 0; i < 3; ++i) { a.sAb[i] = s.sBb[i]; a.sBb[i] = s.sAb[i]; }
        a.sbM = ep.sbN; a.sbN = ep.sbM;
    }
    a.C = C; a.K1 = (int)s.K1; a.K0 = (int)s.K0;
    a.nb1 = (int)s.nb[1]; a.nb2 = (int)s.nb[2];
    for (int i = 0; i < 3; ++i) { a.sCb[i] = s.sCb[i]; a.sbb[i] = ep.sbb[i]; }
    a.alpha = alpha; a.bias = ep.bias;
    a.relu_dropout = ep.relu_dropout ? 1 : 0; a.key = ep.key;
    a.gate = ep.gate; a.colsum = ep.colsum; a.gate_bits_out = ep.gate_bits_out; a.gate_bits = ep.gate_bits;
    a.keep_words = ep.keep_words; a.act = ep.act; a.pre_out = ep.pre_out;
    a.splits = 1; a.partial = nullptr;
    c.ok_c = a.sCN == 1;
    return c;
}

// 0 = scalar, 1 = MFMA
int pick_kind(const Canon& c, bool& akc, bool& bkc) {
    const GemmArgs& a = c.a;
    if (!c.ok_c) return 0;
    if (a.M <= 0 || a.N <= 0 || a.K1 <= 0) return 0;
    akc = a.sAK1 == 1; bkc = a.sBK1 == 1;
    if (!akc && a.sAM != 1) return 0;
    if (!bkc && a.sBN != 1) return 0;
    if (!al16(a.A) || !al16(a.B) || !al16(a.C)) return 0;
    if (a.K0 > 1 && a.K1 % BK != 0) return 0;
    if (a.bias && !(a.sbN == 1 && mult8(a.sbM) && mult8(a.sbb[0]) && mult8(a.sbb[1]) && mult8(a.sbb[2]) &&
                    al16(a.bias)))
        return 0;
    if (a.gate && !(a.sbN == 1 && mult8(a.sbM) && al16(a.gate) && !a.bias && a.colsum)) return 0;
    // GELU: the backward form needs the keep bits, the forward form a place for the pre-activation and for those bits
    if (a.act == ACT_GELU && a.gate && !a.gate_bits) return 0;
    if (a.act == ACT_GELU && a.relu_dropout && !(a.pre_out && al16(a.pre_out) && a.gate_bits_out && !a.keep_words)) return 0;
    // every 16-byte access must be aligned and whole
    bool ok = mult8(a.N) && mult8(a.sCM) && mult8(a.sCb[0]) && mult8(a.sCb[1]) && mult8(a.sCb[2]);
    ok = ok && mult8(a.sAK0) && mult8(a.sAb[0]) && mult8(a.sAb[1]) && mult8(a.sAb[2]);
    ok = ok && mult8(a.sBK0) && mult8(a.sBb[0]) && mult8(a.sBb[1]) && mult8(a.sBb[2]);
    if (akc) ok = ok && mult8(a.K1) && mult8(a.sAM); else ok = ok && mult8(a.M) && mult8(a.sAK1);
    if (bkc) ok = ok && mult8(a.K1) && mult8(a.sBN); else ok = ok && mult8(a.N) && mult8(a.sBK1);
    return ok && tiles_take(TileProduct{a, akc, bkc}) ? 1 : 0;
}

// Whole 256 x 256 tiles: the shape the eight-wave kernel takes.
bool whole_256(const GemmArgs& a) { return a.M % 256 == 0 && a.N % 256 == 0 && a.K1 % BK == 0 && a.splits == 1; }

// Do these tiles keep the CUs busy?  Asked for the products with an activation in their epilogue, which other tiles do not have.
// With an operand that is read through the slower LDS transpose path the bar is higher: three quarters of a round
// is not enough then (measured).
bool fills_256(const GemmArgs& a, long batch, bool akc, bool bkc) {
    const long tiles = (long)(a.M / 256) * (a.N / 256) * batch;
    const double fill = (double)tiles / (double)((tiles + 255) / 256 * 256);
    return whole_256(a) && fill >= (akc && bkc ? 0.7 : 0.9);
}

template <int TM, int TN, int S, int NW, int EPI>
void launch_dma3(const GemmArgs& a, bool akc, bool bkc, dim3 grid, hipStream_t st) {
    if (akc && bkc) hipLaunchKernelGGL((k_gemm_dma<TM, TN, true, true, S, NW, EPI>), grid, dim3(NW * 64), 0, st, a);
    else if (akc) hipLaunchKernelGGL((k_gemm_dma<TM, TN, true, false, S, NW, EPI>), grid, dim3(NW * 64), 0, st, a);
    else if (bkc) hipLaunchKernelGGL((k_gemm_dma<TM, TN, false, true, S, NW, EPI>), grid, dim3(NW * 64), 0, st, a);
    else hipLaunchKernelGGL((k_gemm_dma<TM, TN, false, false, S, NW, EPI>), grid, dim3(NW * 64), 0, st, a);
}

template <int TM, int TN, int S, int NW>
void launch_dma2(const GemmArgs& a, bool akc, bool bkc, dim3 grid, hipStream_t st) {
    if (a.relu_dropout || a.gate) {
        // only the eight-wave 256x256 kernel carries these epilogues
        if constexpr (NW == 8) {
            if (a.gate && a.act == ACT_GELU) launch_dma3<TM, TN, S, NW, EPI_GELU_GATE_COLSUM>(a, akc, bkc, grid, st);
            else if (a.gate) launch_dma3<TM, TN, S, NW, EPI_GATE_COLSUM>(a, akc, bkc, grid, st);
            else if (a.act == ACT_GELU) launch_dma3<TM, TN, S, NW, EPI_GELU_DROPOUT>(a, akc, bkc, grid, st);
            else if (a.keep_words) launch_dma3<TM, TN, S, NW, EPI_RELU_DROPOUT_PRE>(a, akc, bkc, grid, st);
            else launch_dma3<TM, TN, S, NW, EPI_RELU_DROPOUT>(a, akc, bkc, grid, st);
            return;
        } else {
            fail("gemm: this kernel variant has no ReLU-dropout or gate epilogue");
        }
    }
    launch_dma3<TM, TN, S, NW, EPI_PLAIN>(a, akc, bkc, grid, st);
}

void launch_dma(const GemmArgs& a, bool akc, bool bkc, long batch, hipStream_t st) {
    const long tiles = (long)(a.M / 256) * (a.N / 256) * batch;
    if (tiles > 0x7fffffffL - a.side_blocks) fail("gemm: too many tiles");
    launch_dma2<4, 2, 2, 8>(a, akc, bkc, dim3((unsigned)tiles + a.side_blocks), st);
}

void launch_splitk_reduce(const GemmArgs& a, hipStream_t st) {
    const long n = a.nbatch * (long)a.M * (a.N / 4);
    hipLaunchKernelGGL(k_gemm_splitk_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, a.nbatch);
}

constexpr size_t kSplitMaxOut = 2u << 20;     // largest output (elements) whose contraction is split
constexpr long kSplitTarget = 256;            // workgroups a split product aims for (the CUs of the device)

// How many ways to split k so that a small output still fills the chip: the
// weight-gradient products have few output tiles and a long contraction.
int pick_splits(const GemmArgs& a, long batch, size_t ws_floats) {
    const long tiles = (long)((a.M + 127) / 128) * ((a.N + 127) / 128) * batch;
    const int nkt = a.K0 * ((a.K1 + BK - 1) / BK);
    // one workgroup per CU: a second, partly filled round costs more than it gains
    int splits = (int)(kSplitTarget / tiles);
    if (splits > 8) splits = 8;
    while (splits > 1 && nkt / splits < 8) --splits;
    const size_t need = (size_t)batch * a.M * a.N;          // floats per split
    while (splits > 1 && need * splits > ws_floats) --splits;
    if (a.N % 4 != 0) splits = 1;
    return splits < 1 ? 1 : splits;
}

}  // namespace

int gemm_kernel_kind(const GemmShape& s, const void* A, const void* B, const void* C,
                     const GemmEpilogue& ep) {
    Canon c = canonicalise(s, (const half_t*)A, (const half_t*)B, (half_t*)C, 1.f, ep);
    bool akc, bkc;
    return pick_kind(c, akc, bkc);
}

bool gemm_relu_dropout_ok(const GemmShape& s, const void* A, const void* B, const void* C,
                          const GemmEpilogue& ep) {
    if (s.batch() != 1 || s.sCN != 1 || s.sCM != s.N) return false;       // one dense row-major output
    Canon c = canonicalise(s, (const half_t*)A, (const half_t*)B, (half_t*)C, 1.f, ep);
    bool akc, bkc;
    return pick_kind(c, akc, bkc) == 1 && fills_256(c.a, 1, akc, bkc);
}

size_t gemm_splitk_ws_floats(const GemmShape& s) {
    // only small outputs are split (measured: beyond ~2M elements the fp32 partial
    // traffic costs more than the extra workgroups gain)
    size_t per = (size_t)s.batch() * s.M * s.N;
    long tiles = ((s.M + 127) / 128) * ((s.N + 127) / 128) * s.batch();
    if (tiles > kSplitTarget / 2 || per > kSplitMaxOut) return 0;
    size_t splits = kSplitTarget / tiles;
    if (splits > 8) splits = 8;
    return per * splits;
}

namespace {

// What launch_gemm_pair would launch: the two products as the kernel takes them and, when one is offered and
// its place in the launch costs less than a launch of its own, a third one.
struct PairSel {
    TileProduct p[3];
    TileChoice c;
    int n = 0;
};

// What a product takes in a launch of its own.
TileChoice choose_single(const TileProduct& p, size_t ws_floats) {
    return choose_tiles(&p, 1, kRingForms | (whole_256(p.a) ? 1u << TILE_256x256 : 0u), ws_floats);
}

bool pair_select(const GemmShape* const sh[2], const Canon cin[2], float* ws, size_t ws_floats, const PairThird* third,
                 PairSel& out) {
    constexpr double gap = 1.5;                          // between two launches (us)
    auto take = [&](int i, const Canon& c, const GemmShape& s) {
        out.p[i].a = c.a;
        out.p[i].a.nbatch = s.batch();
        return s.batch() > 0 && pick_kind(c, out.p[i].akc, out.p[i].bkc) == 1;
    };
    double alone = gap;
    for (int i = 0; i < 2; ++i) {
        if (!take(i, cin[i], *sh[i])) return false;
        alone += choose_single(out.p[i], ws_floats).us;
    }
    out.n = 2;
    out.c = choose_tiles(out.p, 2, kRingForms, ws_floats);
    if (out.c.form < 0 || out.c.us > alone) return false;
    if (third && third->shape &&
        take(2, canonicalise(*third->shape, third->A, third->B, third->C, third->alpha, GemmEpilogue{}), *third->shape)) {
        const TileChoice all = choose_tiles(out.p, 3, kRingForms, ws_floats);
        if (all.form >= 0 && all.us < out.c.us + gap + choose_single(out.p[2], ws_floats).us) { out.n = 3; out.c = all; }
    }
    if (out.c.splits > 1) {
        out.p[out.c.split].a.splits = out.c.splits;
        out.p[out.c.split].a.partial = ws;
    }
    return true;
}

}  // namespace

bool gemm_pair_ok(const GemmShape& s1, const half_t* A1, const half_t* B1, half_t* C1, const GemmEpilogue& ep1,
                  const GemmShape& s2, const half_t* A2, const half_t* B2, half_t* C2, const GemmEpilogue& ep2,
                  float* ws, size_t ws_floats) {
    const GemmShape* sh[2] = {&s1, &s2};
    const Canon c[2] = {canonicalise(s1, A1, B1, C1, 1.f, ep1), canonicalise(s2, A2, B2, C2, 1.f, ep2)};
    PairSel sel;
    return pair_select(sh, c, ws, ws_floats, nullptr, sel);
}

bool gemm_pair_takes_third(const GemmShape& s1, const half_t* A1, const half_t* B1, half_t* C1,
                           const GemmEpilogue& ep1, const GemmShape& s2, const half_t* A2, const half_t* B2,
                           half_t* C2, const GemmEpilogue& ep2, float* ws, size_t ws_floats,
                           const PairThird& third) {
    const GemmShape* sh[2] = {&s1, &s2};
    const Canon c[2] = {canonicalise(s1, A1, B1, C1, 1.f, ep1), canonicalise(s2, A2, B2, C2, 1.f, ep2)};
    PairSel sel;
    return pair_select(sh, c, ws, ws_floats, &third, sel) && sel.n == 3;
}

// Two or three products in one launch.  What it gains over launches of their own: the last round of the one is filled with
// tiles of the next, and a workgroup's way into a tile overlaps with the one before (dXlin1 + dWlin1 at 4096 x 1024 x 4096
// each: 78 -> 65 us against the launch of register-staged 256 x 128 tiles before, 75 for the two alone; at 2613 x 768 x 3072
// 77 -> 36 us).  Returns false, having launched nothing, where the products do not share a launch or are expected to be
// faster alone; the caller then launches them one after the other.
bool launch_gemm_pair(const GemmShape& s1, const half_t* A1, const half_t* B1, half_t* C1, float alpha1,
                      const GemmEpilogue& ep1, const GemmShape& s2, const half_t* A2, const half_t* B2,
                      half_t* C2, float alpha2, const GemmEpilogue& ep2, hipStream_t st, float* ws,
                      size_t ws_floats, FinishJobs* tail, PairThird* third) {
    const GemmShape* sh[2] = {&s1, &s2};
    const Canon cin[2] = {canonicalise(s1, A1, B1, C1, alpha1, ep1), canonicalise(s2, A2, B2, C2, alpha2, ep2)};
    PairSel sel;
    if (!pair_select(sh, cin, ws, ws_floats, third, sel)) return false;
    // (none of the column sums in `tail` may be one that this launch itself contributes to)
    launch_tiles(sel.p, sel.n, sel.c.form, tail, st);
    if (sel.n == 3) third->taken = true;
    if (sel.c.splits > 1) launch_splitk_reduce(sel.p[sel.c.split].a, st);
    check_launch("gemm pair");
    return true;
}

void launch_split_sums(const SplitSums& sums, half_t* C, long rows, long row, hipStream_t st) {
    GemmArgs a{};
    a.C = C; a.M = (int)rows; a.N = (int)row; a.sCM = row; a.sCN = 1; a.nb1 = a.nb2 = 1; a.nbatch = 1;
    a.alpha = sums.alpha; a.splits = sums.splits; a.partial = const_cast<float*>(sums.p);
    launch_splitk_reduce(a, st);
    check_launch("gemm split sums");
}

void launch_gemm(const GemmShape& s, const half_t* A, const half_t* B, half_t* C, float alpha,
                 const GemmEpilogue& ep, hipStream_t st, float* ws, size_t ws_floats, GemmSideJob* side) {
    long batch = s.batch();
    if (batch == 0 || s.M == 0 || s.N == 0) return;
    Canon c = canonicalise(s, A, B, C, alpha, ep);
    bool akc = false, bkc = false;
    int kind = pick_kind(c, akc, bkc);
    if (kind == 1) {
        TileProduct tp{c.a, akc, bkc};
        tp.a.nbatch = batch;
        const bool in_epilogue = ep.relu_dropout || ep.gate;
        if (in_epilogue && (!fills_256(c.a, batch, akc, bkc) || batch != 1 || s.sCN != 1 || s.sCM != s.N))
            fail("gemm: the ReLU-dropout epilogue needs the 256x256 asynchronous kernel (see gemm_relu_dropout_ok)");
        // A forward pass sums in an order that depends on the product's shape alone (pick_splits), whatever the tile.
        const bool small = ws && (size_t)batch * c.a.M * c.a.N <= kSplitMaxOut && !in_epilogue;
        if (small && !ep.any_split) tp.a.splits = pick_splits(c.a, batch, ws_floats);
        TileChoice choice;
        choice.form = TILE_256x256;
        if (!in_epilogue) choice = choose_single(tp, small && ep.any_split ? ws_floats : 0);
        if (side) side->tiles_done = 0;
        if (side && side->keep && side->key.thr && choice.form == TILE_256x256 && !in_epilogue) {
            // CUs the tiles leave idle draw attention keep bits meanwhile: what fits into the time the
            // product takes (about 9 us + 1.5 us per k-tile; the rate per CU and us is the measured break-even:
            // 12 of the 16 key tiles of the bench workload cost the launch 0.3 us, 14 cost it 2.5, all 16 6 us)
            const long tiles = (long)(c.a.M / 256) * (c.a.N / 256) * batch;
            const long idle = 256 - tiles, nkt = (long)c.a.K0 * (c.a.K1 / BK);
            if (tiles >= 128 && idle >= 32 && side->nk % 32 == 0) {
                const double groups = (double)idle * (9.0 + 1.5 * (double)nkt) * 1600.0;
                long td = (long)(groups / (4.0 * (double)side->rows));
                if (td > side->nk / 32) td = side->nk / 32;
                if (td > 0) {
                    c.a.side_first = (unsigned)tiles; c.a.side_blocks = (unsigned)idle;
                    c.a.side_key = side->key; c.a.side_keep = side->keep;
                    c.a.side_rows = side->rows; c.a.side_nk = side->nk; c.a.side_tiles_done = (uint32_t)td;
                    side->tiles_done = (uint32_t)td;
                }
            }
        }
        if (choice.form == TILE_256x256) {
            launch_dma(c.a, akc, bkc, batch, st);
        } else {
            tp.a.splits = choice.splits;
            if (tp.a.splits > 1) tp.a.partial = ws;
            launch_tiles(&tp, 1, choice.form, nullptr, st);
            if (tp.a.splits > 1) {
                if (ep.sums && batch == 1 && !tp.a.bias && tp.a.sCM == tp.a.N)
                    *ep.sums = SplitSums{ws, tp.a.splits, (long)tp.a.M * tp.a.N, alpha};
                else
                    launch_splitk_reduce(tp.a, st);
            }
        }
    } else {
        if (ep.relu_dropout || ep.gate) fail("gemm: the ReLU-dropout epilogue needs the MFMA kernel");
        const long blocks = batch * ((c.a.M + FB - 1) / FB) * ((c.a.N + FB - 1) / FB);
        if (blocks > 0x7fffffffL) fail("gemm: problem too large for the scalar kernel");
        auto words = [&](const half_t* p, long s_row, long s_k, long s_k0, const long (&sb)[3]) {
            return s_k == 1 && al16(p) && mult8(s_row) && mult8(c.a.K1) && mult8(s_k0) && mult8(sb[0]) && mult8(sb[1]) && mult8(sb[2]);
        };
        hipLaunchKernelGGL(k_gemm_fma, dim3((unsigned)blocks), dim3(256), 0, st, c.a,
                           words(c.a.A, c.a.sAM, c.a.sAK1, c.a.sAK0, c.a.sAb), words(c.a.B, c.a.sBN, c.a.sBK1, c.a.sBK0, c.a.sBb));
    }
    check_launch("gemm");
}

}  // namespace sub
