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

// ---------------------------------------------------------------------------
// Any strides, any sizes: what the half-precision matrix instructions do not take (mostly rows that are not whole 16-byte words: the
// score-sized products of sequence lengths that are not multiples of 8).  128 x 64 outputs per workgroup, 32 x 64 per wave, 32 k of
// both operands in LDS at a time, the next 32 on their way meanwhile.  Every output is one fp32 chain of fused multiply-adds in the
// order of k, which is what v_mfma_f32_32x32x2_f32 does with its two k (204800 sums of 256 compared with fmaf, bit for bit; k past the
// end are zeros in both operands, which leave a sum as it is).  With v_fma_f32, 4 x 4 outputs per thread, the same bits took half the
// rate at best, and eight times the reads from LDS.  us of the scores and of the product with V, before and now, H 12, P 64: 13 x 201
// 41 and 52, 24 and 30; 24 x 77 21 and 23, 14 and 15; 3 x 300 22 and 67, 15 and 30; 2 x 1500, H 16: 215 and 321, 109 and 172 (a third
// of that instruction's rate: the single elements of a row that starts anywhere).
// ---------------------------------------------------------------------------
// A product of up to 64 rows has tiles of 64 x 64, 32 x 32 per wave, where half of the waves would have none; one of up to 24 k goes by steps of
// 8, read one by one: with 32 a thread brings 24 elements, most of them zeros.  us with v_fma_f32, with 128 x 64 and 32 k alone, and now: product with
// V, H 12, P 64, 24 x 33 9.9, 11.1, 7.2; 1 x 1 4.4, 5.9, 3.7; 24 x 7 6.1, 6.7, 4.1; weight gradient of 4 rows, 2000 x 500, 5.9, 7.2, 5.4.  (17 to 24 k:
// 1024 x 5 of 20 7.6, 8.2, 6.9, the product with V of 1 x 17 6.6, 4.6 with 32, 5.0.)
constexpr int FN = 64;
typedef float f16v __attribute__((ext_vector_type(16)));
enum : int { FMA_SINGLE = 0, FMA_ALONG_K = 1, FMA_ALONG_ROWS = 2 };       // how an operand is read: whole 16-byte words or not

// What a thread brings of an operand's ROWS x FK elements: words, or elements that lie side by side over the threads along k or
// along the rows.  What lies outside is read from a place that there is, and put down as zero where it is a k: no branch around a
// load, where the wait for it would go.  Single elements are kept apart: of two in a register, the second's load waits for the first's.
// In LDS [row][k], as half values: 16 bytes are four steps of a matrix instruction.
template <int ROWS, int HOW, int FK>
struct FmaPart {
    static constexpr int N = ROWS * FK / 256, WORDS = HOW == FMA_SINGLE ? 1 : N / 8, L = HOW == FMA_SINGLE ? N : WORDS, FPITCH = FK + 8;
    static_assert(HOW == FMA_SINGLE || FK == 32, "words of 8 k");
    int row, k, drow, dk;                    // of the first, and on to the next
    h8 word[WORDS];
    uint16_t one[N];
    __device__ __forceinline__ FmaPart(bool k_first, int tid) {
        if (HOW == FMA_ALONG_K) { row = tid >> 2; k = (tid & 3) * 8; drow = 64; dk = 0; }
        else if (HOW == FMA_ALONG_ROWS) { row = tid % (ROWS / 8) * 8; k = tid / (ROWS / 8); drow = 0; dk = 256 / (ROWS / 8); }
        else if (k_first) { row = tid / FK; k = tid % FK; drow = 256 / FK; dk = 0; }
        else { row = tid % ROWS; k = tid / ROWS; drow = 0; dk = 256 / ROWS; }
    }
    // (p: the step's first element, of which there are rows x ks.  Spelled out as memory that is not LDS.)
    __device__ __forceinline__ void fetch(const half_t* p, long s_row, long s_k, int rows, int ks) {
        const long first = row < rows && k < ks ? (long)row * s_row + (long)k * s_k : 0, step = (long)drow * s_row + (long)dk * s_k;
        const __attribute__((address_space(1))) half_t* const q = (const __attribute__((address_space(1))) half_t*)p + first;
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const bool in = row + i * drow < rows && k + i * dk < ks;
            const auto at = q + (in ? i * step : 0);
            if constexpr (HOW == FMA_SINGLE) one[i] = *(const __attribute__((address_space(1))) uint16_t*)at;
            else word[i] = *(const __attribute__((address_space(1))) h8*)at;
        }
    }
    __device__ __forceinline__ void put(half_t (*to)[FPITCH], int ks) const {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const bool in = k + i * dk < ks;
            if constexpr (HOW == FMA_SINGLE) to[row + i * drow][k + i * dk] = in ? __builtin_bit_cast(half_t, one[i]) : (half_t)0.0f;
            else {
                const h8 v = in ? word[i] : (h8)(half_t)0.0f;
                if constexpr (HOW == FMA_ALONG_K) *reinterpret_cast<h8*>(&to[row + i * drow][k]) = v;
                else
#pragma unroll
                    for (int e = 0; e < 8; ++e) to[row + e][k + i * dk] = v[e];
            }
        }
    }
};

template <int HOW_A, int HOW_B, int FM, int FK>
__global__ __launch_bounds__(256, 4) void k_gemm_fma(GemmArgs g) {
    constexpr int FPITCH = FK + 8, NACC = FM / 64;
    __shared__ __attribute__((aligned(16))) half_t ta[2][FM][FPITCH], tb[2][FN][FPITCH];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % (FM / 32) * 32, wn = wave / (FM / 32) * 32;
    const unsigned tiles_m = (g.M + FM - 1) / FM, tiles_n = (g.N + FN - 1) / FN;
    unsigned id = blockIdx.x;
    const unsigned n0 = id % tiles_n * FN; id /= tiles_n;
    const unsigned m0 = id % tiles_m * FM; id /= tiles_m;
    const long b2 = id % g.nb2; id /= g.nb2;
    const long b1 = id % g.nb1, b0 = id / g.nb1;
    const half_t* const a = g.A + b0 * g.sAb[0] + b1 * g.sAb[1] + b2 * g.sAb[2] + (long)m0 * g.sAM;
    const half_t* const b = g.B + b0 * g.sBb[0] + b1 * g.sBb[1] + b2 * g.sBb[2] + (long)n0 * g.sBN;
    const int rows = min(g.M - (int)m0, FM), cols = min(g.N - (int)n0, FN);
    FmaPart<FM, HOW_A, FK> pa(g.sAK1 == 1, tid);
    FmaPart<FN, HOW_B, FK> pb(g.sBK1 == 1, tid);
    const bool working = wm < rows && wn < cols;             // (a wave whose outputs all lie outside only helps with the operands)
    f16v acc[NACC];
#pragma unroll
    for (int v = 0; v < 16 * NACC; ++v) acc[v / 16][v % 16] = 0.f;
    auto fetch = [&](int k0, int k) __attribute__((always_inline)) {
        pa.fetch(a + (long)k0 * g.sAK0 + (long)k * g.sAK1, g.sAM, g.sAK1, rows, g.K1 - k);
        pb.fetch(b + (long)k0 * g.sBK0 + (long)k * g.sBK1, g.sBN, g.sBK1, cols, g.K1 - k);
    };
    fetch(0, 0);
    int buf = 0;
    for (int k0 = 0; k0 < g.K0; ++k0)
        for (int k = 0; k < g.K1; k += FK) {
            const int ks = min(FK, g.K1 - k);
            pa.put(ta[buf], ks);
            pb.put(tb[buf], ks);
            __syncthreads();                                 // (the other buffer is free as well: every wave is done with the step before)
            const bool same = k + FK < g.K1;
            if (same || k0 + 1 < g.K0) fetch(same ? k0 : k0 + 1, same ? k + FK : 0);
            if (working) {
                // (the halves of the wave take the k of a pair: half a register each)
                auto value = [&](uint32_t pair) __attribute__((always_inline)) {
                    return (float)__builtin_bit_cast(half_t, (uint16_t)(pair >> (16 * hi)));
                };
                typedef uint32_t u4 __attribute__((ext_vector_type(4)));
                auto read = [&](const half_t* p) __attribute__((always_inline)) { return *reinterpret_cast<const u4*>(p); };
                constexpr int R = FK < 16 ? 1 : 2;           // reads of 8 k
                const half_t *const x = ta[buf][wm + l32], *const y = tb[buf][wn + l32];
                for (int i = 0; i < ks; i += 8 * R) {
                    u4 fx[R], fy[NACC][R];
#pragma unroll
                    for (int r = 0; r < R; ++r) fx[r] = read(x + i + 8 * r);
#pragma unroll
                    for (int r = 0; r < NACC * R; ++r) fy[r / R][r % R] = read(y + r / R * 32 * FPITCH + i + 8 * (r % R));
#pragma unroll
                    for (int p = 0; p < 4 * R; ++p) {
                        const float xv = value(fx[p >> 2][p & 3]);
#pragma unroll
                        for (int t = 0; t < NACC; ++t)
                            acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv, value(fy[t][p >> 2][p & 3]), acc[t], 0, 0, 0);
                    }
                }
            }
            buf ^= 1;
        }
    if (!working) return;
    // register v of a lane: row 8 (v / 4) + 4 hi + v % 4 of the wave's, column l32 of 32.  Of 64 columns the halves of the wave trade, so that
    // a lane has column `lane` of rows 8 (v / 4) + v % 4 and of those 4 further: rows of 128 bytes for an instruction.
    const int n = (int)n0 + (NACC == 2 ? lane : wn + l32);
    half_t* const c = g.C + b0 * g.sCb[0] + b1 * g.sCb[1] + b2 * g.sCb[2] + (long)n * g.sCN;
    auto store = [&](int m, float sum) __attribute__((always_inline)) {
        if (m >= g.M || n >= g.N) return;
        half_t out = (half_t)(sum * g.alpha);
        if (g.bias)     // same two roundings as the product followed by a separate add
            out = (half_t)((float)out + (float)g.bias[b0 * g.sbb[0] + b1 * g.sbb[1] + b2 * g.sbb[2] +
                                                      (long)m * g.sbM + (long)n * g.sbN]);
        c[(long)m * g.sCM] = out;
    };
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int m = (int)m0 + wm + (v >> 2) * 8 + (v & 3);
        if constexpr (NACC == 2) {
            const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[0][v]), __float_as_uint(acc[1][v]), false, false);
            store(m, __uint_as_float(both[0]));
            store(m + 4, __uint_as_float(both[1]));
        } else {
            store(m + 4 * hi, acc[0][v]);
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
    a.keep_words = ep.keep_words; a.act = ep.act; a.pre_out = ep.pre_out; a.alone = ep.alone ? 1 : 0; a.same_order = ep.same_order ? 1 : 0;
    if (ep.alone) a.gate_bits_out = nullptr;
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
    if (a.act == ACT_GELU && a.relu_dropout && !(a.pre_out && al16(a.pre_out) && (a.gate_bits_out || a.alone) && !a.keep_words)) return 0;
    // every 16-byte access must be aligned and whole
    bool ok = mult8(a.N) && mult8(a.sCM) && mult8(a.sCb[0]) && mult8(a.sCb[1]) && mult8(a.sCb[2]);
    ok = ok && mult8(a.sAK0) && mult8(a.sAb[0]) && mult8(a.sAb[1]) && mult8(a.sAb[2]);
    ok = ok && mult8(a.sBK0) && mult8(a.sBb[0]) && mult8(a.sBb[1]) && mult8(a.sBb[2]);
    if (akc) ok = ok && mult8(a.K1) && mult8(a.sAM); else ok = ok && mult8(a.M) && mult8(a.sAK1);
    if (bkc) ok = ok && mult8(a.K1) && mult8(a.sBN); else ok = ok && mult8(a.N) && mult8(a.sBK1);
    return ok && tiles_take(TileProduct{a, akc, bkc}) ? 1 : 0;
}

void launch_splitk_reduce(const GemmArgs& a, hipStream_t st) {
    const long n = a.nbatch * (long)a.M * (a.N / 4);
    hipLaunchKernelGGL(k_gemm_splitk_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, a.nbatch);
}

constexpr size_t kSplitMaxOut = 2u << 20;     // largest output (elements) whose contraction is split
constexpr long kSplitTarget = 256;            // workgroups a split product aims for (the CUs of the device)

// Scratch (floats) for the sums of a product's splits.  Only small outputs are split (measured: beyond ~2M elements the fp32
// partial traffic costs more than the extra workgroups gain).
size_t split_floats(long M, long N, long batch) {
    const size_t per = (size_t)batch * M * N;
    const long tiles = ((M + 127) / 128) * ((N + 127) / 128) * batch;
    if (tiles > kSplitTarget / 2 || per > kSplitMaxOut) return 0;
    return per * (size_t)std::min(kSplitTarget / tiles, 8L);
}

unsigned forms_for(const TileProduct* p, int n) {
    unsigned forms = kRingForms | 1u << TILE_256x256;
    for (int i = 0; i < n; ++i)
        if (!wide_takes(p[i])) forms = kRingForms;
    return forms;
}

// What a product takes in a launch of its own.
TileChoice choose_single(const TileProduct& p, size_t ws_floats, double reduce_us = kReduceLaunch) {
    return choose_tiles(&p, 1, forms_for(&p, 1), ws_floats, reduce_us);
}

// In how many parts a forward pass sums a product, by its shape and the order of its operands alone: as is fastest, within the
// scratch that every caller brings.  A product that does not widen its rows has a LayerNorm behind it in the layers, which takes
// the parts in place of their sum (3.9 us without, 5.7 with six parts of 64 x 768, 0.6 of that for their bytes).  (Splits to fill
// the CUs as far as 8 steps each were left of it, which was the rule here before, cost more than they gave where the fp32 sums are
// many: us of lin2 and the LayerNorm behind it, 2613 x 768 x 3072 in two parts 32 and in one 29, 1024 x 768 x 3072 in five 21.4
// and in one 19.9; and a product of 512 x 4096 x 1024 in two parts had no activation in its epilogue, 28 with its activation and
// now 14.)
// In front of a ReLU the rule is that of old, which fills the CUs as long as eight steps a part are left of it.
int forward_splits(const TileProduct& p) {
    if (p.a.same_order) {
        const long tiles = (long)((p.a.M + 127) / 128) * ((p.a.N + 127) / 128) * p.a.nbatch;
        const int nkt = p.a.K0 * ((p.a.K1 + BK - 1) / BK);
        int splits = (int)std::min(kSplitTarget / tiles, 8L);
        while (splits > 1 && nkt / splits < 8) --splits;
        return p.a.N % 4 != 0 || (size_t)p.a.nbatch * p.a.M * p.a.N > kSplitMaxOut ? 1 : std::max(splits, 1);
    }
    const bool widens = p.a.N > (long)p.a.K0 * p.a.K1;
    return choose_single(p, split_floats(p.a.M, p.a.N, p.a.nbatch), widens ? kReduceLaunch : 1.4).splits;
}

}  // namespace

int gemm_kernel_kind(const GemmShape& s, const void* A, const void* B, const void* C,
                     const GemmEpilogue& ep) {
    Canon c = canonicalise(s, (const half_t*)A, (const half_t*)B, (half_t*)C, 1.f, ep);
    bool akc, bkc;
    return pick_kind(c, akc, bkc);
}

// The tiles that a product with an activation in its epilogue runs in, -1 if it does not.
static int act_form(const GemmShape& s, const void* A, const void* B, const void* C, const GemmEpilogue& ep) {
    if (s.batch() != 1 || s.sCN != 1 || s.sCM != s.N || s.N % 32 != 0) return -1;       // one dense row-major output
    TileProduct p;
    Canon c = canonicalise(s, (const half_t*)A, (const half_t*)B, (half_t*)C, 1.f, ep);
    if (pick_kind(c, p.akc, p.bkc) != 1) return -1;
    p.a = c.a; p.a.nbatch = 1;
    // A small output whose contraction a forward pass splits keeps the order of its sums, with or without an activation behind
    // it: split, and the operators.
    if (forward_splits(p) > 1) return -1;
    return choose_act_form(p);
}

bool gemm_relu_dropout_ok(const GemmShape& s, const void* A, const void* B, const void* C,
                          const GemmEpilogue& ep) {
    return act_form(s, A, B, C, ep) >= 0;
}

int gemm_colsum_rows(const GemmShape& s, const void* A, const void* B, const void* C, const GemmEpilogue& ep) {
    const int form = act_form(s, A, B, C, ep);
    if (form < 0) fail("gemm: no activation in this product's epilogue (see gemm_relu_dropout_ok)");
    const long bm = tile_form(form).bm;
    return (int)(2 * ((s.M + bm - 1) / bm));             // two rows of waves
}

size_t gemm_splitk_ws_floats(const GemmShape& s) {
    return split_floats(s.M, s.N, s.batch());
}

namespace {

constexpr double kGap = 1.5;                             // between two launches (us)

// A job as the kernel takes it.
bool take(const GemmJob& j, TileProduct& p) {
    if (j.shape->batch() == 0 || j.shape->M == 0 || j.shape->N == 0) return false;
    const Canon c = canonicalise(*j.shape, j.A, j.B, j.C, j.alpha, j.ep);
    p.a = c.a;
    p.a.nbatch = j.shape->batch();
    return pick_kind(c, p.akc, p.bkc) == 1;
}

}  // namespace

void GemmLaunch::drop(int j) {
    for (int i = 0; i < n; ++i)
        if (job[i] == j) {
            if (split == i) splits = 1;
            if (split >= i && split > 0) --split;
            for (--n; i < n; ++i) job[i] = job[i + 1];
            return;
        }
}

// Several products in one launch.  What it gains over launches of their own: the last round of the one is filled with
// tiles of the next, and a workgroup's way into a tile overlaps with the one before (dXlin1 + dWlin1 at 4096 x 1024 x 4096
// each: 78 -> 65 us against the launch of register-staged 256 x 128 tiles before, 75 for the two alone; at 2613 x 768 x 3072
// 77 -> 36 us).
double plan_gemm_stage(const GemmJob* jobs, const int* ids, int n, bool together, size_t ws_floats, GemmStage& out) {
    TileProduct p[kMaxProducts];
    int id[kMaxProducts], m = 0;                         // the jobs that tiles take
    double alone[kMaxProducts], sum = 0.;
    out.n = 0;
    auto launch = [&](const int* job, int count) -> GemmLaunch& {
        GemmLaunch& l = out.launch[out.n++];
        l = GemmLaunch{};
        l.n = count;
        for (int i = 0; i < count; ++i) l.job[i] = job[i];
        return l;
    };
    for (int i = 0; i < n; ++i) {
        sum += i ? kGap : 0.;
        if (!take(jobs[ids[i]], p[m])) {                 // (misaligned, say: by itself, and the others without it)
            launch(ids + i, 1);
            continue;
        }
        const bool small = (size_t)p[m].a.nbatch * p[m].a.M * p[m].a.N <= kSplitMaxOut;
        alone[m] = choose_single(p[m], small ? ws_floats : 0).us;
        sum += alone[m];
        id[m++] = ids[i];
    }
    const double in_front = kGap * out.n;
    double best = sum;
    TileChoice how;
    int from = m;                                        // jobs `from` .. of the list in one launch, those in front of it alone
    for (int f : {1, 0}) {
        if (!together || m - f < 2) continue;
        const TileChoice c = choose_tiles(p + f, m - f, forms_for(p + f, m - f), ws_floats);
        const double us = in_front + c.us + (f ? alone[0] + kGap : 0.);
        if (c.form < 0 || us >= best) continue;
        best = us; how = c; from = f;
    }
    for (int i = 0; i < from; ++i) launch(id + i, 1);
    if (from < m) {
        GemmLaunch& l = launch(id + from, m - from);
        l.form = how.form; l.split = how.split; l.splits = how.splits;
    }
    return best;
}

void plan_backward_products(const GemmJob (&jobs)[7], bool together, bool late, size_t ws_floats, BackwardPlan& out) {
    // what every place takes with every set of the weight gradients that may wait (bits 0, 1, 2: jobs 1, 2, 4)
    GemmStage plan[3][8];
    double us[3][8];
    for (int at = 0; at < 3; ++at)
        for (int set = 0; set < (at ? 8 : 4); ++set) {
            if (!together && set != (at == 0 ? 3 : at == 1 ? 4 : 0)) continue;
            int ids[kMaxProducts], n = 0;
            ids[n++] = at == 0 ? 0 : at == 1 ? 3 : 5;
            if (at == 2) ids[n++] = 6;
            if (set & 4) ids[n++] = 4;
            if (set & 1) ids[n++] = 1;
            if (set & 2) ids[n++] = 2;
            us[at][set] = plan_gemm_stage(jobs, ids, n, together, ws_floats, plan[at][set]);
        }
    double best = -1.;
    for (int w1 = 0; w1 < (together ? 3 : 1); ++w1)
        for (int w2 = 0; w2 < (together ? 3 : 1); ++w2)
            for (int wo = 1; wo < (together && late ? 3 : 2); ++wo) {
                int set[3] = {0, 0, 0};
                set[w1] |= 1; set[w2] |= 2; set[wo] |= 4;
                const double t = us[0][set[0]] + us[1][set[1]] + us[2][set[2]];
                if (best >= 0. && t >= best) continue;
                best = t;
                for (int at = 0; at < 3; ++at) out.stage[at] = plan[at][set[at]];
            }
}

void launch_gemm_together(const GemmJob* jobs, const GemmLaunch& l, hipStream_t st, float* ws, size_t ws_floats, FinishJobs* tail) {
    TileProduct p[kMaxProducts];
    int k1, k2;
    bool fits = l.form >= 0 && l.form < TILE_FORMS;
    for (int i = 0; i < l.n; ++i) {
        fits = fits && take(jobs[l.job[i]], p[i]) && (l.form != TILE_256x256 || (l.splits == 1 && wide_takes(p[i])));
        if (fits && l.splits > 1 && l.split == i) {
            fits = p[i].a.N % 4 == 0 && (size_t)p[i].a.nbatch * p[i].a.M * p[i].a.N * l.splits <= ws_floats;
            p[i].a.splits = l.splits;
            p[i].a.partial = ws;
        }
    }
    if (!fits || !orientations(p, l.n, k1, k2)) {
        // (a plan that is not one for these products: none that is kept should be)
        for (int i = 0; i < l.n; ++i) {
            const GemmJob& j = jobs[l.job[i]];
            launch_gemm(*j.shape, j.A, j.B, j.C, j.alpha, j.ep, st, ws, ws_floats);
        }
        return;
    }
    // (none of the column sums in `tail` may be one that this launch itself contributes to)
    launch_tiles(p, l.n, l.form, tail, st);
    if (l.splits > 1) launch_splitk_reduce(p[l.split].a, st);
    check_launch("gemm group");
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
        if (ep.relu_dropout || ep.gate) {
            const int form = act_form(s, A, B, C, ep);
            if (form < 0 || alpha != 1.0f) fail("gemm: no activation in this product's epilogue (see gemm_relu_dropout_ok)");
            launch_tiles_act(tp, form, st);
            check_launch("gemm");
            return;
        }
        const bool small = ws && (size_t)batch * c.a.M * c.a.N <= kSplitMaxOut;
        if (small && !ep.any_split) {
            tp.a.splits = forward_splits(tp);
            if (tp.a.splits > 1 && (size_t)batch * c.a.M * c.a.N * tp.a.splits > ws_floats)
                fail("gemm: scratch for the sums of a split product is smaller than gemm_splitk_ws_floats");
        }
        const unsigned forms = !tp.a.same_order ? forms_for(&tp, 1) : summed_wide(tp) ? 1u << TILE_256x256 : kRingForms;
        const TileChoice choice = choose_tiles(&tp, 1, forms, small && ep.any_split ? ws_floats : 0);
        unsigned side_blocks = 0;
        if (side) side->tiles_done = 0;
        if (side && side->keep && side->key.thr && choice.form == TILE_256x256 && choice.splits == 1) {
            // CUs the tiles leave idle draw attention keep bits meanwhile: what fits into the time the
            // product takes (about 9 us + 1.5 us per k-tile; the rate per CU and us is the measured break-even.  At 8 x 512, E 1024,
            // us of this launch and of the attention behind it with 10 of the 16 key tiles drawn here: 32.5 and 23.5, 11: 32.5 and
            // 23.1, 12 (what the rule gives): 32.5 and 22.7, 14: 34.7 and 22.0, all 16: 38.3 and 20.9)
            const long tiles = (long)((c.a.M + 255) / 256) * ((c.a.N + 255) / 256) * batch;
            const long idle = 256 - tiles, nkt = (long)c.a.K0 * ((c.a.K1 + BK - 1) / BK);
            if (tiles >= 128 && idle >= 32 && side->nk % 32 == 0) {
                const double groups = (double)idle * (9.0 + 1.5 * (double)nkt) * 1600.0;
                long td = (long)(groups / (4.0 * (double)side->rows));
                if (td > side->nk / 32) td = side->nk / 32;
                if (td > 0) {
                    side_blocks = (unsigned)idle;
                    c.a.side_key = side->key; c.a.side_keep = side->keep;
                    c.a.side_rows = side->rows; c.a.side_nk = side->nk; c.a.side_tiles_done = (uint32_t)td;
                    side->tiles_done = (uint32_t)td;
                }
            }
        }
        tp.a = c.a; tp.a.nbatch = batch;
        if (side_blocks) {
            launch_wide(&tp, 1, nullptr, side_blocks, st);
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
        const bool low = c.a.M <= 64;
        const long blocks = batch * (low ? 1 : (c.a.M + 127) / 128) * ((c.a.N + FN - 1) / FN);
        if (blocks > 0x7fffffffL) fail("gemm: problem too large for the scalar kernel");
        const bool few_k = c.a.K1 <= 24;
        // whole 16-byte words along k, or else along the operand's rows (of the output: m resp. n)
        auto how = [&](const half_t* p, long rows, long s_row, long s_k, long s_k0, const long (&sb)[3]) {
            const bool apart = al16(p) && mult8(s_k0) && mult8(sb[0]) && mult8(sb[1]) && mult8(sb[2]);
            if (apart && s_k == 1 && mult8(s_row) && mult8(c.a.K1)) return FMA_ALONG_K;
            return apart && s_row == 1 && mult8(s_k) && mult8(rows) ? FMA_ALONG_ROWS : FMA_SINGLE;
        };
        const int how_a = how(c.a.A, c.a.M, c.a.sAM, c.a.sAK1, c.a.sAK0, c.a.sAb), how_b = how(c.a.B, c.a.N, c.a.sBN, c.a.sBK1, c.a.sBK0, c.a.sBb);
        auto launch = [&](auto ha, auto hb, auto fk) {
            const dim3 grid((unsigned)blocks);
            if (low) hipLaunchKernelGGL((k_gemm_fma<ha(), hb(), 64, fk()>), grid, dim3(256), 0, st, c.a);
            else hipLaunchKernelGGL((k_gemm_fma<ha(), hb(), 128, fk()>), grid, dim3(256), 0, st, c.a);
        };
        auto run = [&](auto ha) {
            auto with = [&](auto hb) { launch(ha, hb, std::integral_constant<int, 32>{}); };
            if (how_b == FMA_ALONG_K) with(std::integral_constant<int, FMA_ALONG_K>{});
            else if (how_b == FMA_ALONG_ROWS) with(std::integral_constant<int, FMA_ALONG_ROWS>{});
            else with(std::integral_constant<int, FMA_SINGLE>{});
        };
        if (few_k) launch(std::integral_constant<int, FMA_SINGLE>{}, std::integral_constant<int, FMA_SINGLE>{}, std::integral_constant<int, 8>{});
        else if (how_a == FMA_ALONG_K) run(std::integral_constant<int, FMA_ALONG_K>{});
        else if (how_a == FMA_ALONG_ROWS) run(std::integral_constant<int, FMA_ALONG_ROWS>{});
        else run(std::integral_constant<int, FMA_SINGLE>{});
    }
    check_launch("gemm");
}

}  // namespace sub
