// What the contraction kernels share: their arguments, the asynchronous operand tiles, the reductions behind a split.
#pragma once

#include "sub_ops.hpp"

namespace sub {

constexpr int BK = 64;            // k per LDS tile

typedef float f16v __attribute__((ext_vector_type(16)));

struct GemmArgs {
    const half_t* A; const half_t* B; half_t* C;
    int M, N, K1, K0;
    long sAM, sAK1, sAK0;
    long sBN, sBK1, sBK0;
    long sCM, sCN;
    int nb1, nb2;                 // sizes of batch dims 1 and 2 (dim 0 is the quotient)
    long sAb[3], sBb[3], sCb[3];
    float alpha;
    const half_t* bias; long sbM, sbN, sbb[3];
    int splits;                   // > 1: the k range is split, fp32 partial tiles go to `partial`
    float* partial;               // [split][batch][M][N]
    long nbatch = 1;              // batches in all
    int relu_dropout = 0;         // the activation and dropout after the addend
    PhiloxKey key;
    const half_t* gate = nullptr; // or: the activation's backward pass (strides of `bias`), with column sums per row of waves
    float* colsum = nullptr;
    const uint32_t* keep_words = nullptr;  // relu_dropout: the keep bits, drawn ahead (relu_dropout_keep_words)
    uint32_t* gate_bits_out = nullptr;     // relu_dropout: one bit per output, set where it is positive
    const uint32_t* gate_bits = nullptr;   // gate: those bits instead of the values of `gate`
    int act = ACT_RELU;                    // the activation of relu_dropout / gate (GemmEpilogue::act)
    half_t* pre_out = nullptr;             // GELU with dropout: where the rounded sum before the activation goes
    int same_order = 0;                    // GemmEpilogue::same_order
    int alone = 0;                         // no backward pass follows (GemmEpilogue::alone)
    // GemmSideJob of the 256 x 256 kernel: the workgroups behind those of the tiles draw
    // the attention keep words of key tiles 0 .. side_tiles_done - 1 of side_rows score rows
    PhiloxKey side_key;
    uint32_t* side_keep = nullptr;
    uint32_t side_rows = 0, side_nk = 0, side_tiles_done = 0;
};

// The arguments every tile of a product needs, fetched in one go at the start of the workgroup
// (fetch_args_now): the index arithmetic between them would otherwise be interleaved with four or
// five scalar round trips.
template <typename Args>
__device__ __forceinline__ void fetch_gemm_args(Args& g) {
    fetch_args_now(g.A, g.B, g.C, g.M, g.N, g.K1, g.K0, g.sAM, g.sAK1, g.sAK0, g.sBN, g.sBK1, g.sBK0, g.sCM, g.nb1, g.nb2,
                   g.sAb[0], g.sAb[1], g.sAb[2], g.sBb[0], g.sBb[1], g.sBb[2], g.sCb[0], g.sCb[1], g.sCb[2], g.alpha,
                   g.bias, g.sbM, g.splits);
}

typedef short s4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef __attribute__((address_space(1))) const void* global_void_ptr;

constexpr int waitcnt_vm(int vm) { return (vm & 0xF) | ((vm >> 4) << 14) | 0x0F70; }

// FRAG: rows of the fragments that are read from it (of v_mfma_f32_32x32x16_f16, of v_mfma_f32_16x16x32_f16).
//
// Where the 16-byte units go is what keeps the lanes that LDS serves at a time in different banks (64 of 4 bytes): of 16-byte
// reads lanes 0-3, 12-15 and 20-27 together, lanes 4-11, 16-19 and 28-31, and the same 32 further; of transposing 8-byte reads lanes 0-31.
// That is what the counters of these kernels fit: with the order for 32-row fragments, 16-row fragments had as many conflict
// cycles as cycles of use, by both kinds of reads, 32-row ones none.
template <int ROWS, bool KC, int NW, int FRAG = 32>
struct DTile {
    static constexpr int HALVES = ROWS * BK;
    static constexpr int NV = ROWS / (8 * NW);      // loads per thread: the tile is ROWS / 8 slabs of 1024 bytes
    static constexpr int VPR = ROWS / 8;            // 16-byte units per k-row (!KC)

    static __device__ __forceinline__ int kc_swz(int row) { return FRAG == 16 ? row >> 1 : row ^ (row >> 3); }
    static __device__ __forceinline__ int kc_off(int row, int slot) {
        return row * BK + ((slot ^ kc_swz(row)) & 7) * 8;
    }
    // !KC: [k][free] with the 16-byte unit index xor-ed so that the four k-rows a
    // 16-lane group of the transpose read touches fall into different banks; two such groups next to each other
    // are 16 rows apart in a 32-row fragment and 8 k apart in a 16-row one.
    static __device__ __forceinline__ int mc_swz(int k) {
        if (FRAG == 16) return ((k & 3) << 2) | (((k >> 3) & 1) << 1);
        return VPR >= 16 ? ((k & 3) << 2) : (((k >> 1) & 1) << 2);
    }

    // Element offset (from the tile's first element in global memory) of the
    // chunk lane `lane` of wave `wave` fetches with its i-th load.
    static __device__ __forceinline__ void offsets(unsigned (&off)[NV], long sF, long sK, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int inst = wave * NV + i;          // which 1024-byte slab of the tile
            if (KC) {
                int row = inst * 8 + (lane >> 3), pslot = lane & 7;
                int lslot = (pslot ^ kc_swz(row)) & 7;
                off[i] = (unsigned)((long)row * sF + lslot * 8);
            } else {
                constexpr int KPI = 64 / VPR;        // k-rows per instruction
                int k = inst * KPI + lane / VPR, punit = lane % VPR;
                int lunit = punit ^ mc_swz(k);
                off[i] = (unsigned)((long)k * sK + lunit * 8);
            }
        }
    }

    static __device__ __forceinline__ void issue(half_t* stage, const half_t* tile, const unsigned (&off)[NV],
                                                 int wave) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            __builtin_amdgcn_global_load_lds((global_void_ptr)(tile + off[i]),
                                             (lds_void_ptr)(stage + (wave * NV + i) * 512), 16, 0, 0);
    }

    // KC fragments from one address register per wave and operand: with
    // base = kc_off(row0 + lane % 32, lane / 32) (row0 a multiple of 32), the fragment of the
    // idx-th 32-row block below row0 at k-step ks lies at
    //   (base ^ ((2 ks ^ 4 (idx & 1)) * 8)) + idx * 32 * BK
    // (32 rows further the swizzle flips bit 2 of the slot, a k-step further the slot moves
    // by 2, and neither carries).
    static __device__ __forceinline__ h8 frag_at(const half_t* lds, int base, int idx, int ks) {
        return *reinterpret_cast<const h8*>(lds + ((base ^ (((2 * ks) ^ (4 * (idx & 1))) * 8)) + idx * 32 * BK));
    }

    static __device__ __forceinline__ h8 frag(const half_t* lds, int row0, int ks, int lane) {
        if (KC) {
            return *reinterpret_cast<const h8*>(lds + kc_off(row0 + (lane & 31), ks * 2 + (lane >> 5)));
        } else {
            const int g = lane >> 4, l = lane & 15;
            const int k = ks * 16 + 8 * (g >> 1) + (l >> 2);       // and k + 4 for the second half
            const int m = row0 + 16 * (g & 1) + 4 * (l & 3);
            // k & 3 == (k + 4) & 3 and ((k+4) >> 1) & 1 differs: recompute the swizzle per row
            const half_t* p0 = lds + k * ROWS + (((m >> 3) ^ mc_swz(k)) << 3) + (m & 7);
            const half_t* p1 = lds + (k + 4) * ROWS + (((m >> 3) ^ mc_swz(k + 4)) << 3) + (m & 7);
            typedef s4v __attribute__((address_space(3))) * lds_s4;
            s4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(p0));
            s4v hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(p1));
            typedef short s8 __attribute__((ext_vector_type(8)));
            s8 r = __builtin_shufflevector(lo, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
            return __builtin_bit_cast(h8, r);
        }
    }
};


// k_gemm_tiles.hip: products in tiles of five sizes, up to kMaxProducts in one launch.
enum { TILE_64x64 = 0, TILE_128x64, TILE_128x128, TILE_256x128, TILE_256x256, TILE_FORMS };
constexpr unsigned kRingForms = (1u << TILE_256x256) - 1;
struct TileProduct {
    GemmArgs a;                   // with splits (and, if more than one, partial) and nbatch set
    bool akc, bkc;                // operands contiguous along k
};
// Products of one launch may be read in one way, or in the two of which an instance exists.
inline bool orientations(const TileProduct* p, int n, int& k1, int& k2) {
    int seen = 0;
    for (int i = 0; i < n; ++i) seen |= 1 << ((p[i].akc ? 1 : 0) | (p[i].bkc ? 2 : 0));
    for (int k = 0; k < 4; ++k)
        if (seen == 1 << k) { k1 = k2 = k; return true; }
    k1 = seen == 9 ? 3 : 1; k2 = 0;
    return seen == 3 || seen == 9;
}
// Which workgroup takes which tiles of a launch's list (tiles of the same length next to each other, the longest in front):
// `rounds` rounds of all workgroups, tile r n + l to workgroup l, then parts of the list that go to neighbouring workgroups.
struct SchedulePart { unsigned worker, tile, count; };
constexpr int kMaxParts = 12;
struct Schedule { unsigned rounds = 0, n = 0; SchedulePart part[kMaxParts]; };
// The schedule of cnt[i] tiles of len[i] steps, i < n, for `workers` workgroups, and the steps of the one that takes longest (a tile's
// way out counted as out_steps of them).
double schedule_tiles(const long* len, const long* cnt, int n, long workers, double out_steps, Schedule& s);
struct TileChoice {
    int form = -1;                // none where the orientations do not share a launch
    double us = 0.;               // what the launch is expected to take
    int split = 0, splits = 1;    // product `split` in `splits` parts
};
bool tiles_take(const TileProduct& p);                        // within the range of the loads' offsets
// The best of `forms` (a bit each).  ws_floats > 0: the longest contraction may be split over that much scratch; reduce_us: what
// adding up the parts takes besides a pass over them.
constexpr double kReduceLaunch = 3.0;
TileChoice choose_tiles(const TileProduct* p, int n, unsigned forms, size_t ws_floats, double reduce_us = kReduceLaunch);
// `tail`: column sums of earlier launches, finished by workgroups behind the tiles (tail->n = 0 then).
// Outputs of a tile of form f, and workgroups of that form on a CU.
// out_steps: the way out of a tile in steps of it.
struct TileForm { int bm, bn, per_cu; double out_steps; };
TileForm tile_form(int form);
// The best form for a product with an activation in its epilogue (-1: none), and its launch.
int choose_act_form(const TileProduct& p);
// With same_order: whether the product is summed in the order of 256 x 256 tiles (k slices of 32; the others': 16).
bool summed_wide(const TileProduct& p);
void launch_tiles_act(const TileProduct& p, int form, hipStream_t st);
// k_gemm_wide.hip: 256 x 256 tiles.
bool wide_takes(const TileProduct& p);
// side_blocks: workgroups behind the tiles, for GemmArgs::side_*
void launch_wide(const TileProduct* p, int n, FinishJobs* tail, unsigned side_blocks, hipStream_t st);
void launch_tiles(const TileProduct* p, int n, int form, FinishJobs* tail, hipStream_t st);

}  // namespace sub
