// et_gemm_common.hpp -- what the expert grouped GEMM kernels share: operand
// types, arguments, epilogue kinds and the range-checked output stores.
#pragma once

#include <algorithm>

#include "et_common.hpp"

namespace et {

struct GemmArgs {
    const unsigned char* a;         // gather: X [a_rows, K]; else A [cap, K] (bf16, or fp8 e4m3)
    const int32_t* sorted_token;    // [cap] (gather only)
    const unsigned char* w;         // [E, N, K] (bf16, or fp8 e4m3)
    const int32_t* expert_offsets;  // [E + 1]
    uint16_t* c;                    // [cap, N] bf16
    const float* row_scale;         // [cap] (EPI_ROW_SCALE only)
    const float* a_scale;           // fp8: [a_rows], the scale of each row of a
    const float* w_scale;           // fp8: [E, N], the scale of each weight row
    int64_t a_rows;
    int64_t cap;
    int K, N, E;                    // N: rows of each expert's weight (2 F for SwiGLU)
};

// The thin kernel (et_expert_gemm_thin.hip) on its experts (ThinSplit, thin_rows
// = -1 to decide on the device).
int launch_expert_gemm_thin(bool fp8, bool gather, int epilogue, const GemmArgs& args, int64_t thin_rows, int cus,
                            hipStream_t s);

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_t;

// Word 3 of a gfx9 buffer descriptor for raw (untyped, stride 0) access.
constexpr int kBufDword3 = 0x00020000;
// A byte offset past every descriptor's num_records (all < 2^31): loads return
// 0 and stores are dropped.
constexpr uint32_t kOOR = 0x80000000u;

// Epilogues: the plain product; the product times a per-slot factor; or SwiGLU,
// h = silu(g) * u of the gate rows g (weight rows 0..F-1) and the up rows u
// (rows F..2F-1) of the same hidden unit.
constexpr int EPI_PLAIN = ET_GEMM_PLAIN;
constexpr int EPI_ROW_SCALE = ET_GEMM_ROW_SCALE;
constexpr int EPI_SWIGLU = ET_GEMM_SWIGLU;

// Tiles of expert_gemm_kernel: 256 slots x 256 weight rows (SwiGLU: 128 hidden
// units), one block per CU.
constexpr int kBM = 256;
constexpr int kBN = 256;
// Tiles of expert_gemm_thin_kernel: up to 128 slots x 128 weight rows (fp8:
// 256; SwiGLU: half as many hidden units), two blocks per CU.
constexpr int kThinTile = 128;
template <int EPI, bool FP8>
constexpr int kThinBlockCols = (FP8 ? 256 : 128) / (EPI == EPI_SWIGLU ? 2 : 1);

// Which experts the thin kernel takes, and in tiles of how many slots.
struct ThinSplit {
    int64_t rows;   // those with at most this many slots (0: none, INT64_MAX: all)
    int tile;       // kThinTile, or half of it
};
// Both kernels evaluate this on the device, where the slot counts are, with
// one whole wave; given >= 0 is the host's answer for rows.
//
// The costs compared are in 1/50 of the time of a 256-row tile and in rounds
// of one tile per CU, as either kernel's time goes (a second thin tile on a CU
// shares its LDS and matrix pipes).  Measured per round: bf16 (128 experts, K =
// 4096, N = 3072) 125 us a 256-row tile, and a thin tile 49 us up to 32 slots, 53
// up to 64, 58 up to 96 and 62 up to 128, with a larger share for its start and
// end where K is shorter (64 experts of about 64 slots, K = 1536, N = 2048: 46 and
// 26); fp8 (64 experts, K = 2048, N = 3072) 47, and 35, 37 and 39.  Calls either side of the line, thin against 256-row tiles:
// 128 experts of 96 slots 695 against 750 us, of 128 slots 739 against 755, of
// 256 slots 1242 against 791; 8 experts (N = 1536) of 250 slots 57 against 81;
// 24 experts of 128 slots (288 tiles, two rounds) 112 against 91.  Where every
// tile of 64 slots has a CU of its own these are faster than half as many of
// 128 (8 experts of 128 slots 38 against 54 us; of 250 slots, with more tiles
// than CUs, 70 against 57).
template <int EPI, bool FP8>
__device__ __forceinline__ ThinSplit expert_gemm_split(const GemmArgs& g, int64_t given, int cus)
{
    constexpr int kBig = 50, kHalfTile = kThinTile / 2;
    constexpr int bn = EPI == EPI_SWIGLU ? kBN / 2 : kBN, tn = kThinBlockCols<EPI, FP8>;
    const int width = EPI == EPI_SWIGLU ? g.N / 2 : g.N;
    const int64_t nb = (width + bn - 1) / bn, nt = (width + tn - 1) / tn;
    const int fixed = FP8 ? 0 : min(4, 6144 / g.K);
    auto cost = [fixed](int n) -> int {   // of a tile of n slots
        if (n <= 0) return 0;
        return FP8 ? (n <= 64 ? 37 : n <= 96 ? 39 : 42) : fixed + (n <= 32 ? 19 : n <= 64 ? 21 : n <= 96 ? 23 : 25);
    };
    // slot tiles: thin ones and their cost, thin ones at half the height, 256-row
    // ones; and of the experts of one thin tile alone
    int thin = 0, thin_cost = 0, half = 0, big = 0, few = 0, few_cost = 0;
    for (int e = lane_id(); e < g.E; e += kWave) {
        const int64_t lo = min<int64_t>(g.expert_offsets[e], g.cap);
        const int64_t hi = min<int64_t>(g.expert_offsets[e + 1], g.cap);
        const int n = (int)max<int64_t>(0, hi - lo);
        const int c = n / kThinTile * cost(kThinTile) + cost(n % kThinTile);
        thin += (n + kThinTile - 1) / kThinTile;
        thin_cost += c;
        half += (n + kHalfTile - 1) / kHalfTile;
        big += (n + kBM - 1) / kBM;
        few += n > 0 && n <= kThinTile ? 1 : 0;
        few_cost += n <= kThinTile ? c : 0;
    }
    thin = wave_sum_int(thin);
    thin_cost = wave_sum_int(thin_cost);
    half = wave_sum_int(half);
    big = wave_sum_int(big);
    few = wave_sum_int(few);
    few_cost = wave_sum_int(few_cost);
    ThinSplit r{given, half * nt <= cus ? kHalfTile : kThinTile};
    if (given >= 0) return r;
    auto rounds = [&](int64_t tiles) { return (tiles + cus - 1) / cus; };
    const int64_t all_thin = rounds(thin * nt) * thin_cost / max(thin, 1);
    const int64_t all_big = rounds(big * nb) * kBig;
    const int64_t both = rounds(few * nt) * few_cost / max(few, 1) + rounds((big - few) * nb) * kBig;
    r.rows = all_big <= all_thin && all_big <= both ? 0 : all_thin <= both ? INT64_MAX : kThinTile;
    if (r.rows == kThinTile) r.tile = kThinTile;
    return r;
}

// Output of one 32 x 32 accumulator tile row segment: lane l (kh = l / 32)
// holds features 8 r + 4 kh + 0..3 of its slot in P[r] (two bf16x2 words),
// r = 0..3.  v_permlane32_swap exchanges lanes 32..63 of its first operand
// with lanes 0..31 of its second (lane layout checked on the device): swapping
// P[2p] with P[2p + 1] leaves lane l with features 16 p + 8 kh + 0..7, which it
// stores as one 16-byte write at that column (range-checked offset).
__device__ __forceinline__ void store_row_segment(u32x2_t (&P)[4], __amdgpu_buffer_rsrc_t res, bool row_ok,
                                                  uint32_t row_base, int col0, int ncols, int kh)
{
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        u32x2_t& a = P[2 * p];
        u32x2_t& b = P[2 * p + 1];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const auto r = __builtin_amdgcn_permlane32_swap(a[w], b[w], false, false);
            a[w] = r[0];
            b[w] = r[1];
        }
        const int col = col0 + 16 * p + 8 * kh;
        const u32x4_t v = {a[0], a[1], b[0], b[1]};
        const uint32_t off = (row_ok && col < ncols) ? (row_base + (uint32_t)col) * 2u : kOOR;
        __builtin_amdgcn_raw_buffer_store_b128(v, res, off, 0, 0);
    }
}

// Output of two 16 x 16 accumulator tiles side by side (output columns col0
// ... col0 + 31 of one slot): lane l (16-lane row rho = l / 16) holds columns
// 4 rho + 0..3 of the first tile in v[0..3] and of the second in v[4..7].
// v_permlane16_swap exchanges the odd 16-lane rows of its first operand with
// the even rows of its second (lane layout checked on the device), after
// which lane l holds columns 16 (rho & 1) + 8 (rho >> 1) + 0..7, stored as one
// 16-byte write (range-checked offset; ncols is a multiple of 8).
__device__ __forceinline__ void store_pair16(const float (&v)[8], __amdgpu_buffer_rsrc_t res, bool row_ok,
                                             uint32_t row_base, int col0, int ncols, int rho)
{
    const auto lo = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[4], v[5]), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[2], v[3]), pack_bf16x2(v[6], v[7]), false, false);
    const u32x4_t out = {lo[0], hi[0], lo[1], hi[1]};
    const int col = col0 + 16 * (rho & 1) + 8 * (rho >> 1);
    const uint32_t off = (row_ok && col < ncols) ? (row_base + (uint32_t)col) * 2u : kOOR;
    __builtin_amdgcn_raw_buffer_store_b128(out, res, off, 0, 0);
}

}  // namespace
}  // namespace et
