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

// What a call's tiles take, in 1/1000 of the time of one round (a tile per CU)
// of 256-row tiles of the same call.  Measured over E = 8 to 128, 1 to 400 slots
// per expert, K = 512 to 7168, N = 512 to 4096, in bursts and under sustained
// load, plain and SwiGLU, each kernel on the whole call:
//
// bf16.  One round of thin tiles always wins: 0.45 to 0.55 of a round of 256-row
// tiles up to 64 slots, 0.63 at 128 (0.9 where the weights' HBM stream binds).
// Over many rounds a pair of thin rounds (the same weights as one of the others)
// takes 0.83 to 0.89 of it up to 32 slots, 0.92 to 0.98 up to 64, 1.0 to 1.05 up to
// 96, 1.01 to 1.08 up to 128: the line lies between 64 and 96, and above 128 slots
// thin tiles lose by 20 to 100%.  Just above one round (288 tiles) the last
// tiles run alone: K = 1024 and 2048 0.93 to 1.0 up to 64 slots, K = 4096 1.02 to
// 1.26, K = 7168 1.08 to 1.31.
// fp8.  Both kernels have 256 weight rows to a tile; a thin wave's load covers
// only 32 contiguous bytes of a row, 3.3 TB/s of HBM against the 256-row tiles' 3.6
// to 4.5.  So thin tiles win by their shorter start and end alone: K = 512 0.75 to
// 0.95, K = 1024 0.81 to 1.02 up to 64 slots, K = 2048 0.9 to 1.0 where each has a CU
// and 1.05 to 1.16 over many rounds, K = 4096 1.1 to 1.2, K = 7168 1.2 to 1.4 (gathered
// rows slow the others by a tenth up to K = 1024).  With SwiGLU, whose epilogue is
// dearer on 256 rows (9 us), 0.4 to 0.85 up to K = 2048, 0.9 to 1.0 at 4096, 1.1 to
// 1.2 at 7168.
struct TileCall {
    int K, cus;
    bool fp8, swiglu, gather;
};

// Share of a thin tile of n slots where the call has `tiles` of them.
__host__ __device__ inline int thin_share(const TileCall& c, int n, int tiles)
{
    const int band = n <= 32 ? 0 : n <= 64 ? 1 : n <= 96 ? 2 : 3;
    const auto of = [band](int a, int b, int c, int d) { return band == 0 ? a : band == 1 ? b : band == 2 ? c : d; };
    if (n <= 0) return 0;
    if (c.fp8) {
        const bool light = 4 * tiles <= 3 * c.cus;   // a CU to each tile, and some to spare
        if (c.swiglu) {
            if (c.K <= 1024) return of(620, 680, 720, 800);
            if (c.K <= 2048) return light ? of(700, 760, 800, 880) : of(820, 850, 870, 920);
            if (c.K <= 4096) return light ? of(780, 840, 880, 950) : of(930, 950, 970, 1030);
            return 1150;
        }
        int share = 1150;
        if (c.K <= 512) share = light ? of(820, 880, 900, 980) : of(750, 830, 920, 1020);
        else if (c.K <= 1024) share = light ? of(850, 900, 930, 1000) : of(900, 980, 1080, 1180);
        else if (c.K <= 2048) share = light ? of(900, 950, 980, 1030) : of(1020, 1060, 1100, 1150);
        else if (c.K <= 4096 && light) share = of(950, 1000, 1000, 1030);
        return c.gather && (c.K <= 1024 || (light && c.K <= 2048)) ? share * 9 / 10 : share;
    }
    int share = of(445, c.K > 4096 ? 510 : 480, 515, 535);
    if (c.swiglu) share -= share * 150 / (c.K + 150);   // (the 256-row epilogue)
    if (c.K > 2048 && tiles > c.cus && tiles <= 3 * c.cus) share += n <= (c.K <= 5120 ? 32 : 16) ? 60 : c.K <= 5120 ? 100 : 130;
    return share;
}

// So few thin tiles that they win whatever the slots: one round (bf16, and fp8
// with SwiGLU up to K = 4096: 0.75 to 1.0); fp8 half a round up to K = 4096 (0.92 to
// 1.0), with SwiGLU above that three eighths (0.85 to 0.95), half if gathered.
__host__ __device__ inline bool thin_few(const TileCall& c, int64_t tiles)
{
    if (!c.fp8) return tiles <= c.cus;
    if (c.K <= 4096) return (c.swiglu ? 1 : 2) * tiles <= c.cus;
    return c.swiglu && 8 * tiles <= (c.gather ? 4 : 3) * c.cus;
}

// `tiles` thin tiles of this mean share.
__host__ __device__ inline int thin_time(const TileCall& c, int tiles, int share)
{
    return (tiles + c.cus - 1) / c.cus * (thin_few(c, tiles) && share > 950 ? 950 : share);
}

// `tiles` 256-row tiles in a call of `thin` thin ones.  (From K = 4096 on a full
// round of bf16 weights is bound by HBM: 1.3 times a partial one's time, of which the
// thin kernel pays some too above 5120.)
__host__ __device__ inline int big_time(const TileCall& c, int tiles, int thin)
{
    const int t = (tiles + c.cus - 1) / c.cus * 1000;
    if (c.fp8 || c.K <= 2048 || thin > 3 * c.cus) return t;
    const int hbm = (c.K <= 5120 ? 1300 : 1100) * tiles / c.cus;
    return t > hbm ? t : hbm;
}

// Which experts the thin kernel takes, and in tiles of how many slots.
struct ThinSplit {
    int64_t rows;   // those with at most this many slots (0: none, INT64_MAX: all)
    int tile;       // kThinTile, or half of it
};
// Both kernels evaluate this on the device, where the slot counts are, with
// one whole wave; given >= 0 is the host's answer for rows (expert_gemm_route).
// Where every tile of 64 slots has a CU of its own these are faster than half
// as many of 128 (8 experts of 128 slots 38 against 54 us; of 250 slots, with more
// tiles than CUs, 70 against 57).
template <bool GATHER, int EPI, bool FP8>
__device__ __forceinline__ ThinSplit expert_gemm_split(const GemmArgs& g, int64_t given, int cus)
{
    constexpr int kHalfTile = kThinTile / 2;
    constexpr bool swiglu = EPI == EPI_SWIGLU;
    constexpr int bn = swiglu ? kBN / 2 : kBN, tn = kThinBlockCols<EPI, FP8>;
    const int width = swiglu ? g.N / 2 : g.N;
    const int nb = (width + bn - 1) / bn, nt = (width + tn - 1) / tn;
    const auto slots = [&](int e) -> int {
        const int64_t lo = min<int64_t>(g.expert_offsets[e], g.cap);
        const int64_t hi = min<int64_t>(g.expert_offsets[e + 1], g.cap);
        return (int)max<int64_t>(0, hi - lo);
    };
    // slot tiles: thin ones, thin ones at half the height, 256-row ones; experts of
    // one thin tile
    int thin = 0, half = 0, big = 0, few = 0;
    for (int e = lane_id(); e < g.E; e += kWave) {
        const int n = slots(e);
        thin += (n + kThinTile - 1) / kThinTile;
        half += (n + kHalfTile - 1) / kHalfTile;
        big += (n + kBM - 1) / kBM;
        few += n > 0 && n <= kThinTile ? 1 : 0;
    }
    half = wave_sum_int(half);
    ThinSplit r{given, (int64_t)half * nt <= cus ? kHalfTile : kThinTile};
    if (__builtin_expect(given >= 0, 1)) return r;
    thin = wave_sum_int(thin);
    big = wave_sum_int(big);
    few = wave_sum_int(few);
    // (the host sends calls of up to 512 slots per expert here: 32 bits hold these)
    const TileCall c{g.K, cus, FP8, swiglu, GATHER};
    int thin_shares = 0, few_shares = 0;
    for (int e = lane_id(); e < g.E; e += kWave) {
        const int n = slots(e);
        if (n >= kThinTile) thin_shares += n / kThinTile * thin_share(c, kThinTile, thin * nt);
        thin_shares += thin_share(c, n % kThinTile, thin * nt);
        if (n <= kThinTile) few_shares += thin_share(c, n, few * nt);
    }
    thin_shares = wave_sum_int(thin_shares);
    few_shares = wave_sum_int(few_shares);
    const int all_thin = thin_time(c, thin * nt, thin_shares / max(thin, 1));
    const int all_big = big_time(c, big * nb, thin * nt);
    const int both = thin_time(c, few * nt, few_shares / max(few, 1)) + ((big - few) * nb + cus - 1) / cus * 1000;
    r.rows = 20 * (int64_t)all_thin <= 19 * (int64_t)all_big && all_thin <= both ? INT64_MAX
             : 100 * (int64_t)all_big <= 103 * (int64_t)both                     ? 0
                                                                                 : kThinTile;
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
