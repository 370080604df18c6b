// et_expert_gemm_thin.hip -- the expert grouped GEMM for experts with few
// slots (gfx950): the same products, sums and epilogues as expert_gemm_kernel
// (et_expert_gemm.hip), bit for bit, tiled for reading each weight once.
//
// An expert with up to about a hundred slots does 2 * slots FLOP per weight
// element, so the time is that of streaming its weight from HBM.  A 256 x 256
// tile reads the weight through LDS with 64 KiB in flight per CU and spends
// most of its loads, LDS writes and MFMAs on repeated rows: 4.4 to 4.8 TB/s on 128
// experts of 1 to 128 slots (K = 4096, N = 3072), and 8 experts leave half the
// CUs idle.  Here a block of 4 waves owns the expert's slots (up to 128, in
// MFMA tiles by their number) x 128 weight rows (fp8: 256).  A wave loads its
// own 32 weight rows (fp8: 64) straight into MFMA fragments: lane l of a
// 16-row fragment reads 16 bytes of row l % 16, so one load covers 64
// contiguous bytes of 16 rows, which streams at 6.0-6.1 TB/s (the same rows
// through direct-to-LDS loads: 4.9 to 5.5).  A register ring holds the
// fragments of the next U k-steps: with 8 waves a CU keeps 128 KiB of weight
// in flight.  The rows of A go through LDS, 128 to 512 bytes of each at a
// time: read from L2 by every wave instead they tripled the L2 traffic at 64
// slots, which then bound the kernel (1.17 against 0.63 ms at 128 experts).
//
// Measured (us under sustained load, this kernel against 256-row tiles; the weight
// alone takes 525 and 264 at 6.1 TB/s): 128 experts, K = 4096, N = 3072, of 1 slot
// 526 against 674, of 16 570 / 679, of 64 635 / 690, of 96 697 / 704, of 128 735 /
// 728; K = 7168, N = 1536, of 1 slot 487 / 587, of 64 589 / 601; 24 experts of 16
// slots, K = 7168, N = 3072 240 / 286; 8 experts of 8 slots, K = 4096, N = 3072 39 /
// 84; fp8, 64 experts of 32 slots, K = 2048, N = 3072 with SwiGLU 103 / 124.  Which
// calls come here, and where these lose: thin_share and expert_gemm_route.
//
// Order of the sum: that of expert_gemm_kernel (k-steps of 32 ascending in
// one v_mfma_f32_16x16x32_bf16 each; fp8: 64 in one
// v_mfma_scale_f32_32x32x64_f8f6f4), so an output's bits do not depend on
// which kernel an expert's slot count selects.
#include "et_gemm_common.hpp"

namespace et {
namespace {

constexpr int kThreads = 256;

// 16 bytes per lane at byte offset voff + soff (soff uniform, inside the row
// that voff names; voff marked out of range reads 0).
__device__ __forceinline__ u32x4_t load16(__amdgpu_buffer_rsrc_t res, uint32_t voff, uint32_t soff)
{
    return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(res, (int)voff, (int)soff, 0));
}

__device__ __forceinline__ uint64_t uniform64(uint64_t v)
{
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

// One block's tile, n0 one wave's.  All wave-uniform.
struct ThinTile {
    int64_t s0;   // first slot
    int rows;     // slots
    int e;        // expert
    int n0;       // first weight row (plain) or hidden unit (SwiGLU) of the wave
};

// A chunk of the rows of A in LDS: CS k-steps of 64 bytes, rows padded so that
// 16 rows' pieces fall on distinct banks.
template <int CS>
struct ThinChunk {
    static constexpr int BYTES = 64 * CS;
    static constexpr int PITCH = BYTES + 16;
    static constexpr int SEGS = BYTES / 16;   // 16-byte segments per row
};
constexpr int kXBuf = kThinTile * ThinChunk<2>::PITCH;   // one of the two buffers

// The operand rows of A of a tile (XROWS of them): XR loads of 16 bytes per
// thread and chunk, thread t the segment t % SEGS of rows t / SEGS + (kThreads
// / SEGS) i.  Chunk c + 2 is loaded while chunk c is multiplied and chunk c + 1
// waits in registers.
template <bool GATHER, int XROWS, int CS, int ES>
struct ThinRows {
    using C = ThinChunk<CS>;
    static constexpr int STEP = kThreads / C::SEGS;   // rows per load of the block
    static constexpr int XR = XROWS / STEP;
    static constexpr int kChunk = C::BYTES;
    static_assert(XR * STEP == XROWS && XROWS * C::PITCH <= kXBuf, "whole loads, inside the buffer");
    __amdgpu_buffer_rsrc_t res;
    uint32_t off[XR];
    int klim;                 // chunks in which this thread's segment lies below K
    int clast;                // the last chunk that begins below K
    u32x4_t reg[2][XR];

    __device__ __forceinline__ void setup(const GemmArgs& g, const ThinTile& t)
    {
        const uint32_t pitch = (uint32_t)g.K * ES;
        const int seg = (int)threadIdx.x % C::SEGS, r0 = (int)threadIdx.x / C::SEGS;
        res = GATHER ? __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(g.a), (short)0,
                                                         (int)(g.a_rows * g.K * ES), kBufDword3)
                     : __builtin_amdgcn_make_buffer_rsrc((void*)uniform64((uint64_t)(uintptr_t)(g.a + t.s0 * g.K * ES)),
                                                         (short)0, t.rows * g.K * ES, kBufDword3);
        klim = (g.K * ES - 16 * seg + kChunk - 1) / kChunk;
        clast = (g.K * ES - 1) / kChunk;
        // rows past the tile repeat its last slot (their outputs are not
        // stored); invalid tokens read 0
#pragma unroll
        for (int i = 0; i < XR; ++i) {
            const int r = min(STEP * i + r0, t.rows - 1);
            if constexpr (GATHER) {
                const uint32_t tok = (uint32_t)g.sorted_token[t.s0 + r];
                off[i] = tok < (uint32_t)g.a_rows ? tok * pitch + 16u * seg : kOOR;
            } else {
                off[i] = (uint32_t)r * pitch + 16u * seg;
            }
        }
    }
    // (segments past K read 0, so the chunks that pad K to whole ring turns do)
    __device__ __forceinline__ void load(int c, int b)
    {
        const bool in = c < klim;
        const uint32_t soff = (uint32_t)min(c, clast) * kChunk;
#pragma unroll
        for (int i = 0; i < XR; ++i) reg[b][i] = load16(res, in ? off[i] : kOOR, soff);
    }
    __device__ __forceinline__ void store(unsigned char* lds, int b)
    {
#pragma unroll
        for (int i = 0; i < XR; ++i)
            *reinterpret_cast<u32x4_t*>(lds + (STEP * i + (int)threadIdx.x / C::SEGS) * C::PITCH +
                                        16 * ((int)threadIdx.x % C::SEGS)) = reg[b][i];
    }
};

// The K loop of both kernels: U k-steps of weight fragments in a register
// ring, the rows of A through two LDS buffers (one barrier per chunk).  K is
// padded to whole turns of the ring with k-steps of zeros, which leave every
// sum as it is.  load_w(ks, u) loads k-step ks into ring slot u, mma(u, x)
// multiplies ring slot u with the k-step whose A fragments start at x.
// (Letting the two streams run on from one tile of a block to the next, with
// the tiles dealt out in contiguous runs for it, gained nothing at whole
// multiples of 512 tiles and cost 5 to 25% elsewhere: two blocks per CU hide a
// tile's start already.)
template <int CS, int U, typename Rows, typename LoadW, typename Mma>
__device__ __forceinline__ void thin_loop(const GemmArgs& g, const ThinTile& t, Rows& rows, unsigned char* lds, int nks,
                                          LoadW load_w, Mma mma)
{
    // chunks per turn of the loop: ring slots and LDS buffers are constants in it
    constexpr int NB = U > 2 * CS ? U / CS : 2;
    static_assert(U % CS == 0 && NB * CS % U == 0 && NB % 2 == 0, "whole chunks per ring turn");
    const int nc = (nks + CS - 1) / CS;
    auto pin = [] { __builtin_amdgcn_sched_barrier(0); };
    // The weight first: its addresses need no slot data.  (Order kept
    // throughout: each wait of the loop then covers its oldest loads only.)
#pragma unroll
    for (int u = 0; u < U; ++u) {
        load_w(u, u);
        pin();
    }
    rows.setup(g, t);
    rows.load(0, 0);
    pin();
    rows.load(1, 1);
    pin();
    rows.store(lds, 0);
    pin();
    rows.load(2, 0);
    __syncthreads();
    for (int c = 0; c < nc; c += NB) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            // chunk c + b is in buffer b & 1; the next one goes to the other,
            // which every wave has read before the barrier that ended the last
            // chunk
            rows.store(lds + ((b & 1) ^ 1) * kXBuf, (b & 1) ^ 1);
            pin();
            rows.load(c + b + 3, (b & 1) ^ 1);
            pin();
#pragma unroll
            for (int s = 0; s < CS; ++s) {
                const int u = (CS * b + s) % U;
                mma(u, lds + (b & 1) * kXBuf + 64 * s);
                pin();
                load_w(CS * (c + b) + s + U, u);
                pin();
            }
            __syncthreads();
        }
    }
}

// bf16: MT tiles of 16 slots x NT = 2 tiles of 16 weight rows (SwiGLU: 16 gate
// rows and their 16 up rows).  Lane l holds operand row l % 16, k = 8 (l / 16)
// + 0..7 of a k-step of 32, and slot l % 16, weight rows 4 (l / 16) + 0..3 of
// an accumulator tile.
template <bool GATHER, int EPI, int MT>
__device__ __forceinline__ void thin_tile_bf16(const GemmArgs& g, const ThinTile& t, unsigned char* lds)
{
    // (16 slots or fewer: a deeper ring, for the calls with few tiles)
    constexpr int NT = 2, CS = MT == 1 ? 8 : MT > 4 ? 2 : 4, U = MT == 1 ? 16 : 8;
    constexpr int kPitch = ThinChunk<CS>::PITCH;
    const int lane = lane_id();
    const int r16 = lane & 15, rho = lane >> 4;
    const int K = g.K, N = g.N, F = N / 2;
    ThinRows<GATHER, 16 * MT, CS, 2> rows;
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)uniform64((uint64_t)(uintptr_t)(g.w + (int64_t)t.e * N * K * 2)), (short)0, N * K * 2, kBufDword3);
    uint32_t wo[NT];          // weight rows past N read 0
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n = t.n0 + (EPI == EPI_SWIGLU ? (j ? F : 0) : 16 * j) + r16;
        const bool ok = EPI == EPI_SWIGLU ? t.n0 + r16 < F : n < N;
        wo[j] = ok ? (uint32_t)n * (uint32_t)K * 2u + 16u * rho : kOOR;
    }
    float sc[MT];
    if constexpr (EPI == EPI_ROW_SCALE) {
#pragma unroll
        for (int i = 0; i < MT; ++i) sc[i] = g.row_scale[t.s0 + min(16 * i + r16, t.rows - 1)];
    }
    const int nks = (K + 31) / 32;
    const int nlim = (K - 8 * rho + 31) / 32;   // k-steps in which this lane's 8 k lie below K
    u32x4_t wf[U][NT];
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{};
    const int ncols = EPI == EPI_SWIGLU ? F : N;
    const __amdgpu_buffer_rsrc_t cres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)uniform64((uint64_t)(uintptr_t)(g.c + t.s0 * ncols)), (short)0, t.rows * ncols * 2, kBufDword3);
    thin_loop<CS, U>(
        g, t, rows, lds, nks,
        [&](int ks, int u) {
            const bool in = ks < nlim;
            const uint32_t soff = (uint32_t)min(ks, nks - 1) * 64u;
#pragma unroll
            for (int j = 0; j < NT; ++j) wf[u][j] = load16(wres, in ? wo[j] : kOOR, soff);
        },
        [&](int u, const unsigned char* x) {
            const unsigned char* xl = x + r16 * kPitch + 16 * rho;
            u32x4_t xf[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) xf[i] = *reinterpret_cast<const u32x4_t*>(xl + 16 * i * kPitch);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[u][j]),
                                                                        __builtin_bit_cast(bf16x8_t, xf[i]),
                                                                        acc[i][j], 0, 0, 0);
        });
    // epilogue, as expert_gemm_kernel's
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = 16 * i + r16;
        if constexpr (EPI == EPI_SWIGLU) {
            const int col = t.n0 + 4 * rho;
            float h[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float gv = acc[i][0][e];
                h[e] = (gv * sigmoid(gv)) * acc[i][1][e];
            }
            const u32x2_t out = {pack_bf16x2(h[0], h[1]), pack_bf16x2(h[2], h[3])};
            const uint32_t off =
                (row < t.rows && col < F) ? ((uint32_t)row * (uint32_t)F + (uint32_t)col) * 2u : kOOR;
            __builtin_amdgcn_raw_buffer_store_b64(out, cres, off, 0, 0);
        } else {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float a = acc[i][e >> 2][e & 3];
                v[e] = EPI == EPI_ROW_SCALE ? sc[i] * a : a;
            }
            store_pair16(v, cres, row < t.rows, (uint32_t)row * (uint32_t)N, t.n0, N, rho);
        }
    }
}

// fp8: MT tiles of 32 slots x 2 tiles of 32 weight rows (SwiGLU: 32 gate rows
// and their 32 up rows).  Lane l holds operand row l % 32; of a k-step's 64
// bytes it takes the 16-byte pieces 16 (l / 32) and 32 + 16 (l / 32) (the
// MFMA's sum does not depend on how k is dealt to the lanes as long as both
// operands agree), so one load covers 32 contiguous bytes of 32 rows.
template <bool GATHER, int EPI, int MT>
__device__ __forceinline__ void thin_tile_fp8(const GemmArgs& g, const ThinTile& t, unsigned char* lds)
{
    constexpr int NT = 2, CS = MT > 2 ? 2 : 4, U = 4;
    constexpr int kPitch = ThinChunk<CS>::PITCH;
    const int lane = lane_id();
    const int r32 = lane & 31, kh = lane >> 5;
    const int K = g.K, N = g.N, F = N / 2;
    ThinRows<GATHER, 32 * MT, CS, 1> rows;
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)uniform64((uint64_t)(uintptr_t)(g.w + (int64_t)t.e * N * K)), (short)0, N * K, kBufDword3);
    uint32_t wo[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n = t.n0 + (EPI == EPI_SWIGLU ? (j ? F : 0) : 32 * j) + r32;
        const bool ok = EPI == EPI_SWIGLU ? t.n0 + r32 < F : n < N;
        wo[j] = ok ? (uint32_t)n * (uint32_t)K + 16u * kh : kOOR;
    }
    const int nks = (K + 63) / 64;
    // k-steps in which the lane's first and second piece lie below K (a
    // multiple of 16)
    const int nlim0 = (K - 16 * kh + 63) / 64;
    const int nlim1 = (K - 16 * kh + 31) / 64;
    u32x8_t wf[U][NT];
    f32x16_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16_t{};
    auto pair = [](u32x4_t a, u32x4_t b) { return u32x8_t{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}; };
    const int ncols = EPI == EPI_SWIGLU ? F : N;
    const float* ws = g.w_scale + (int64_t)t.e * N;
    const __amdgpu_buffer_rsrc_t cres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)uniform64((uint64_t)(uintptr_t)(g.c + t.s0 * ncols)), (short)0, t.rows * ncols * 2, kBufDword3);
    thin_loop<CS, U>(
        g, t, rows, lds, nks,
        [&](int ks, int u) {
            const bool in0 = ks < nlim0, in1 = ks < nlim1;
            const uint32_t soff = (uint32_t)min(ks, nks - 1) * 64u;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const uint32_t o = wo[j];
                wf[u][j] = pair(load16(wres, in0 ? o : kOOR, soff), load16(wres, in1 ? o : kOOR, soff + 32u));
            }
        },
        [&](int u, const unsigned char* x) {
            const unsigned char* xl = x + r32 * kPitch + 16 * kh;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const u32x4_t x0 = *reinterpret_cast<const u32x4_t*>(xl + 32 * i * kPitch);
                const u32x4_t x1 = *reinterpret_cast<const u32x4_t*>(xl + 32 * i * kPitch + 32);
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                        __builtin_bit_cast(i32x8_t, wf[u][j]), __builtin_bit_cast(i32x8_t, pair(x0, x1)), acc[i][j], 0,
                        0, 0, 127, 0, 127);
            }
        });
    // the scales of the lane's slots (0 for an invalid token)
    float sa[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int64_t s = t.s0 + min(32 * i + r32, t.rows - 1);
        if constexpr (GATHER) {
            const uint32_t tok = (uint32_t)g.sorted_token[s];
            sa[i] = tok < (uint32_t)g.a_rows ? g.a_scale[tok] : 0.0f;
        } else {
            sa[i] = g.a_scale[s];
        }
    }
#pragma unroll
    for (int j = 0; j < (EPI == EPI_SWIGLU ? 1 : NT); ++j) {
        u32x2_t P[MT][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // scales of 4 of the lane's weight rows (and their up
            // rows): few at a time, beside the ring's registers
            __builtin_amdgcn_sched_barrier(0);
            float w0[4], w1[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = min(t.n0 + 32 * j + 8 * r + 4 * kh + e, ncols - 1);
                w0[e] = ws[n];
                w1[e] = EPI == EPI_SWIGLU ? ws[F + n] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = (acc[i][j][4 * r + e] * sa[i]) * w0[e];
                    if constexpr (EPI == EPI_SWIGLU) {
                        const float uv = (acc[i][1][4 * r + e] * sa[i]) * w1[e];
                        v[e] = (v[e] * sigmoid(v[e])) * uv;
                    }
                }
                P[i][r] = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const int row = 32 * i + r32;
            store_row_segment(P[i], cres, row < t.rows, (uint32_t)row * (uint32_t)ncols, t.n0 + 32 * j, ncols, kh);
        }
    }
}

// The experts that expert_gemm_split gives to this kernel; each block walks
// tiles of 4 waves side by side in the weight rows.  XCD x (blocks b % 8 = x)
// takes a contiguous range of tiles; within an expert the slot tiles are
// innermost, so they read a weight row through the same L2.
template <bool GATHER, int EPI, bool FP8>
__global__ __launch_bounds__(kThreads, 2) void expert_gemm_thin_kernel(GemmArgs g, int64_t thin_rows, int cus)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * kXBuf];
    __shared__ int ptile[ET_MAX_EXPERTS + 1];     // prefix of the experts' slot tiles
    __shared__ int32_t eoff[ET_MAX_EXPERTS + 1];  // expert_offsets below the capacity
    __shared__ int tile_rows;                     // slots per tile
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int E = g.E;
    if (wave == 0) {
        const ThinSplit sp = expert_gemm_split<GATHER, EPI, FP8>(g, thin_rows, cus);
        int carry = 0;
        for (int e0 = 0; e0 < E; e0 += kWave) {
            const int e = e0 + lane;
            int n = 0;
            if (e < E) {
                const int64_t lo = min<int64_t>(g.expert_offsets[e], g.cap);
                const int64_t hi = min<int64_t>(g.expert_offsets[e + 1], g.cap);
                eoff[e] = (int32_t)lo;
                eoff[e + 1] = (int32_t)hi;   // (the next expert's lo)
                const int64_t rows = max<int64_t>(0, hi - lo);
                n = rows <= sp.rows ? (int)((rows + sp.tile - 1) / sp.tile) : 0;
            }
            const int inc = wave_incl_scan(n) + carry;
            if (e < E) ptile[e + 1] = inc;
            carry = __shfl(inc, kWave - 1, kWave);
        }
        if (lane == 0) {
            ptile[0] = 0;
            tile_rows = sp.tile;
        }
    }
    __syncthreads();
    constexpr int cols = kThinBlockCols<EPI, FP8>;
    const int width = EPI == EPI_SWIGLU ? g.N / 2 : g.N;
    const int nN = (width + cols - 1) / cols;
    const int Q = __builtin_amdgcn_readfirstlane(ptile[E]) * nN;
    const int tm = __builtin_amdgcn_readfirstlane(tile_rows);
    const int per = (Q + 7) / 8;
    const int nloc = (int)(gridDim.x >> 3);
    for (int l = (int)(blockIdx.x >> 3); l < per; l += nloc) {
        const int q = (int)(blockIdx.x & 7) * per + l;
        if (q >= Q) break;
        int lo = 0, hi = E;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (ptile[mid] <= q / nN) lo = mid;
            else hi = mid;
        }
        ThinTile t;
        t.e = __builtin_amdgcn_readfirstlane(lo);
        const int p0 = __builtin_amdgcn_readfirstlane(ptile[t.e]);
        const int mte = __builtin_amdgcn_readfirstlane(ptile[t.e + 1]) - p0;
        const int qq = q - p0 * nN;
        const int first = __builtin_amdgcn_readfirstlane(eoff[t.e]);
        const int end = __builtin_amdgcn_readfirstlane(eoff[t.e + 1]);
        t.s0 = first + (qq % mte) * tm;
        t.rows = min(tm, end - (int)t.s0);
        t.n0 = (qq / mte) * cols + wave * (cols / 4);
        // (waves past the weight's rows take part in the barriers)
        if constexpr (FP8) {
            if (t.rows <= 32) thin_tile_fp8<GATHER, EPI, 1>(g, t, lds);
            else if (t.rows <= 64) thin_tile_fp8<GATHER, EPI, 2>(g, t, lds);
            else if (t.rows <= 96) thin_tile_fp8<GATHER, EPI, 3>(g, t, lds);
            else thin_tile_fp8<GATHER, EPI, 4>(g, t, lds);
        } else {
            if (t.rows <= 16) thin_tile_bf16<GATHER, EPI, 1>(g, t, lds);
            else if (t.rows <= 32) thin_tile_bf16<GATHER, EPI, 2>(g, t, lds);
            else if (t.rows <= 64) thin_tile_bf16<GATHER, EPI, 4>(g, t, lds);
            else if (t.rows <= 96) thin_tile_bf16<GATHER, EPI, 6>(g, t, lds);
            else thin_tile_bf16<GATHER, EPI, 8>(g, t, lds);
        }
    }
}

}  // namespace

int launch_expert_gemm_thin(bool fp8, bool gather, int epilogue, const GemmArgs& args, int64_t thin_rows, int cus,
                            hipStream_t s)
{
    // slot tiles at most: one for each expert and each 64 slots (the half height)
    const int cols = (fp8 ? 256 : 128) / (epilogue == EPI_SWIGLU ? 2 : 1);
    const int64_t width = epilogue == EPI_SWIGLU ? args.N / 2 : args.N;
    const int64_t qmax = std::min<int64_t>(args.cap, args.cap / (kThinTile / 2) + args.E) * ((width + cols - 1) / cols);
    const int64_t blocks = std::min<int64_t>(2 * (int64_t)cus, qmax);
    const dim3 grid((unsigned)(8 * ((blocks + 7) / 8))), block(kThreads);
    if (fp8) {
        switch ((epilogue == EPI_SWIGLU ? 2 : 0) + (gather ? 1 : 0)) {
            case 0: expert_gemm_thin_kernel<false, EPI_PLAIN, true><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            case 1: expert_gemm_thin_kernel<true, EPI_PLAIN, true><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            case 2: expert_gemm_thin_kernel<false, EPI_SWIGLU, true><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            default: expert_gemm_thin_kernel<true, EPI_SWIGLU, true><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
        }
    } else {
        switch (epilogue * 2 + (gather ? 1 : 0)) {
            case 0: expert_gemm_thin_kernel<false, EPI_PLAIN, false><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            case 1: expert_gemm_thin_kernel<true, EPI_PLAIN, false><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            case 2: expert_gemm_thin_kernel<false, EPI_ROW_SCALE, false><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            case 3: expert_gemm_thin_kernel<true, EPI_ROW_SCALE, false><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            case 4: expert_gemm_thin_kernel<false, EPI_SWIGLU, false><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
            default: expert_gemm_thin_kernel<true, EPI_SWIGLU, false><<<grid, block, 0, s>>>(args, thin_rows, cus); break;
        }
    }
    return check_launch("expert_gemm_thin_kernel");
}

}  // namespace et
