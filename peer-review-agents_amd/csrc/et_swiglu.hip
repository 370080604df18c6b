// et_swiglu.hip -- the SwiGLU activation of the expert FFN and its backward,
// element-wise over the routed slots (gfx950):
//
//   forward   h[s, j]  = (g * sigmoid(g)) * u,                 g = gu[s, j], u = gu[s, F + j]
//   backward  dgu[s, j]     = (dh * u) * (sigmoid(g) * (1 + g * (1 - sigmoid(g))))
//             dgu[s, F + j] = dh * (g * sigmoid(g)),           dh = dh[s, j]
//
// for s below min(expert_offsets[E], slot_capacity), j < F; bf16 in and out,
// binary32 arithmetic, every operation separately rounded in the order written
// (no contraction), the sigmoid the routing uses.  gu is the gate/up
// projection's output [cap, 2F] (gate rows of the weight first), as the plain
// expert GEMM writes it: a training forward keeps it for the backward, where
// the GEMM's fused SwiGLU epilogue (the inference form) writes h alone.
//
// Both kernels stream HBM once: 6F bytes per slot forward, 10F backward.  A
// thread takes 8 hidden units of one slot (16-byte loads of g, u and dh) and
// the slot count is read on the device, so the launch does not depend on the
// routing (no host synchronisation).  HBM bounds them: with a block for every
// 256 vectors they reach 5.9 TB/s at 524288 slots of F = 1536 (0.83 and 1.36 ms
// forward and backward; 0.97 and 1.52 with 128 looping blocks per CU, 1.09 and
// 1.72 with 16, whose waves drift apart and widen the range in flight).  The
// launch, though, only knows how many slots there can be: see swiglu_blocks.
#include <algorithm>

#include "et_common.hpp"

namespace et {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
// Blocks per CU: at least where there are vectors for them, and at most.
constexpr int64_t kMinBlocksPerCu = 16;
constexpr int64_t kMaxBlocksPerCu = 2048;

// A block for every 256 vectors of the slots that the caller knows to be there
// (all of them after a read-back, else the batch's tokens, each of which has a
// slot; 0 if nothing is known), the rest of the capacity by looping.  A block
// that finds no slot costs 0.4 ns: a capacity of T * E slots, many times the
// routed ones, took 200 us instead of 59 forward with a block for each of its
// vectors (T = 4096, E = 128, 32768 slots of F = 1536), and takes 53 with 16 per
// CU; 8192 slots of 524288 168 instead of 17, and 15.
int64_t swiglu_blocks(int64_t F, int64_t slot_capacity, int64_t known_slots, int64_t cus)
{
    const auto blocks = [&](int64_t slots) { return (slots * (F / 8) + kThreads - 1) / kThreads; };
    const int64_t known = std::min(blocks(std::clamp<int64_t>(known_slots, 0, slot_capacity)), cus * kMaxBlocksPerCu);
    return std::min(blocks(slot_capacity), std::max(known, cus * kMinBlocksPerCu));
}

__device__ __forceinline__ float silu_grad_factor(float g, float s)
{
    // d/dg (g * sigmoid(g)) = sigmoid(g) * (1 + g * (1 - sigmoid(g)))
    const float t = 1.0f - s;
    const float q = g * t;
    const float r = 1.0f + q;
    return s * r;
}

template <bool BWD>
__global__ __launch_bounds__(kThreads) void swiglu_kernel(const uint16_t* __restrict__ gu,
                                                           const uint16_t* __restrict__ dh,
                                                           uint16_t* __restrict__ out,
                                                           const int32_t* __restrict__ expert_offsets, int E,
                                                           int64_t cap, int F)
{
    const int64_t n = min<int64_t>(max<int64_t>(expert_offsets[E], 0), cap);
    const int vpr = F >> 3;                              // 8-unit vectors per slot
    // flat index idx = s * vpr + v, advanced by the grid's thread count: the
    // (s, v) pair is stepped without a division per element, and started with
    // a block-uniform one and a 32-bit one
    const int64_t stride = (int64_t)gridDim.x * kThreads;
    const int64_t first = (int64_t)blockIdx.x * kThreads;
    const int64_t ds = stride / vpr;
    const int dv = (int)(stride - ds * vpr);
    const int64_t s0 = first / vpr;
    const uint32_t v0 = (uint32_t)(first - s0 * vpr) + threadIdx.x;
    int64_t s = s0 + v0 / (uint32_t)vpr;
    int v = (int)(v0 % (uint32_t)vpr);
    for (; s < n; s += ds, v += dv, s += v >= vpr ? 1 : 0, v -= v >= vpr ? vpr : 0) {
        const int j = v * 8;
        const uint16_t* grow = gu + s * (2 * (int64_t)F);
        const u32x4_t gv = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(grow + j));
        const u32x4_t uv = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(grow + F + j));
        if constexpr (!BWD) {
            u32x4_t hv;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const float g0 = bf16lo(gv[w]), g1 = bf16hi(gv[w]);
                const float h0 = (g0 * sigmoid(g0)) * bf16lo(uv[w]);
                const float h1 = (g1 * sigmoid(g1)) * bf16hi(uv[w]);
                hv[w] = pack_bf16x2(h0, h1);
            }
            __builtin_nontemporal_store(hv, reinterpret_cast<u32x4_t*>(out + s * (int64_t)F + j));
        } else {
            const u32x4_t dv = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(dh + s * (int64_t)F + j));
            u32x4_t dg, du;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float r[2][2];
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const float g = p ? bf16hi(gv[w]) : bf16lo(gv[w]);
                    const float u = p ? bf16hi(uv[w]) : bf16lo(uv[w]);
                    const float d = p ? bf16hi(dv[w]) : bf16lo(dv[w]);
                    const float sg = sigmoid(g);
                    r[0][p] = (d * u) * silu_grad_factor(g, sg);
                    r[1][p] = d * (g * sg);
                }
                dg[w] = pack_bf16x2(r[0][0], r[0][1]);
                du[w] = pack_bf16x2(r[1][0], r[1][1]);
            }
            uint16_t* orow = out + s * (2 * (int64_t)F);
            __builtin_nontemporal_store(dg, reinterpret_cast<u32x4_t*>(orow + j));
            __builtin_nontemporal_store(du, reinterpret_cast<u32x4_t*>(orow + F + j));
        }
    }
}

int launch_swiglu(const char* fn, bool bwd, const void* gu, const void* dh, int64_t F,
                  const int32_t* expert_offsets, int64_t E, int64_t slot_capacity, int64_t known_slots, void* out,
                  void* stream)
{
    if (E < 1 || E > ET_MAX_EXPERTS)
        return fail(ET_ERR_INVALID_ARGUMENT, std::string(fn) + ": num_experts must be in [1, " +
                                                 std::to_string(ET_MAX_EXPERTS) + "]");
    if (F < 8 || F % 8 != 0 || F >= (int64_t(1) << 28))
        return fail(ET_ERR_INVALID_ARGUMENT, std::string(fn) + ": F must be a positive multiple of 8 below 2^28");
    if (slot_capacity < 0 || slot_capacity >= (int64_t(1) << 31))
        return fail(ET_ERR_INVALID_ARGUMENT, std::string(fn) + ": slot_capacity out of range");
    if (slot_capacity == 0) return ET_OK;
    if (!gu || !expert_offsets || !out || (bwd && !dh))
        return fail(ET_ERR_INVALID_ARGUMENT, std::string(fn) + ": null pointer");
    if ((reinterpret_cast<uintptr_t>(gu) & 15) || (reinterpret_cast<uintptr_t>(out) & 15) ||
        (reinterpret_cast<uintptr_t>(dh) & 15))
        return fail(ET_ERR_INVALID_ARGUMENT, std::string(fn) + ": gu, dh and the output must be 16-byte aligned");
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    const int64_t blocks = swiglu_blocks(F, slot_capacity, known_slots, cus);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (bwd)
        swiglu_kernel<true><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(
            static_cast<const uint16_t*>(gu), static_cast<const uint16_t*>(dh), static_cast<uint16_t*>(out),
            expert_offsets, (int)E, slot_capacity, (int)F);
    else
        swiglu_kernel<false><<<dim3((unsigned)blocks), dim3(kThreads), 0, s>>>(
            static_cast<const uint16_t*>(gu), nullptr, static_cast<uint16_t*>(out), expert_offsets, (int)E,
            slot_capacity, (int)F);
    return check_launch(fn);
}

}  // namespace
}  // namespace et

using namespace et;

extern "C" int et_swiglu_fwd(const void* gu, int64_t F, const int32_t* expert_offsets, int64_t num_experts,
                             int64_t slot_capacity, void* h, void* stream)
{
    return launch_swiglu("et_swiglu_fwd", false, gu, nullptr, F, expert_offsets, num_experts, slot_capacity, 0, h,
                         stream);
}

extern "C" int et_swiglu_bwd(const void* gu, const void* dh, int64_t F, const int32_t* expert_offsets,
                             int64_t num_experts, int64_t slot_capacity, void* dgu, void* stream)
{
    return launch_swiglu("et_swiglu_bwd", true, gu, dh, F, expert_offsets, num_experts, slot_capacity, 0, dgu,
                         stream);
}

// The Python API's own forms, not in etmoe.h: as above, for a caller who knows
// that at least known_slots of the capacity's slots are routed.  It only sizes
// the launch: any slot count gives the same result.
extern "C" int et_swiglu_fwd_impl(const void* gu, int64_t F, const int32_t* expert_offsets, int64_t num_experts,
                                  int64_t slot_capacity, void* h, int64_t known_slots, void* stream)
{
    return launch_swiglu("et_swiglu_fwd", false, gu, nullptr, F, expert_offsets, num_experts, slot_capacity,
                         known_slots, h, stream);
}

extern "C" int et_swiglu_bwd_impl(const void* gu, const void* dh, int64_t F, const int32_t* expert_offsets,
                                  int64_t num_experts, int64_t slot_capacity, void* dgu, int64_t known_slots,
                                  void* stream)
{
    return launch_swiglu("et_swiglu_bwd", true, gu, dh, F, expert_offsets, num_experts, slot_capacity, known_slots,
                         dgu, stream);
}

// Blocks of the launch on a device of `cus` compute units (for tests).
extern "C" int64_t et_swiglu_blocks_impl(int64_t F, int64_t slot_capacity, int64_t known_slots, int64_t cus)
{
    return swiglu_blocks(F, slot_capacity, known_slots, cus);
}
