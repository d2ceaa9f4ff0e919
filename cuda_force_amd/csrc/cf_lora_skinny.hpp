// Internal interface of the bf16 LoRA kernels for few rows
// (cf_lora_skinny.hip), used by the C ABI entry points in cf_lora.hip.
#pragma once

#include "cf_common.hpp"

namespace cf {

/// Most rows the kernel takes.
inline constexpr int64_t kSkinnyMaxRows = 64;

/// How a problem is cut.
struct SkinnyPlan {
    int strips;        // of 128 columns of w
    int a_strips;      // of a
    int slices;        // of K
    int slice_blocks;  // 32-row blocks per slice
};

/// True, and the plan, when the few-row kernels take a bf16 problem of these
/// sizes: 1 to 64 rows, K and N multiples of 8, rank up to 256, operands and
/// partials below 2 GiB.
bool lora_skinny_plan(int64_t M, int64_t N, int64_t K, int64_t rank, SkinnyPlan& plan);

/// The alignment they need: 16-byte aligned x, w and b, 8-byte aligned y.
bool lora_skinny_aligned(const void* x, const void* w, const void* a, const void* b, const void* y, int64_t rank);

/// Estimated time of the two launches in microseconds, on the scale of
/// lora_fused_estimate_us (which leaves out some 4 us that every call takes).
float lora_skinny_estimate_us(const SkinnyPlan& plan, int64_t M, int64_t N, int64_t K);

/// Bytes of workspace launch_lora_skinny needs: the slices' fp32 partial
/// x @ w and x @ a.
size_t lora_skinny_workspace_bytes(const SkinnyPlan& plan, int64_t M, int64_t N, int64_t rank);

/// y = x @ w + scale * bf16(x @ a) @ b in two launches; writes the fp32
/// x @ a to xa_out when it is non-null.
cf_status launch_lora_skinny(const SkinnyPlan& plan, const void* x, const void* w, const void* a, const void* b, void* y,
                             float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank,
                             float scale, void* workspace, hipStream_t stream);

}  // namespace cf
