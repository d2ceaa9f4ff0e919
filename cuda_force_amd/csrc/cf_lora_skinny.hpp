// Internal interface of the bf16 LoRA kernels for few rows
// (cf_lora_skinny.hip), used by the C ABI entry points in cf_lora.hip.
#pragma once

#include "cf_common.hpp"

namespace cf {

/// Most rows the kernel takes.
inline constexpr int64_t kSkinnyMaxRows = 64;

/// True when the few-row kernels take this bf16 problem: 1 to 64 rows, K and
/// N multiples of 8, rank up to 256, 16-byte aligned x, w and b, 8-byte
/// aligned y, operands below 2 GiB.
bool lora_skinny_eligible(const void* x, const void* w, const void* a, const void* b, const void* y,
                          int64_t M, int64_t N, int64_t K, int64_t rank);

/// The same on sizes alone (what the workspace query knows).
bool lora_skinny_shape(int64_t M, int64_t N, int64_t K, int64_t rank);

/// Bytes of workspace launch_lora_skinny needs: the slices' fp32 partial
/// x @ w and x @ a.
size_t lora_skinny_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t rank);

/// y = x @ w + scale * bf16(x @ a) @ b in two launches; writes the fp32
/// x @ a to xa_out when it is non-null.
cf_status launch_lora_skinny(const void* x, const void* w, const void* a, const void* b, void* y,
                             float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank,
                             float scale, void* workspace, hipStream_t stream);

}  // namespace cf
