// Internal interface of the tiled bf16 LoRA kernels with the adapter as leading
// K-steps (cf_lora_tile.hip).
#pragma once

#include "cf_common.hpp"

namespace cf {

/// Largest adapter rank of these kernels.
inline constexpr int64_t kTileMaxRank = 128;

/// True when the kernels take this bf16 problem: K and N multiples of 8, any
/// rank up to 128, 16-byte aligned x, w, b and y, operands below 2 GiB.
bool lora_tile_eligible(const void* x, const void* w, const void* a, const void* b, const void* y,
                        int64_t M, int64_t N, int64_t K, int64_t rank);

/// The same on sizes alone (what the workspace query knows).
bool lora_tile_shape(int64_t M, int64_t N, int64_t K, int64_t rank);

/// Estimated time of the launch in microseconds, for the choice between
/// these kernels and the 256x256-tile one of cf_lora_fused.hip.
float lora_tile_estimate_us(int64_t M, int64_t N, int64_t K, int64_t rank);

/// Bytes of workspace launch_lora_tile needs.
size_t lora_tile_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t rank);

/// y = x @ w + scale * bf16(x @ a) @ b; writes the fp32 x @ a to xa_out when
/// it is non-null.
cf_status launch_lora_tile(const void* x, const void* w, const void* a, const void* b, void* y,
                           float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank,
                           float scale, void* workspace, hipStream_t stream);

}  // namespace cf
