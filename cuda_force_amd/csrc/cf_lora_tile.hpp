// Internal interface of the tiled bf16 LoRA kernels with the adapter as leading
// K-steps (cf_lora_tile.hip).
#pragma once

#include "cf_common.hpp"

namespace cf {

/// Largest adapter rank of these kernels.
inline constexpr int64_t kTileMaxRank = 128;

/// How a problem is cut.
struct TilePlan {
    int config;       // tile shape
    int whole;        // tiles of one workgroup
    int slices;       // of the tiles after them
    int slice_steps;
    float us;         // estimated time, for the choice between these kernels
                      // and the 256x256-tile one of cf_lora_fused.hip
};

/// True when the kernels take a bf16 problem of these sizes: K and N multiples
/// of 8, any rank up to 128, operands below 2 GiB.
bool lora_tile_shape(int64_t M, int64_t N, int64_t K, int64_t rank);

/// The alignment they need: 16-byte aligned x, w, b and y.
bool lora_tile_aligned(const void* x, const void* w, const void* a, const void* b, const void* y, int64_t rank);

/// The plan estimated fastest for sizes that they take.
TilePlan lora_tile_plan(int64_t M, int64_t N, int64_t K, int64_t rank);

/// Bytes of workspace launch_lora_tile needs.
size_t lora_tile_workspace_bytes(const TilePlan& plan, int64_t M, int64_t N, int64_t rank);

/// y = x @ w + scale * bf16(x @ a) @ b; writes the fp32 x @ a to xa_out when
/// it is non-null.
cf_status launch_lora_tile(const TilePlan& plan, const void* x, const void* w, const void* a, const void* b, void* y,
                           float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank,
                           float scale, void* workspace, hipStream_t stream);

}  // namespace cf
