// Internal interface of the MFMA LoRA adapter backwards (bf16 cf_lora_bwd.hip,
// fp32 cf_lora_bwd_f32.hip), used by cf_lora_backward in cf_lora.hip.
#pragma once

#include <type_traits>

#include "cf_common.hpp"

namespace cf {

/// Workgroups in y of one launch, at most (the device reports 65536).
inline constexpr int64_t kMaxGridY = 65535;

/// total += at(t) for t = t .. tiles - 1 in that order, loads issued in
/// groups of 32, 16, 4, then 1 so a thread waits for memory a few times
/// rather than once per eight partials.
template <typename At>
__device__ __forceinline__ float ordered_sum(int64_t tiles, At at) {
    float total = 0.0f;
    int64_t t = 0;
    auto groups = [&](auto group) {
        constexpr int kGroup = decltype(group)::value;
        for (; t + kGroup <= tiles; t += kGroup) {
            float v[kGroup];
#pragma unroll
            for (int k = 0; k < kGroup; ++k) v[k] = at(t + k);
#pragma unroll
            for (int k = 0; k < kGroup; ++k) total += v[k];
        }
    };
    groups(std::integral_constant<int, 32>{});
    groups(std::integral_constant<int, 16>{});
    groups(std::integral_constant<int, 4>{});
    groups(std::integral_constant<int, 1>{});
    return total;
}

/// True when the MFMA backward takes this bf16 problem: 0 < rank <= 64,
/// K and N multiples of 8, 16-byte aligned x, dy, b and grad_x, 31-bit offsets.
bool lora_backward_fast_eligible(const void* x, const void* dy, const void* b, const void* grad_x,
                                 int64_t M, int64_t K, int64_t N, int64_t rank);

/// The same on sizes alone.
bool lora_backward_fast_shape(int64_t M, int64_t K, int64_t N, int64_t rank);

/// Workspace bytes of launch_lora_backward_fast (256-byte aligned pieces); 0
/// for sizes it does not take.
size_t lora_backward_fast_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t rank);

/// grad_a = scale * x^T bf16(dy b^T), grad_b = scale * bf16(xa)^T dy (bf16
/// outputs, fp32 accumulation, fixed-order sums); with grad_x, also
/// grad_x += scale * bf16(dy b^T) a^T in place.
cf_status launch_lora_backward_fast(const void* x, const void* dy, const void* a, const void* b,
                                    const float* xa, void* grad_a, void* grad_b, void* grad_x,
                                    int64_t M, int64_t K, int64_t N, int64_t rank, float scale,
                                    void* workspace, hipStream_t stream);

/// True when the fp32 MFMA backward takes this problem: 0 < rank <= 64, K and N
/// multiples of 4, 16-byte aligned x, dy and b.
bool lora_backward_f32_eligible(const void* x, const void* dy, const void* b, int64_t M, int64_t K,
                                int64_t N, int64_t rank);

/// The same on sizes alone.
bool lora_backward_f32_shape(int64_t M, int64_t K, int64_t N, int64_t rank);

/// Workspace bytes of launch_lora_backward_f32; 0 for sizes it does not take.
size_t lora_backward_f32_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t rank);

/// grad_a = scale * x^T (dy b^T), grad_b = scale * xa^T dy in fp32; dy b^T is
/// left at the start of the workspace as [M, rank].
cf_status launch_lora_backward_f32(const float* x, const float* dy, const float* b, const float* xa,
                                   float* grad_a, float* grad_b, int64_t M, int64_t K, int64_t N,
                                   int64_t rank, float scale, void* workspace, hipStream_t stream);

}  // namespace cf
