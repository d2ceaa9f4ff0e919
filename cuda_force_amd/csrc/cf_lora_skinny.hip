// bf16 LoRA linear for few rows (token generation, short batches):
//
//   y[M, N] = x[M, K] @ w[K, N] + scale * bf16(x @ a)[M, r] @ b[r, N],  M <= 64
//
// Bound: reading w once (2 K N bytes). A 256x256-tile workgroup per output
// tile leaves all but N / 256 CUs idle here, so the work is cut the other
// way: a workgroup takes 128 columns (256 contiguous bytes of each w row) and
// one slice of K, enough of both to put several workgroups on every CU, and
// w goes from memory straight into registers.
//
//   * A lane loads 16 bytes (8 columns) of the 8 consecutive rows that one
//     MFMA operand takes along k, an 8x8 block of w, and transposes it with
//     v_perm_b32 (32 per 8 KiB of w): no LDS on the way. The product is
//     computed transposed (w^T x^T), so w is the 16-row operand of
//     v_mfma_f32_16x16x32_bf16 and 16 rows of x are the other; MFMA c of the
//     eight takes column c of every lane's block.
//   * The four waves of a workgroup take every fourth 32-row block of the
//     slice and add their accumulators through LDS in a fixed order.
//   * x @ a rides along as one more column strip over the same slices.
//   * A second launch sums the slices in order, rounds x @ a to bf16 (as the
//     reference materialises it), adds scale * (x @ a) @ b and stores bf16.
//
// Measured, weights rotating over 100 MB, streaming kernel + finish: 4 x 4096
// x 4096 r16 10.6 + 3.8 us (the 256x256-tile kernel: 80.8 us), 4 x 4096 x 11008
// 16.8 + 4.1 us = 5.4 TB/s in the first (81.8 us), 32 x 4096 x 4096 14.4 + 4.0,
// 64 x 4096 x 4096 17.1 + 4.7 (81.3). Two choices behind that: the grid stays
// within one round of resident workgroups, strips of a included (16 workgroups
// over, and the round of 16 doubled the time: 64 rows 25.4 us), and the
// finish kernel requests everything before its first wait (7.1 us when it
// summed x @ a first).
//
// Deterministic: every sum has a fixed order, no atomics.
#include "cf_lora_skinny.hpp"

namespace cf {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kStrip = 128;    // columns per workgroup
constexpr int kBlockK = 32;    // k rows of one MFMA step
constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int64_t kMaxRank = 256;
constexpr uint32_t kOutOfRange = 0x80000000u;

struct SkinnyArgs {
    const uint16_t* x;
    const uint16_t* w;
    const uint16_t* a;
    float* part;     // [slices][M][N]
    float* xa_part;  // [slices][M][rank]
    int64_t M;
    int64_t N;
    int64_t K;
    int64_t rank;
    int strips;       // of w; later workgroups of a slice are strips of a
    int slice_blocks; // 32-row blocks per slice
};

/// kMB: 16-row blocks of x. kDepth: blocks of w in flight per wave.
/// kVectorA: rows of a are whole aligned 16-byte pieces.
template <int kMB, int kDepth, int kPerCu, bool kVectorA>
__global__ __launch_bounds__(kThreads, kPerCu) void lora_skinny_kernel(SkinnyArgs args) {
    // One 16-row block's accumulators of the four waves:
    // [wave][t][lane][8 columns].
    __shared__ __attribute__((aligned(16))) float sums[kWaves][4][64][8];

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4;
    const int jl = lane & 15;
    const int64_t M = args.M;
    const int64_t K = args.K;
    const bool is_a = static_cast<int>(blockIdx.x) >= args.strips;
    const uint16_t* src = is_a ? args.a : args.w;
    const int64_t cols = is_a ? args.rank : args.N;
    const int64_t n0 = static_cast<int64_t>(is_a ? static_cast<int>(blockIdx.x) - args.strips
                                                 : static_cast<int>(blockIdx.x)) * kStrip;
    const int64_t col = n0 + 8 * jl;
    const bool vector = kVectorA || !is_a;
    const int64_t k_blocks = ceil_div<int64_t>(K, kBlockK);
    const int64_t first = static_cast<int64_t>(blockIdx.y) * args.slice_blocks;
    const int64_t last = first + args.slice_blocks < k_blocks ? first + args.slice_blocks : k_blocks;

    const __amdgpu_buffer_rsrc_t wbuf = make_buffer(src, static_cast<uint32_t>(K * cols * 2));
    const __amdgpu_buffer_rsrc_t xbuf = make_buffer(args.x, static_cast<uint32_t>(M * K * 2));

    uint4 wv[kDepth][8];
    uint4 xv[kDepth][kMB];
    // Block `block` of the slice's K range: lane (g, j) takes rows 8 g .. +7
    // and columns 8 j .. +7 of w, and of x row j of each 16-row block, the
    // same 8 k. Past the slice, past K (a multiple of 8, so a lane's 8 rows
    // are all inside or all outside) and past M everything reads as zero
    // without touching memory.
    auto load = [&](int slot, int64_t block) {
        const int64_t k0 = block * kBlockK + 8 * g;
        const bool k_ok = block < last && k0 < K;
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb) {
            const int64_t row = 16 * mb + jl;
            const uint32_t off =
                k_ok && row < M ? static_cast<uint32_t>((row * K + k0) * 2) : kOutOfRange;
            xv[slot][mb] = buffer_load16(xbuf, off, 0);
        }
        if (vector) {
            const bool ok = k_ok && col < cols;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t off =
                    ok ? static_cast<uint32_t>(((k0 + i) * cols + col) * 2) : kOutOfRange;
                wv[slot][i] = buffer_load16_stream(wbuf, off, 0);
            }
        } else {
            // a with a rank that is not a multiple of 8: element loads.
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint32_t h[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    h[e] = 0;
                    if (e < cols) {
                        const uint32_t off = k_ok && col + e < cols
                                                 ? static_cast<uint32_t>(((k0 + i) * cols + col + e) * 2)
                                                 : kOutOfRange;
                        h[e] = buffer_load2(wbuf, off, 0);
                    }
                }
                wv[slot][i] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                                         h[6] | (h[7] << 16));
            }
        }
    };

    f32x4_t acc[8][kMB];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb) acc[c][mb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
    auto multiply = [&](int slot) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            // Columns 2 d (low halves) and 2 d + 1 (high halves) of the
            // lane's block as k-contiguous operands.
            uint32_t lo[4];
            uint32_t hi[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t even = reinterpret_cast<const uint32_t*>(&wv[slot][2 * p])[d];
                const uint32_t odd = reinterpret_cast<const uint32_t*>(&wv[slot][2 * p + 1])[d];
                lo[p] = __builtin_amdgcn_perm(odd, even, 0x05040100u);
                hi[p] = __builtin_amdgcn_perm(odd, even, 0x07060302u);
            }
            const bf16x8_t flo = __builtin_bit_cast(bf16x8_t, make_uint4(lo[0], lo[1], lo[2], lo[3]));
            const bf16x8_t fhi = __builtin_bit_cast(bf16x8_t, make_uint4(hi[0], hi[1], hi[2], hi[3]));
#pragma unroll
            for (int mb = 0; mb < kMB; ++mb) {
                const bf16x8_t fx = __builtin_bit_cast(bf16x8_t, xv[slot][mb]);
                acc[2 * d][mb] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(flo, fx, acc[2 * d][mb], 0, 0, 0);
                acc[2 * d + 1][mb] =
                    __builtin_amdgcn_mfma_f32_16x16x32_bf16(fhi, fx, acc[2 * d + 1][mb], 0, 0, 0);
            }
        }
    };

#pragma unroll
    for (int d = 0; d < kDepth; ++d) load(d, first + wave + d * kWaves);
    for (int64_t block = first + wave; block < last; block += kDepth * kWaves) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            // Slots past the slice hold zeros.
            multiply(d);
            load(d, block + (d + kDepth) * kWaves);
        }
    }

    // acc[c][mb][t] of lane (g, j): row 16 mb + j, column n0 + 8 (4 g + t) + c.
    // Wave t sums what the four waves hold for t and stores it.
    float* part = is_a ? args.xa_part : args.part;
    const int64_t out_col = n0 + 8 * (4 * g + wave);
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb) {
        if (mb > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float4* dst = reinterpret_cast<float4*>(&sums[wave][t][lane][0]);
            dst[0] = make_float4(acc[0][mb][t], acc[1][mb][t], acc[2][mb][t], acc[3][mb][t]);
            dst[1] = make_float4(acc[4][mb][t], acc[5][mb][t], acc[6][mb][t], acc[7][mb][t]);
        }
        __syncthreads();
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = 0.0f;
#pragma unroll
        for (int s = 0; s < kWaves; ++s) {
            const float4* p = reinterpret_cast<const float4*>(&sums[s][wave][lane][0]);
            const float4 p0 = p[0];
            const float4 p1 = p[1];
            v[0] += p0.x;
            v[1] += p0.y;
            v[2] += p0.z;
            v[3] += p0.w;
            v[4] += p1.x;
            v[5] += p1.y;
            v[6] += p1.z;
            v[7] += p1.w;
        }
        const int64_t row = 16 * mb + jl;
        if (row < M && out_col < cols) {
            float* dst = part + (static_cast<int64_t>(blockIdx.y) * M + row) * cols + out_col;
            if (vector) {  // cols is a multiple of 8
                reinterpret_cast<float4*>(dst)[0] = make_float4(v[0], v[1], v[2], v[3]);
                reinterpret_cast<float4*>(dst)[1] = make_float4(v[4], v[5], v[6], v[7]);
            } else {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    if (out_col + c < cols) dst[c] = v[c];
                }
            }
        }
    }
}

struct FinishArgs {
    const float* part;
    const float* xa_part;
    const uint16_t* b;
    uint16_t* y;
    float* xa_out;
    int64_t M;
    int64_t N;
    int64_t rank;
    int slices;
    float scale;
};

constexpr int kFinishThreads = 64;
constexpr int kBatch = 16;  // slices (and rows of b) whose loads are in flight together

/// Row blockIdx.y, columns 256 blockIdx.x .. +255 (four per thread). Bound by
/// memory latency, so nothing waits for what it does not use: the x @ a
/// partials, the first rows of b and the first slices of x @ w are all
/// requested before the first wait.
__global__ __launch_bounds__(kFinishThreads) void lora_skinny_finish_kernel(FinishArgs args) {
    __shared__ float u[kMaxRank];
    const int tid = static_cast<int>(threadIdx.x);
    const int64_t row = blockIdx.y;
    const int64_t M = args.M;
    const int64_t N = args.N;
    const int rank = static_cast<int>(args.rank);
    const int slices = args.slices;
    const int64_t col = (static_cast<int64_t>(blockIdx.x) * kFinishThreads + tid) * 4;
    const __amdgpu_buffer_rsrc_t part = make_buffer(args.part, static_cast<uint32_t>(slices * M * N * 4));
    const __amdgpu_buffer_rsrc_t xa_part =
        make_buffer(args.xa_part, static_cast<uint32_t>(slices * M * rank * 4));
    const __amdgpu_buffer_rsrc_t bbuf = make_buffer(args.b, static_cast<uint32_t>(rank * N * 2));

    // x @ a: lanes l, l + 16, l + 32 and l + 48 share adapter column l % 16
    // of a group and take every fourth slice.
    const int jl = tid & 15;
    const int g = tid >> 4;
    for (int j0 = 0; j0 < rank; j0 += 16) {
        const int j = j0 + jl;
        float v = 0.0f;
        for (int s0 = 0; s0 < slices; s0 += 4 * kBatch) {
            float p[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int s = s0 + 4 * i + g;
                const uint32_t off = s < slices && j < rank
                                         ? static_cast<uint32_t>(((s * M + row) * rank + j) * 4)
                                         : kOutOfRange;
                p[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xa_part, off, 0, 0));
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) v += p[i];
        }
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (g == 0 && j < rank) {
            if (args.xa_out != nullptr && blockIdx.x == 0) args.xa_out[row * rank + j] = v;
            u[j] = bf16_bits_to_f32(static_cast<uint16_t>(f32_to_bf16_bits(v)));
        }
    }

    auto load_b = [&](u32x2_t (&bits)[kBatch], int j0) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const uint32_t off = j0 + i < rank && col < N
                                     ? static_cast<uint32_t>(((j0 + i) * N + col) * 2)
                                     : kOutOfRange;
            bits[i] = __builtin_amdgcn_raw_buffer_load_b64(bbuf, off, 0, 0);
        }
    };
    auto load_part = [&](f32x4_t (&v)[kBatch], int s0) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const uint32_t off = s0 + i < slices && col < N
                                     ? static_cast<uint32_t>((((s0 + i) * M + row) * N + col) * 4)
                                     : kOutOfRange;
            v[i] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(part, off, 0, 0));
        }
    };
    f32x4_t v[kBatch];
    u32x2_t bits[kBatch];
    load_part(v, 0);
    load_b(bits, 0);
    f32x4_t total = v[0];
#pragma unroll
    for (int i = 1; i < kBatch; ++i) total += v[i];
    for (int s0 = kBatch; s0 < slices; s0 += kBatch) {
        load_part(v, s0);
#pragma unroll
        for (int i = 0; i < kBatch; ++i) total += v[i];
    }
    __syncthreads();
    f32x4_t adapter = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int j0 = 0; j0 < rank; j0 += kBatch) {
        if (j0 > 0) load_b(bits, j0);
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            // Past the rank u is not read: its place may hold anything.
            const float uj = j0 + i < rank ? u[j0 + i] : 0.0f;
            adapter[0] += uj * bf16_bits_to_f32(bits[i][0] & 0xFFFFu);
            adapter[1] += uj * bf16_bits_to_f32(bits[i][0] >> 16);
            adapter[2] += uj * bf16_bits_to_f32(bits[i][1] & 0xFFFFu);
            adapter[3] += uj * bf16_bits_to_f32(bits[i][1] >> 16);
        }
    }
    if (col >= N) return;
    if (rank > 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) total[e] += args.scale * adapter[e];
    }
    uint2 packed;
    packed.x = f32x2_to_bf16x2_canon(total[0], total[1]);
    packed.y = f32x2_to_bf16x2_canon(total[2], total[3]);
    *reinterpret_cast<uint2*>(args.y + row * N + col) = packed;
}

/// Workgroups of the streaming kernel that fit a CU, by their registers (140
/// with one 16-row block of x, 192 to 214 with more; the element loads of a
/// rank that is not a multiple of 8 spill 65 at three).
int per_cu(int64_t M, int64_t rank) { return M <= 16 && rank % 8 == 0 ? 3 : 2; }

SkinnyPlan plan_for(int64_t M, int64_t N, int64_t K, int64_t rank) {
    SkinnyPlan plan;
    plan.strips = static_cast<int>(ceil_div<int64_t>(N, kStrip));
    plan.a_strips = static_cast<int>(ceil_div<int64_t>(rank, kStrip));
    const int64_t blocks = ceil_div<int64_t>(K, kBlockK);
    // One round of workgroups, strips of a included: a second round would
    // take as long as the first.
    int64_t slices = per_cu(M, rank) * 256 / (plan.strips + plan.a_strips);
    slices = slices < 1 ? 1 : slices;
    // Whole blocks for each of the four waves.
    plan.slice_blocks =
        static_cast<int>(ceil_div<int64_t>(ceil_div<int64_t>(blocks, slices), kWaves) * kWaves);
    plan.slices = static_cast<int>(ceil_div<int64_t>(blocks, plan.slice_blocks));
    return plan;
}

size_t align256(size_t bytes) { return (bytes + 255) / 256 * 256; }

}  // namespace

bool lora_skinny_plan(int64_t M, int64_t N, int64_t K, int64_t rank, SkinnyPlan& plan) {
    if (M < 1 || M > kSkinnyMaxRows || N <= 0 || K <= 0 || N % 8 != 0 || K % 8 != 0 || rank < 0 ||
        rank > kMaxRank) {
        return false;
    }
    // Each operand, and the partials, are read through a buffer whose offsets
    // are 32-bit with the out-of-range marker at 2^31. (The partials of x @ a,
    // at most 768 slices of 64 x 256, are 50 MB.)
    constexpr int64_t kLimit = 1LL << 31;
    if (K >= kLimit || N >= kLimit || K * N * 2 >= kLimit || M * K * 2 >= kLimit || K * rank * 2 >= kLimit ||
        rank * N * 2 >= kLimit) {
        return false;
    }
    plan = plan_for(M, N, K, rank);
    return plan.slices * M * N * 4 < kLimit;
}

bool lora_skinny_aligned(const void* x, const void* w, const void* a, const void* b, const void* y, int64_t rank) {
    return host_aligned(x, 16) && host_aligned(w, 16) && host_aligned(y, 8) &&
           (rank == 0 || (host_aligned(a, 2) && host_aligned(b, 16)));
}

// Two launches, w at the rate of a launch that ramps, and for each output its
// bf16 and its fp32 partials written and read. Of short reductions little is left
// to split, and the 256x256-tile kernel's one launch is the faster way: whole
// call, that one and these, 1 x 64 x 4096 r16 8.3 and 9.3 us, 64 x 128 x 32000
// 10.5 and 22.3, 48 x 1024 x 32000 26.8 and 29.9; 4 x 192 x 4096 11.0 and 9.5, 64 x
// 512 x 4096 17.0 and 11.2, 32 x 2048 x 32000 45 and 36. (Fitted to 174 sizes, K 64
// to 4096 and N 64 to 32000.)
float lora_skinny_estimate_us(const SkinnyPlan& plan, int64_t M, int64_t N, int64_t K) {
    const float outputs = static_cast<float>(M * N);
    const float us = 0.4f + static_cast<float>(K * N * 2) / 5.5e6f +
                     outputs * (5.5f + 3.5f * static_cast<float>(plan.slices)) / 1e6f;
    return us > 5.0f ? us : 5.0f;
}

size_t lora_skinny_workspace_bytes(const SkinnyPlan& plan, int64_t M, int64_t N, int64_t rank) {
    return align256(static_cast<size_t>(plan.slices) * M * N * 4) +
           align256(static_cast<size_t>(plan.slices) * M * rank * 4);
}

cf_status launch_lora_skinny(const SkinnyPlan& plan, const void* x, const void* w, const void* a, const void* b, void* y,
                             float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank,
                             float scale, void* workspace, hipStream_t stream) {
    SkinnyArgs args;
    args.x = static_cast<const uint16_t*>(x);
    args.w = static_cast<const uint16_t*>(w);
    args.a = static_cast<const uint16_t*>(a);
    args.part = static_cast<float*>(workspace);
    args.xa_part = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) +
                                            align256(static_cast<size_t>(plan.slices) * M * N * 4));
    args.M = M;
    args.N = N;
    args.K = K;
    args.rank = rank;
    args.strips = plan.strips;
    args.slice_blocks = plan.slice_blocks;

    const dim3 grid(static_cast<unsigned>(plan.strips + plan.a_strips), static_cast<unsigned>(plan.slices));
    const bool vector_a = rank % 8 == 0 && host_aligned(a, 16);
    auto run = [&](auto vector, auto element) {
        launch(vector_a ? vector : element, grid, dim3(kThreads), 0, stream, args);
    };
    if (M <= 16) {
        run(lora_skinny_kernel<1, 2, 3, true>, lora_skinny_kernel<1, 2, 2, false>);
    } else if (M <= 32) {
        run(lora_skinny_kernel<2, 2, 2, true>, lora_skinny_kernel<2, 2, 2, false>);
    } else {
        run(lora_skinny_kernel<4, 1, 2, true>, lora_skinny_kernel<4, 1, 2, false>);
    }
    FinishArgs finish;
    finish.part = args.part;
    finish.xa_part = args.xa_part;
    finish.b = static_cast<const uint16_t*>(b);
    finish.y = static_cast<uint16_t*>(y);
    finish.xa_out = xa_out;
    finish.M = M;
    finish.N = N;
    finish.rank = rank;
    finish.slices = plan.slices;
    finish.scale = scale;
    launch(lora_skinny_finish_kernel,
           dim3(static_cast<unsigned>(ceil_div<int64_t>(N, 4 * kFinishThreads)), static_cast<unsigned>(M)),
           dim3(kFinishThreads), 0, stream, finish);
    return check_launch("launching the few-row bf16 LoRA kernels", stream);
}

}  // namespace cf
