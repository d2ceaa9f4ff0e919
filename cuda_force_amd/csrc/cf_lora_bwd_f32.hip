// Adapter backward of the LoRA linear in fp32 on the fp32 MFMA (gfx950):
//
//   G      = dy @ b^T                [M, r]
//   grad_b = scale * xa^T @ dy       [r, N]
//   grad_a = scale * x^T @ G         [K, r]
//
// derivatives of the reference's _lora_linear_reference
// (python/cudaforge/ops.py:178-185). v_mfma_f32_16x16x4_f32 multiplies and adds
// in fp32, so the results keep the accuracy of fp32 FMA sums.
//
// What bounds it at the sizes of fp32 training (128 x 4096 x 4096): latency, on
// a few MB of operands. One wave per row of G and 256-row chunks left 128
// waves and 64 workgroups on the GPU (G 225 us, each column reduction 42 us),
// so the work is cut small instead: 128 columns x 32 rows per workgroup (128
// or 256 rows of long problems, which still fill the GPU and leave fewer
// partials), straight from memory into MFMA operands (a tile of 32
// rows is 16 KiB and its second use comes from cache), partial sums in the
// workspace, summed in a fixed order by a launch each:
//   1. the dy pass: G partials per 64 columns, grad_b partials per tile of
//      rows;
//   2. their sums;
//   3. the x pass with G: grad_a partials;
//   4. their sum, stored transposed.
// Measured, whole entry: 128 x 4096 x 4096 r16 178.6 -> 15.2 us, 1024 x 4096 x
// 4096 r64 1544 -> 48, 8192 x 4096 x 4096 r16 1032 -> 91.
// Operand layouts: an MFMA takes one k value per 16 lanes. For G a lane loads
// four consecutive columns of its row of dy (and b) and each of four MFMAs
// takes one of them; for the column reductions a lane loads four consecutive
// columns of one row and the four MFMAs produce one column each.
#include "cf_lora_bwd.hpp"

namespace cf {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kTileCols = 128;
constexpr int kHalfCols = 64;
constexpr int64_t kMaxRank = 64;

struct PassArgs {
    const float* v;     // [M, C], the operand reduced over rows
    const float* p;     // [M, rank], the other factor
    const float* b;     // [rank, C] (dy pass)
    float* colpart;     // [row tiles][rank][C]
    float* gpart;       // [ceil(C / 64)][M][rank] (dy pass)
    int64_t M;
    int64_t C;
    int rank;
};

/// Rows kRows blockIdx.y .., columns 128 blockIdx.x ..
template <bool kRowDot, int kRB, int kRows>
__global__ __launch_bounds__(kThreads) void column_f32_kernel(PassArgs args) {
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int g = lane >> 4;
    const int jl = lane & 15;
    const int64_t M = args.M;
    const int64_t C = args.C;
    const int rank = args.rank;
    const int64_t m0 = static_cast<int64_t>(blockIdx.y) * kRows;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * kTileCols + (wave & 1) * kHalfCols;
    const f32x4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};

    if constexpr (kRowDot) {
        // G over this wave's 64 columns for every other block of 16 rows:
        // A = b (row j), B = dy (column m).
        f32x4_t bv[kRB][4];
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
            const int j = 16 * rb + jl;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t n = n0 + 16 * i + 4 * g;
                bv[rb][i] = j < rank && n < C ? *reinterpret_cast<const f32x4_t*>(args.b + j * C + n) : zero;
            }
        }
#pragma unroll 1
        for (int block = wave >> 1; block < kRows / 16; block += 2) {
            const int64_t m = m0 + 16 * block + jl;
            f32x4_t dv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t n = n0 + 16 * i + 4 * g;
                dv[i] = m < M && n < C ? *reinterpret_cast<const f32x4_t*>(args.v + m * C + n) : zero;
            }
            f32x4_t acc[kRB];
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
                acc[rb] = zero;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        acc[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[rb][i][e], dv[i][e], acc[rb], 0, 0, 0);
                    }
                }
            }
            // acc[rb] lane: G[m][16 rb + 4 g + t] over these columns.
            if (m < M && n0 < C) {
                float* dst = args.gpart + (n0 / kHalfCols * M + m) * rank;
#pragma unroll
                for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int j = 16 * rb + 4 * g + t;
                        if (j < rank) dst[j] = acc[rb][t];
                    }
                }
            }
        }
    }

    // The column reduction, two waves taking half the tile's rows each: A = p
    // (row j, k = m),
    // B = v (k = m, column n); MFMA e of the four takes column e of a lane's
    // four.
    const int half = wave >> 1;
    const int64_t n = n0 + 4 * jl;
    f32x4_t acc[kRB][4];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[rb][e] = zero;
    }
    constexpr int kSteps = kRows / 2 / 4;
    constexpr int kGroup = 4;  // K-steps whose loads are in flight together
#pragma unroll 1
    for (int s0 = 0; s0 < kSteps; s0 += kGroup) {
        f32x4_t vv[kGroup];
        float pv[kGroup][kRB];
#pragma unroll
        for (int s = 0; s < kGroup; ++s) {
            const int64_t m = m0 + half * (kRows / 2) + 4 * (s0 + s) + g;
            vv[s] = m < M && n < C ? *reinterpret_cast<const f32x4_t*>(args.v + m * C + n) : zero;
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
                const int j = 16 * rb + jl;
                pv[s][rb] = m < M && j < rank ? args.p[m * rank + j] : 0.0f;
            }
        }
#pragma unroll
        for (int s = 0; s < kGroup; ++s) {
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[rb][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(pv[s][rb], vv[s][e], acc[rb][e], 0, 0, 0);
                }
            }
        }
    }
    // acc[rb][e] lane: [16 rb + 4 g + t][n + e]. The second half's sums reach
    // the first half's waves through LDS.
    __shared__ __attribute__((aligned(16))) f32x4_t sums[2][kRB][4][64];
    if (half == 1) {
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
            for (int e = 0; e < 4; ++e) sums[wave & 1][rb][e][lane] = acc[rb][e];
        }
    }
    __syncthreads();
    if (half == 0 && n < C) {
        float* dst = args.colpart + static_cast<int64_t>(blockIdx.y) * rank * C + n;
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[rb][e] += sums[wave][rb][e][lane];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int64_t j = 16 * rb + 4 * g + t;
                if (j < rank) {
                    *reinterpret_cast<f32x4_t*>(dst + j * C) =
                        f32x4_t{acc[rb][0][t], acc[rb][1][t], acc[rb][2][t], acc[rb][3][t]};
                }
            }
        }
    }
}

/// out[j, n] (or, kTransposed, out[n, j]) = scale * sum over parts of
/// colpart[part][j][n]; thread i handles element i.
template <bool kTransposed>
__device__ __forceinline__ void finish(const float* __restrict__ colpart, float* __restrict__ out, int64_t parts,
                                       int64_t rank, int64_t C, float scale, int64_t i) {
    const int64_t size = rank * C;
    if (i >= size) return;
    const float total = ordered_sum(parts, [&](int64_t t) { return colpart[t * size + i]; });
    const int64_t j = i / C;
    out[kTransposed ? (i - j * C) * rank + j : i] = scale * total;
}

/// grad_b's sum (the first grad_b_blocks workgroups) and G's (the rest).
__global__ __launch_bounds__(kThreads) void after_dy_f32_kernel(const float* __restrict__ colpart,
                                                                float* __restrict__ grad_b,
                                                                const float* __restrict__ gpart,
                                                                float* __restrict__ g, int64_t grad_b_blocks,
                                                                int64_t row_parts, int64_t col_parts,
                                                                int64_t M, int64_t N, int64_t rank,
                                                                float scale) {
    const int64_t block = blockIdx.x;
    if (block < grad_b_blocks) {
        finish<false>(colpart, grad_b, row_parts, rank, N, scale, block * kThreads + threadIdx.x);
        return;
    }
    const int64_t i = (block - grad_b_blocks) * kThreads + threadIdx.x;
    const int64_t size = M * rank;
    if (i < size) g[i] = ordered_sum(col_parts, [&](int64_t t) { return gpart[t * size + i]; });
}

__global__ __launch_bounds__(kThreads) void finish_grad_a_f32_kernel(const float* __restrict__ colpart,
                                                                     float* __restrict__ grad_a,
                                                                     int64_t parts, int64_t rank, int64_t K,
                                                                     float scale) {
    finish<true>(colpart, grad_a, parts, rank, K, scale,
                 static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x);
}

size_t align256(size_t bytes) { return (bytes + 255) / 256 * 256; }

/// Rows of a tile, in both passes: 256 where the narrower one still has a
/// workgroup per CU (4096 x 4096 x 4096 r16 58.7 -> 51.2 us, 8192 x 4096 x 4096
/// r64 328 -> 280; 6000 x 512 x 512 r16, 96 workgroups, 28.0 -> 30.6).
int64_t rows_for(int64_t M, int64_t K, int64_t N) {
    const int64_t columns = ceil_div<int64_t>(K < N ? K : N, kTileCols);
    if (M >= 4096 && ceil_div<int64_t>(M, 256) * columns >= 256) return 256;
    return M >= 512 ? 128 : 32;
}

int64_t row_parts(int64_t M, int64_t K, int64_t N) { return ceil_div<int64_t>(M, rows_for(M, K, N)); }

/// Rows whose G partials are held at a time, whole tiles of every size: all of
/// them while those take 256 MiB (one partial per 64 columns is r / 64 of dy),
/// more in turn.
int64_t panel_rows(int64_t M, int64_t N, int64_t rank) {
    constexpr int64_t kLimit = 256LL << 20;
    const int64_t fit = kLimit / (ceil_div<int64_t>(N, kHalfCols) * rank * 4) / 256 * 256;
    return M <= fit ? M : fit > 256 ? fit : 256;
}

/// `rows`: of a tile, as rows_for the whole problem.
template <bool kRowDot, int kRB>
void launch_pass(const PassArgs& args, int64_t rows, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(ceil_div<int64_t>(args.C, kTileCols)),
                    static_cast<unsigned>(ceil_div<int64_t>(args.M, rows)));
    if (rows == 256) {
        launch(column_f32_kernel<kRowDot, kRB, 256>, grid, dim3(kThreads), 0, stream, args);
    } else if (rows == 128) {
        launch(column_f32_kernel<kRowDot, kRB, 128>, grid, dim3(kThreads), 0, stream, args);
    } else {
        launch(column_f32_kernel<kRowDot, kRB, 32>, grid, dim3(kThreads), 0, stream, args);
    }
}

template <bool kRowDot>
void launch_pass(const PassArgs& args, int64_t rows, hipStream_t stream) {
    if (args.rank <= 16) {
        launch_pass<kRowDot, 1>(args, rows, stream);
    } else if (args.rank <= 32) {
        launch_pass<kRowDot, 2>(args, rows, stream);
    } else {
        launch_pass<kRowDot, 4>(args, rows, stream);
    }
}

}  // namespace

bool lora_backward_f32_shape(int64_t M, int64_t K, int64_t N, int64_t rank) {
    return M > 0 && K > 0 && N > 0 && rank > 0 && rank <= kMaxRank && K % 4 == 0 && N % 4 == 0 &&
           ceil_div<int64_t>(M, 32) <= kMaxGridY;
}

bool lora_backward_f32_eligible(const void* x, const void* dy, const void* b, int64_t M, int64_t K,
                                int64_t N, int64_t rank) {
    return lora_backward_f32_shape(M, K, N, rank) && host_aligned(x, 16) && host_aligned(dy, 16) &&
           host_aligned(b, 16);
}

size_t lora_backward_f32_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t rank) {
    if (!lora_backward_f32_shape(M, K, N, rank)) return 0;
    const int64_t widest = K > N ? K : N;
    return align256(static_cast<size_t>(M * rank) * 4) +
           align256(static_cast<size_t>(ceil_div<int64_t>(N, kHalfCols) * panel_rows(M, N, rank) * rank) * 4) +
           static_cast<size_t>(row_parts(M, K, N) * rank * widest) * 4;
}

cf_status launch_lora_backward_f32(const float* x, const float* dy, const float* b, const float* xa,
                                   float* grad_a, float* grad_b, int64_t M, int64_t K, int64_t N,
                                   int64_t rank, float scale, void* workspace, hipStream_t stream) {
    uint8_t* ws = static_cast<uint8_t*>(workspace);
    float* g = reinterpret_cast<float*>(ws);
    ws += align256(static_cast<size_t>(M * rank) * 4);
    float* gpart = reinterpret_cast<float*>(ws);
    const int64_t panel = panel_rows(M, N, rank);
    ws += align256(static_cast<size_t>(ceil_div<int64_t>(N, kHalfCols) * panel * rank) * 4);
    float* colpart = reinterpret_cast<float*>(ws);

    const int64_t rows = rows_for(M, K, N);
    for (int64_t m0 = 0; m0 < M; m0 += panel) {
        const int64_t count = M - m0 < panel ? M - m0 : panel;
        launch_pass<true>(PassArgs{dy + m0 * N, xa + m0 * rank, b, colpart + m0 / rows * rank * N, gpart, count, N,
                                   static_cast<int>(rank)},
                          rows, stream);
        // G of these rows, and with the last of them grad_b.
        const int64_t grad_b_blocks = m0 + count == M ? ceil_div<int64_t>(rank * N, kThreads) : 0;
        const int64_t g_blocks = ceil_div<int64_t>(count * rank, kThreads);
        launch(after_dy_f32_kernel, dim3(static_cast<unsigned>(grad_b_blocks + g_blocks)), dim3(kThreads), 0,
               stream, colpart, grad_b, gpart, g + m0 * rank, grad_b_blocks, row_parts(M, K, N),
               ceil_div<int64_t>(N, kHalfCols), count, N, rank, scale);
    }
    launch_pass<false>(PassArgs{x, g, nullptr, colpart, nullptr, M, K, static_cast<int>(rank)}, rows, stream);
    launch(finish_grad_a_f32_kernel, dim3(static_cast<unsigned>(ceil_div<int64_t>(rank * K, kThreads))),
           dim3(kThreads), 0, stream, colpart, grad_a, row_parts(M, K, N), rank, K, scale);
    return check_launch("launching the fp32 LoRA backward", stream);
}

}  // namespace cf
