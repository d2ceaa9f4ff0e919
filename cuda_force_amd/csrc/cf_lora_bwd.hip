// Adapter backward of the LoRA linear on bf16 MFMA (gfx950), op layout:
//
//   G      = dy @ b^T                 [M, r]   rounded to bf16 (ATen autograd
//                                              sees a bf16 intermediate)
//   grad_b = scale * bf16(xa)^T @ dy  [r, N]
//   grad_a = scale * x^T @ bf16(G)    [K, r]
//
// derivatives of the reference's _lora_linear_reference
// (python/cudaforge/ops.py:178-185, tests/python/test_autograd.py:81-91).
//
// The work is two reductions over M of HBM-sized operands, so the design
// reads dy once and x once (the HBM floor) and keeps everything else small:
//   1. One pass over dy in tiles of 512, 256 or 128 rows x 256 columns (Mp = M
//      rounded up to 512), two 64-row chunks in flight per workgroup, loaded
//      with the non-temporal hint (every byte is read once): each chunk goes
//      HBM -> registers -> LDS; G partial rows = chunk @
//      b^T (16x16x32 MFMA, row fragments by ds_read_b128, b fragments held in
//      registers up to rank 16, in LDS above) and grad_b partials +=
//      bf16(xa)^T-chunk @ chunk (16x16x32
//      MFMA; the chunk's fp32 xa arrives with one 16-byte load per thread
//      and 16 of rank and is rounded and transposed into LDS, the m-contiguous
//      operand is read by ds_read_b64_tr_b16 and meets every block of 16 of
//      the rank). Partials
//      go to fp32 workspaces, one slice per 256-column tile (G) and per
//      row tile (grad_b). Tall tiles mean few partials (512 rows against 256:
//      37.8 against 39.5 us at 8192 x 4096 x 4096 r16, operands cache-cold),
//      so they are lowered only where CUs would idle (chunks_for); three or
//      four chunks in flight were slower.
//   2. One launch sums both in a fixed order: grad_b (times scale, cast) and
//      G -> GT (bf16 [rank padded to 16, 32 or 64, Mp]).
//   3. The same column-reduction pass over x with GT: grad_a partials.
//   4. Their fixed-order sum, times scale, cast, stored transposed.
//   5. With grad_x (dy @ w^T from the caller's GEMM): += scale * G @ a^T.
// Measured, operands rotating: 2000 x 4096 x 4096 r64 31.9 us (1910 on the
// generic path), r16 18.6 (23.7 with 512-row tiles), 4096 x 4096 x 4096 r16
// 23.4 (26.3), 8192 x 4096 x 4096 r16 34.7 as before. The sums are compiled
// per rank padding: with it as a variable they held 32 addresses in 130
// registers and took 1.3 us longer.
// Deterministic: every sum has a fixed order, no atomics.
#include "cf_lora_bwd.hpp"

namespace cf {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;
typedef __attribute__((address_space(3))) uint8_t lds_u8_t;

constexpr int kTileRows = 512;   // rows (M) per workgroup, at most
constexpr int kTileCols = 256;   // columns per workgroup
constexpr int kChunkRows = 64;   // rows staged in LDS at a time
constexpr int kInFlight = 2;     // chunks loaded ahead per workgroup
constexpr int kThreads = 256;
constexpr int kMaxRank = 64;     // the rank is padded to 16, 32 or 64 (kRB MFMA blocks of 16)
constexpr int kRowBytes = kTileCols * 2;
constexpr int kPiecesPerThread = kChunkRows * kTileCols * 2 / 16 / kThreads;  // 8
constexpr uint32_t kOutOfRange = 0x80000000u;
constexpr int kXatStride = kChunkRows + 8;  // bf16 per row of the transposed xa chunk

/// Chunk swizzle of the staged tile (512-byte rows of 32 16-byte chunks).
/// Even, so transposed reads keep their 32-byte column pairs; distinct over
/// rows 0-7 and over rows 8-15 (ds_read_b128 of 16 rows), and distinct in
/// its upper bits over rows {0-3, 8-11} and {4-7, 12-15} (the rows one
/// ds_read_b64_tr_b16 cycle touches).
__device__ __forceinline__ int tile_swizzle(int row) {
    return 2 * ((row & 3) + 4 * (((row >> 2) ^ (row >> 3)) & 1));
}

__device__ __forceinline__ int tile_offset(int row, int chunk) {
    return row * kRowBytes + ((chunk ^ tile_swizzle(row)) << 4);
}

__device__ __forceinline__ s16x4_t lds_read_tr(const uint8_t* base, int offset) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4_t*)((lds_u8_t*)(const_cast<uint8_t*>(base)) + offset));
}

__device__ __forceinline__ bf16x8_t concat(s16x4_t lo, s16x4_t hi) {
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

__device__ __forceinline__ bf16x8_t as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

__device__ __forceinline__ uint32_t buffer_load4(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset,
                                                  uint32_t soffset) {
    return __builtin_amdgcn_raw_buffer_load_b32(rsrc, voffset, soffset, 0);
}

struct ColumnArgs {
    const uint16_t* v;     // [M, C] bf16, the operand reduced over rows
    const uint16_t* pt;    // [16 kRB, Mp] bf16, the other factor, m-contiguous (x pass)
    const float* xa;       // [M, rank] fp32, the other factor of the dy pass
    const uint16_t* b;     // [rank, C] bf16 (row-dot pass only)
    float* colpart;        // [row tiles][16 kRB][C] fp32
    float* gpart;          // [ceil(C / 256)][Mp][16 kRB] fp32 (row-dot pass only)
    int64_t M;
    int64_t Mp;
    int64_t C;
    int64_t rank;
};

/// One tile of kChunks x 64 rows and 256 columns of v: colpart[tile row][j][n] =
/// sum_m pt[j, m] * v[m, n] over the tile's rows; with kRowDot also
/// gpart[tile column][m][j] = sum_n v[m, n] * b[j, n] over its columns.
template <bool kRowDot, int kRB, int kChunks>
__global__ __launch_bounds__(kThreads, kRB == 1 ? 1 : 2) void column_mfma_kernel(ColumnArgs args) {
    constexpr int kRankPad = 16 * kRB;
    constexpr int kXaLoads = kRB;  // 16-byte loads per thread of a chunk's xa (64 rows x rank fp32)
    __shared__ __attribute__((aligned(16))) uint8_t tile[kChunkRows * kRowBytes];  // 32 KiB
    // dy pass: the chunk's xa, rounded to bf16 and transposed ([16 j][64 m],
    // rows padded by 16 bytes); rows j >= rank stay zero.
    __shared__ __attribute__((aligned(16))) uint16_t xat[kRowDot ? kRankPad : 1][kXatStride];
    // dy pass with more than one rank block: b's 256 columns (rows of 512
    // bytes, laid out as the tile's); one block's fragments stay in registers.
    constexpr bool kLdsB = kRowDot && kRB > 1;
    __shared__ __attribute__((aligned(16))) uint8_t btile[kLdsB ? kRankPad * kRowBytes : 16];

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int g = lane >> 4;
    const int jl = lane & 15;
    const int64_t C = args.C;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x) * kTileCols;
    const int64_t mt = blockIdx.y;
    const int64_t m0 = mt * (kChunks * kChunkRows);

    // Staging roles: piece i of thread tid is row 8 i + tid / 32, chunk
    // tid % 32 of the chunk; one wave reads two 512-byte row segments.
    // Rows past M and columns past C read as zero (buffer range check and an
    // out-of-range offset), so they add nothing to either reduction.
    const __amdgpu_buffer_rsrc_t vbuf =
        make_buffer(args.v, static_cast<uint32_t>(args.M * C * 2));
    const int piece_chunk = tid & 31;
    const int64_t piece_col = n0 + 8 * piece_chunk;
    const bool col_ok = piece_col < C;
    // kInFlight chunks in flight: slot s of each staging array holds chunk c
    // with c % kInFlight == s (the chunk loop below is unrolled, so slots are
    // registers).
    uint4 staged[kInFlight][kPiecesPerThread];
    // dy pass: thread t also loads pieces t, t + 256, ... of the chunk's xa rows
    // (64 x rank fp32, contiguous): element q of piece p is flat element
    // 4 p + q = xa[row][col], stored at xat[col][row].
    uint4 staged_xa[kInFlight][kXaLoads];
#pragma unroll
    for (int s = 0; s < kInFlight; ++s) {
#pragma unroll
        for (int p = 0; p < kXaLoads; ++p) staged_xa[s][p] = make_uint4(0u, 0u, 0u, 0u);
    }
    // x pass: the chunk's pt fragments, pt[j = lane % 16][row0 + 32 ms +
    // 8 (lane / 16) .. +7], loaded with the chunk so that waiting for them
    // never waits for a later chunk's loads.
    bf16x8_t staged_pt[kInFlight][kRB][2];
    int xat_at[kXaLoads][4];
    if constexpr (kRowDot) {
#pragma unroll
        for (int p = 0; p < kXaLoads; ++p) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int idx = 4 * (tid + p * kThreads) + q;
                const int rank = static_cast<int>(args.rank);
                xat_at[p][q] = (idx % rank) * kXatStride + idx / rank;
            }
        }
        // Rows j >= rank of the transposed chunk are never written: zero
        // them once (the loop's first barrier orders this before any read).
        for (int i = tid; i < kRankPad * kXatStride; i += kThreads) (&xat[0][0])[i] = 0;
    }
    const __amdgpu_buffer_rsrc_t xabuf = make_buffer(
        args.xa, static_cast<uint32_t>(kRowDot ? args.M * args.rank * 4 : 0));
    const __amdgpu_buffer_rsrc_t ptbuf =
        make_buffer(args.pt, static_cast<uint32_t>(kRowDot ? 0 : kRankPad * args.Mp * 2));
    auto load_chunk = [&](int slot, int64_t row0) {
#pragma unroll
        for (int i = 0; i < kPiecesPerThread; ++i) {
            const int64_t row = row0 + 8 * i + (tid >> 5);
            const uint32_t off =
                col_ok ? static_cast<uint32_t>((row * C + piece_col) * 2) : kOutOfRange;
            staged[slot][i] = buffer_load16_stream(vbuf, off, 0);
        }
        if constexpr (kRowDot) {
            // Past the chunk's kChunkRows x rank elements, or past M: zeros.
#pragma unroll
            for (int p = 0; p < kXaLoads; ++p) {
                const int at = 4 * (tid + p * kThreads);
                const uint32_t off = at < kChunkRows * args.rank
                                         ? static_cast<uint32_t>((row0 * args.rank + at) * 4)
                                         : kOutOfRange;
                staged_xa[slot][p] = buffer_load16(xabuf, off, 0);
            }
        } else {
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
                for (int ms = 0; ms < 2; ++ms) {
                    const uint32_t off =
                        static_cast<uint32_t>(((16 * rb + jl) * args.Mp + row0 + 32 * ms + 8 * g) * 2);
                    staged_pt[slot][rb][ms] = as_bf16x8(buffer_load16(ptbuf, off, 0));
                }
            }
        }
    };
    auto store_chunk = [&](int slot) {
#pragma unroll
        for (int i = 0; i < kPiecesPerThread; ++i) {
            const int row = 8 * i + (tid >> 5);
            *reinterpret_cast<uint4*>(tile + tile_offset(row, piece_chunk)) = staged[slot][i];
        }
        if constexpr (kRowDot) {
#pragma unroll
            for (int p = 0; p < kXaLoads; ++p) {
                if (4 * (tid + p * kThreads) >= kChunkRows * args.rank) continue;
                const uint32_t v[4] = {staged_xa[slot][p].x, staged_xa[slot][p].y, staged_xa[slot][p].z,
                                       staged_xa[slot][p].w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    (&xat[0][0])[xat_at[p][q]] =
                        static_cast<uint16_t>(f32_to_bf16_bits(__uint_as_float(v[q])));
                }
            }
        }
    };

    // Row-dot role: wave w owns chunk rows 16 w .. +15; b fragment s holds
    // b[j = lane % 16][n0 + 32 s + 8 (lane / 16) .. +7].
    bf16x8_t bfrag[kLdsB ? 1 : 8];
    if constexpr (kLdsB) {
        const __amdgpu_buffer_rsrc_t bbuf =
            make_buffer(args.b, static_cast<uint32_t>(args.rank * C * 2));
#pragma unroll
        for (int i = 0; i < kRankPad / 8; ++i) {
            const int row = 8 * i + (tid >> 5);
            const uint32_t off = row < args.rank && col_ok
                                     ? static_cast<uint32_t>((row * C + piece_col) * 2)
                                     : kOutOfRange;
            *reinterpret_cast<uint4*>(btile + tile_offset(row, piece_chunk)) = buffer_load16(bbuf, off, 0);
        }
    } else if constexpr (kRowDot) {
        const __amdgpu_buffer_rsrc_t bbuf =
            make_buffer(args.b, static_cast<uint32_t>(args.rank * C * 2));
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const int64_t col = n0 + 32 * s + 8 * g;
            const uint32_t off = (jl < args.rank && col < C)
                                     ? static_cast<uint32_t>((jl * C + col) * 2)
                                     : kOutOfRange;
            bfrag[s] = as_bf16x8(buffer_load16(bbuf, off, 0));
        }
    }

    // Column-reduction role: wave w owns column blocks 4 w .. 4 w + 3 (16
    // columns each); accumulator lane holds [j = 4 (lane / 16) + t][column
    // 16 cb + lane % 16].
    f32x4_t acc[kRB][4];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[rb][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }

#pragma unroll
    for (int c = 0; c < kInFlight && c < kChunks; ++c) load_chunk(c, m0 + c * kChunkRows);
#pragma unroll
    for (int chunk = 0; chunk < kChunks; ++chunk) {
        const int slot = chunk % kInFlight;
        const int64_t row0 = m0 + static_cast<int64_t>(chunk) * kChunkRows;
        __syncthreads();  // previous chunk's readers are done
        store_chunk(slot);
        __syncthreads();

        // pt fragments. The dy pass reads them from the transposed bf16 copy
        // of the chunk's xa in LDS (rounded as the transposed copy of the x
        // pass is); rows past M and columns past the rank are zero.
        bf16x8_t ptfrag[kRB][2];
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
            for (int ms = 0; ms < 2; ++ms) {
                if constexpr (kRowDot) {
                    ptfrag[rb][ms] =
                        *reinterpret_cast<const bf16x8_t*>(&xat[16 * rb + jl][32 * ms + 8 * g]);
                } else {
                    ptfrag[rb][ms] = staged_pt[slot][rb][ms];
                }
            }
        }
        if (chunk + kInFlight < kChunks) load_chunk(slot, row0 + kInFlight * kChunkRows);

#pragma unroll
        for (int ms = 0; ms < 2; ++ms) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int cb = 4 * wave + c;
                const int row = 32 * ms + 8 * g + (jl >> 2);
                const int ch = 2 * cb + ((jl & 3) >> 1);
                const int off = tile_offset(row, ch) + (jl & 1) * 8;
                // Four rows further down: same swizzle parity pattern, so
                // recompute rather than add.
                const int off_hi = tile_offset(row + 4, ch) + (jl & 1) * 8;
                const bf16x8_t vfrag = concat(lds_read_tr(tile, off), lds_read_tr(tile, off_hi));
#pragma unroll
                for (int rb = 0; rb < kRB; ++rb) {
                    acc[rb][c] =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(ptfrag[rb][ms], vfrag, acc[rb][c], 0, 0, 0);
                }
            }
        }

        if constexpr (kRowDot) {
            f32x4_t gacc[kRB];
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) gacc[rb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            const int row = 16 * wave + jl;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const bf16x8_t afrag =
                    *reinterpret_cast<const bf16x8_t*>(tile + tile_offset(row, 4 * s + g));
#pragma unroll
                for (int rb = 0; rb < kRB; ++rb) {
                    bf16x8_t fb;
                    if constexpr (kLdsB) {
                        fb = *reinterpret_cast<const bf16x8_t*>(btile + tile_offset(16 * rb + jl, 4 * s + g));
                    } else {
                        fb = bfrag[s];
                    }
                    gacc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(afrag, fb, gacc[rb], 0, 0, 0);
                }
            }
            // gacc[rb] lane holds G[row 16 wave + 4 (lane / 16) + t][j = 16 rb + lane % 16].
            float* gp = args.gpart + (static_cast<int64_t>(blockIdx.x) * args.Mp + row0 +
                                      16 * wave + 4 * g) * kRankPad + jl;
#pragma unroll
            for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
                for (int t = 0; t < 4; ++t) gp[t * kRankPad + 16 * rb] = gacc[rb][t];
            }
        }
    }

    // colpart[mt][j][n]: lane holds j = 16 rb + 4 (lane / 16) + t, n = n0 + 16 cb + lane % 16.
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int64_t col = n0 + 16 * (4 * wave + c) + jl;
        if (col >= C) continue;
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                args.colpart[(mt * kRankPad + 16 * rb + 4 * g + t) * C + col] = acc[rb][c][t];
            }
        }
    }
}

/// gt[j, m] = bf16(sum over column tiles of gpart[tile][m][j]), fixed order,
/// and the same row by row in g when that is wanted; thread i of the launch
/// handles element i. Zero past the rank, where the partials of a row with an
/// infinite dy hold NaN (infinity times the padding of b).
template <int kRankPad>
__device__ __forceinline__ void sum_g(const float* __restrict__ gpart, uint16_t* __restrict__ gt,
                                      uint16_t* __restrict__ g, int64_t M, int64_t Mp, int64_t rank, int64_t tiles,
                                      int64_t i) {
    if (i >= kRankPad * Mp) return;
    const int64_t m = i / kRankPad;
    const int64_t j = i % kRankPad;
    // Rows past M are zero, whether or not the dy pass's tiles reach them
    // (the x pass's may be taller).
    float total = 0.0f;
    if (m < M && j < rank) total = ordered_sum(tiles, [&](int64_t t) { return gpart[(t * Mp + m) * kRankPad + j]; });
    const uint16_t bits = static_cast<uint16_t>(f32_to_bf16_bits(total));
    gt[j * Mp + m] = bits;
    if (g != nullptr) g[i] = bits;
}

/// out = scale * sum over row tiles of colpart[tile][j][n], j < rank, as
/// [rank, C] or (kTransposed) [C, rank]; fixed order; thread i handles
/// element i.
template <bool kTransposed, int kRankPad>
__device__ __forceinline__ void finish(const float* __restrict__ colpart, uint16_t* __restrict__ out,
                                       int64_t tiles, int64_t rank, int64_t C, float scale, int64_t i) {
    if (i >= rank * C) return;
    const int64_t j = i / C;
    const int64_t n = i % C;
    const float total =
        ordered_sum(tiles, [&](int64_t t) { return colpart[(t * kRankPad + j) * C + n]; });
    const int64_t dst = kTransposed ? n * rank + j : j * C + n;
    out[dst] = static_cast<uint16_t>(f32_to_bf16_bits(scale * total));
}

/// After the dy pass: grad_b's fixed-order sum (first grad_b_blocks
/// workgroups) and G's (the rest) are independent, so one launch does both.
template <int kRankPad>
__global__ __launch_bounds__(kThreads) void after_dy_kernel(const float* __restrict__ colpart,
                                                            uint16_t* __restrict__ grad_b,
                                                            const float* __restrict__ gpart,
                                                            uint16_t* __restrict__ gt,
                                                            uint16_t* __restrict__ g,
                                                            int64_t grad_b_blocks, int64_t row_tiles,
                                                            int64_t rank, int64_t N, float scale,
                                                            int64_t M, int64_t Mp,
                                                            int64_t col_tiles) {
    const int64_t block = blockIdx.x;
    if (block < grad_b_blocks) {
        finish<false, kRankPad>(colpart, grad_b, row_tiles, rank, N, scale, block * kThreads + threadIdx.x);
    } else {
        sum_g<kRankPad>(gpart, gt, g, M, Mp, rank, col_tiles, (block - grad_b_blocks) * kThreads + threadIdx.x);
    }
}

/// grad_a's fixed-order sum after the x pass, stored transposed ([K, rank]).
template <int kRankPad>
__global__ __launch_bounds__(kThreads) void finish_grad_a_kernel(const float* __restrict__ colpart,
                                                                 uint16_t* __restrict__ grad_a,
                                                                 int64_t row_tiles, int64_t rank,
                                                                 int64_t K, float scale) {
    finish<true, kRankPad>(colpart, grad_a, row_tiles, rank, K, scale,
                 static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x);
}

constexpr int kUpdateCols = 256;  // columns of a workgroup

/// Rows of a workgroup: the smallest a is cheaper to read again than to hold
/// fewer workgroups for (4096 x 4096 r16 17.1 us with 16 rows, 19.4 with 64;
/// 2000 x 4096 r64 15.8 and 10.1).
constexpr int update_rows(int rank_blocks) { return rank_blocks == 1 ? 16 : 64; }

struct UpdateArgs {
    const uint16_t* g;  // [Mp, 16 kRB] bf16(dy @ b^T), zero past the rank
    const uint16_t* a;  // [K, rank]
    uint16_t* grad_x;   // [M, K]
    int64_t M;
    int64_t K;
    int rank;
    float scale;
    bool vector_a;      // rows of a are whole aligned 16-byte pieces
};

/// grad_x += scale * g @ a^T in place, the sum and the product in fp32 and one
/// rounding. Bound by reading and writing grad_x once: a wave takes 64 columns
/// (whole 128-byte lines) of 16 or 64 rows, reading their rows of a once, 16
/// rows at a time with two loads of grad_x per lane (all eight before the first store
/// ran slower). The two MFMAs of 32 columns
/// take the rows of a in an order that leaves a lane eight consecutive columns
/// (16 bytes): row i of the first is column 8 (i / 4) + i % 4, of the second
/// four further.
template <int kRB>
__global__ __launch_bounds__(kThreads) void lora_update_kernel(UpdateArgs args) {
    constexpr int kRankPad = 16 * kRB;
    constexpr int kSteps = (kRankPad + 31) / 32;
    constexpr int kRowBlocks = update_rows(kRB) / 16;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int g = lane >> 4;
    const int jl = lane & 15;
    const int64_t row0 = static_cast<int64_t>(blockIdx.y) * (16 * kRowBlocks) + jl;
    const int64_t col0 = static_cast<int64_t>(blockIdx.x) * kUpdateCols + 64 * wave;
    const int64_t M = args.M;
    const int64_t K = args.K;
    auto load_a = [&](int64_t k, int j) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (k >= K || j >= args.rank) return as_bf16x8(v);
        const uint16_t* src = args.a + k * args.rank + j;
        if (args.vector_a) return as_bf16x8(*reinterpret_cast<const uint4*>(src));
        uint32_t h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = j + e < args.rank ? src[e] : 0u;
        return as_bf16x8(make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                                    h[6] | (h[7] << 16)));
    };
    bf16x8_t af[2][2][kSteps];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int64_t k = col0 + 32 * p + 8 * (jl >> 2) + (jl & 3);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            af[p][0][s] = load_a(k, 32 * s + 8 * g);
            af[p][1][s] = load_a(k + 4, 32 * s + 8 * g);
        }
    }
#pragma unroll 1
    for (int i = 0; i < kRowBlocks; ++i) {
        const int64_t row = row0 + 16 * i;
        uint4 old[2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int64_t col = col0 + 32 * p + 8 * g;
            old[p] = make_uint4(0u, 0u, 0u, 0u);
            if (row < M && col < K) old[p] = *reinterpret_cast<const uint4*>(args.grad_x + row * K + col);
        }
        bf16x8_t gf[kSteps];
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const int j = 32 * s + 8 * g;
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if (row < M && j < kRankPad) v = *reinterpret_cast<const uint4*>(args.g + row * kRankPad + j);
            gf[s] = as_bf16x8(v);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            f32x4_t lo = {0.0f, 0.0f, 0.0f, 0.0f};
            f32x4_t hi = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                lo = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[p][0][s], gf[s], lo, 0, 0, 0);
                hi = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[p][1][s], gf[s], hi, 0, 0, 0);
            }
            const int64_t col = col0 + 32 * p + 8 * g;
            float v[8];
            unpack16<bf16_t>(old[p], v);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v[t] += args.scale * lo[t];
                v[4 + t] += args.scale * hi[t];
            }
            if (row < M && col < K) store_stream16(args.grad_x + row * K + col, pack16<bf16_t>(v));
        }
    }
}

struct Workspace {
    uint16_t* gt;
    uint16_t* g;
    float* gpart;
    float* colpart;
};

size_t align256(size_t bytes) { return (bytes + 255) / 256 * 256; }

int rank_pad_of(int64_t rank) { return rank <= 16 ? 16 : rank <= 32 ? 32 : 64; }

/// Chunks of 64 rows per workgroup: 8, 4 or 2; shorter tiles fill more CUs and
/// leave more partials. Up to rank 16, 512 rows, halved while that still makes
/// one round of a workgroup per CU (2000 x 4096 x 4096 r16 23.7 us, with 128 rows
/// 18.6; 9000 x 2048 x 2048 28.1, with 256 rows, 288 workgroups, 33.4) and at
/// most 64 partials, which few threads would sum (20000 x 1024 x 1024 30.1 with
/// 40, 37.4 with 79). Above, where two workgroups share a CU, the most that still
/// give each CU one; at most 4 for four rank blocks, whose eight unrolled chunks
/// spill.
int chunks_for(int64_t M, int64_t cols, int rank_pad) {
    constexpr int64_t kMaxParts = 64;
    const int64_t tiles = ceil_div<int64_t>(cols, kTileCols);
    for (int chunks = rank_pad == 64 ? 4 : 8; chunks > 2; chunks /= 2) {
        const int64_t parts = ceil_div<int64_t>(M, chunks * kChunkRows);
        const int64_t halved = ceil_div<int64_t>(M, chunks / 2 * kChunkRows);
        if (rank_pad == 16 ? halved * tiles > 256 || halved > kMaxParts : parts * tiles >= 256) return chunks;
    }
    return 2;
}

int64_t padded_rows(int64_t M) { return ceil_div<int64_t>(M, kTileRows) * kTileRows; }

size_t colpart_bytes(int64_t M, int64_t cols, int rank_pad) {
    return static_cast<size_t>(ceil_div<int64_t>(M, chunks_for(M, cols, rank_pad) * kChunkRows) * rank_pad * cols) * 4;
}

Workspace carve(void* base, int64_t M, int64_t N, int rank_pad) {
    const int64_t Mp = padded_rows(M);
    uint8_t* p = static_cast<uint8_t*>(base);
    Workspace ws;
    ws.gt = reinterpret_cast<uint16_t*>(p);
    p += align256(static_cast<size_t>(rank_pad * Mp) * 2);
    ws.g = reinterpret_cast<uint16_t*>(p);
    p += align256(static_cast<size_t>(rank_pad * Mp) * 2);
    ws.gpart = reinterpret_cast<float*>(p);
    p += align256(static_cast<size_t>(ceil_div<int64_t>(N, kTileCols) * Mp * rank_pad) * 4);
    ws.colpart = reinterpret_cast<float*>(p);
    return ws;
}

template <bool kRowDot, int kRB>
void launch_pass(const ColumnArgs& args, int chunks, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(ceil_div<int64_t>(args.C, kTileCols)),
                    static_cast<unsigned>(ceil_div<int64_t>(args.M, chunks * kChunkRows)));
    if (kRB < 4 && chunks == 8) {
        launch(column_mfma_kernel<kRowDot, kRB < 4 ? kRB : 1, 8>, grid, dim3(kThreads), 0, stream, args);
    } else if (chunks == 4) {
        launch(column_mfma_kernel<kRowDot, kRB, 4>, grid, dim3(kThreads), 0, stream, args);
    } else {
        launch(column_mfma_kernel<kRowDot, kRB, 2>, grid, dim3(kThreads), 0, stream, args);
    }
}

template <bool kRowDot>
void launch_pass(const ColumnArgs& args, int rank_pad, int chunks, hipStream_t stream) {
    if (rank_pad == 16) {
        launch_pass<kRowDot, 1>(args, chunks, stream);
    } else if (rank_pad == 32) {
        launch_pass<kRowDot, 2>(args, chunks, stream);
    } else {
        launch_pass<kRowDot, 4>(args, chunks, stream);
    }
}

}  // namespace

bool lora_backward_fast_shape(int64_t M, int64_t K, int64_t N, int64_t rank) {
    // Buffer offsets are 32-bit with an out-of-range marker at 2^31.
    const int64_t Mp = padded_rows(M);
    return M > 0 && K > 0 && N > 0 && rank > 0 && rank <= kMaxRank && K % 8 == 0 && N % 8 == 0 &&
           Mp * K * 2 < (1LL << 31) && Mp * N * 2 < (1LL << 31) && rank * N * 2 < (1LL << 31) &&
           kMaxRank * Mp * 2 < (1LL << 31) && Mp * rank * 4 < (1LL << 31);
}

size_t lora_backward_fast_workspace_bytes(int64_t M, int64_t K, int64_t N, int64_t rank) {
    if (!lora_backward_fast_shape(M, K, N, rank)) return 0;
    const int64_t Mp = padded_rows(M);
    const int rank_pad = rank_pad_of(rank);
    const size_t dy = colpart_bytes(M, N, rank_pad);
    const size_t x = colpart_bytes(M, K, rank_pad);
    return 2 * align256(static_cast<size_t>(rank_pad * Mp) * 2) +
           align256(static_cast<size_t>(ceil_div<int64_t>(N, kTileCols) * Mp * rank_pad) * 4) +
           (dy > x ? dy : x);
}

bool lora_backward_fast_eligible(const void* x, const void* dy, const void* b, const void* grad_x,
                                 int64_t M, int64_t K, int64_t N, int64_t rank) {
    return lora_backward_fast_shape(M, K, N, rank) && host_aligned(x, 16) && host_aligned(dy, 16) &&
           host_aligned(b, 16) && host_aligned(grad_x, 16);
}

cf_status launch_lora_backward_fast(const void* x, const void* dy, const void* a, const void* b,
                                    const float* xa, void* grad_a, void* grad_b, void* grad_x,
                                    int64_t M, int64_t K, int64_t N, int64_t rank, float scale,
                                    void* workspace, hipStream_t stream) {
    const int64_t Mp = padded_rows(M);
    const int rank_pad = rank_pad_of(rank);
    const Workspace ws = carve(workspace, M, N, rank_pad);

    ColumnArgs dy_pass;
    dy_pass.v = static_cast<const uint16_t*>(dy);
    dy_pass.pt = nullptr;
    dy_pass.xa = xa;
    dy_pass.b = static_cast<const uint16_t*>(b);
    dy_pass.colpart = ws.colpart;
    dy_pass.gpart = ws.gpart;
    dy_pass.M = M;
    dy_pass.Mp = Mp;
    dy_pass.C = N;
    dy_pass.rank = rank;
    const int dy_chunks = chunks_for(M, N, rank_pad);
    launch_pass<true>(dy_pass, rank_pad, dy_chunks, stream);
    const int64_t grad_b_blocks = ceil_div<int64_t>(rank * N, kThreads);
    const int64_t g_blocks = ceil_div<int64_t>(rank_pad * Mp, kThreads);
    auto after_dy = [&](auto kernel) {
        launch(kernel, dim3(static_cast<unsigned>(grad_b_blocks + g_blocks)), dim3(kThreads), 0, stream,
               ws.colpart, static_cast<uint16_t*>(grad_b), ws.gpart, ws.gt,
               grad_x != nullptr ? ws.g : nullptr, grad_b_blocks,
               ceil_div<int64_t>(M, dy_chunks * kChunkRows), rank, N, scale, M, Mp,
               ceil_div<int64_t>(N, kTileCols));
    };
    rank_pad == 16   ? after_dy(after_dy_kernel<16>)
    : rank_pad == 32 ? after_dy(after_dy_kernel<32>)
                     : after_dy(after_dy_kernel<64>);

    ColumnArgs x_pass;
    x_pass.v = static_cast<const uint16_t*>(x);
    x_pass.pt = ws.gt;
    x_pass.xa = nullptr;
    x_pass.b = nullptr;
    x_pass.colpart = ws.colpart;
    x_pass.gpart = nullptr;
    x_pass.M = M;
    x_pass.Mp = Mp;
    x_pass.C = K;
    x_pass.rank = rank;
    const int x_chunks = chunks_for(M, K, rank_pad);
    launch_pass<false>(x_pass, rank_pad, x_chunks, stream);
    auto finish_grad_a = [&](auto kernel) {
        launch(kernel, dim3(static_cast<unsigned>(ceil_div<int64_t>(rank * K, kThreads))), dim3(kThreads), 0,
               stream, ws.colpart, static_cast<uint16_t*>(grad_a),
               ceil_div<int64_t>(M, x_chunks * kChunkRows), rank, K, scale);
    };
    rank_pad == 16   ? finish_grad_a(finish_grad_a_kernel<16>)
    : rank_pad == 32 ? finish_grad_a(finish_grad_a_kernel<32>)
                     : finish_grad_a(finish_grad_a_kernel<64>);
    if (grad_x != nullptr) {
        // As many rows a launch as grid.y takes.
        const int rows_each = update_rows(rank_pad / 16);
        const int64_t rows_per_launch = rows_each * kMaxGridY;
        for (int64_t row0 = 0; row0 < M; row0 += rows_per_launch) {
            UpdateArgs update;
            update.g = ws.g + row0 * rank_pad;
            update.a = static_cast<const uint16_t*>(a);
            update.grad_x = static_cast<uint16_t*>(grad_x) + row0 * K;
            update.M = M - row0 < rows_per_launch ? M - row0 : rows_per_launch;
            update.K = K;
            update.rank = static_cast<int>(rank);
            update.scale = scale;
            update.vector_a = rank % 8 == 0 && host_aligned(a, 16);
            const dim3 grid(static_cast<unsigned>(ceil_div<int64_t>(K, kUpdateCols)),
                            static_cast<unsigned>(ceil_div<int64_t>(update.M, rows_each)));
            if (rank_pad == 16) {
                launch(lora_update_kernel<1>, grid, dim3(kThreads), 0, stream, update);
            } else if (rank_pad == 32) {
                launch(lora_update_kernel<2>, grid, dim3(kThreads), 0, stream, update);
            } else {
                launch(lora_update_kernel<4>, grid, dim3(kThreads), 0, stream, update);
            }
        }
    }
    return check_launch("launching the bf16 LoRA backward", stream);
}

}  // namespace cf
