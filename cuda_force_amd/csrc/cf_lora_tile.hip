// bf16 LoRA linear in tiles below 256x256, any rank up to 128, K and N any
// multiples of 8:
//
//   y[M, N] = x[M, K] @ w[K, N] + scale * bf16(x @ a)[M, r] @ b[r, N]
//
// The adapter is the start of the reduction: with u = bf16(x @ a), the first
// one to four K-steps run over the rows of b, the accumulators are multiplied
// by the scale once, in fp32, and the K-steps of x @ w add on. So the adapter
// is scale * (u @ b) in fp32, as written above, for any scale and any b
// (infinities included), and the epilogue knows no adapter.
//
//   * lora_down_kernel forms x @ a first (16 rows per workgroup, its waves
//     splitting K) and rounds it to bf16 (as the reference materialises it)
//     into u.
//   * lora_tile_kernel: K-step 32, operands HBM -> LDS by buffer loads with the
//     LDS destination into a ring of stages, one barrier per K-step; the
//     fragments of step j + 1 are read while step j is multiplied, and the
//     copies of step j + stages - 1 are spread through its MFMAs.
//   * Few output tiles split the K-steps over grid.y; the slices' fp32 partial
//     tiles are summed in order by a last launch.
//
// What bounds it: copying the operands into LDS, not the MFMAs. Timing-only
// copies at 1000 x 4096 x 4096 (256 tiles of 128x128, no adapter): whole
// kernel 53.4 us without the fragments read ahead and 43 us with them, copies
// alone 40.8, MFMAs alone 22.4; deeper rings change nothing, and shapes that
// fill the CUs move 11-13 TB/s from L2 to LDS (42-51 GB/s per CU; by kernel
// trace 1000 x 4096 x 4096 11.1, 1237 x 4096 x 8192 12.9, 6000 x 11008 x 4096
// 12.2). So the widest tile that still fills the CUs wins, and the kernel and
// slice counts are chosen by an estimate (below) from measured times per K-step. Before, these problems
// ran 256x256 tiles on a fraction of the CUs or, for a rank above 16 or K not
// a multiple of 64, fp32 FMA tiles: 333 x 4096 x 11008 r16 92 -> 58 us, 100 x
// 4096 x 4096 r16 81 -> 23, 1237 x 4096 x 8192 r64 2801 -> 108, 3530 x 984 x
// 11008 r16 1367 -> 107, 6000 x 11008 x 4096 r32 12650 -> 573.
//
// Everything past an edge reads as zero: rows past M and columns past N by the
// buffer range, k past K by an offset bit (x) and by the range (w).
#include "cf_lora_tile.hpp"
#include "cf_lds_dma.hpp"

#include <cmath>

namespace cf {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;
typedef __attribute__((address_space(3))) uint8_t lds_u8_t;

constexpr int kBK = 32;

__device__ __forceinline__ s16x4_t lds_read_tr(const uint8_t* base, int offset) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4_t*)((lds_u8_t*)(const_cast<uint8_t*>(base)) + offset));
}

__device__ __forceinline__ bf16x8_t concat(s16x4_t lo, s16x4_t hi) {
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

/// Chunk swizzle of a k-contiguous tile (64-byte rows of four 16-byte
/// chunks): rows 4 apart trade places with the chunk two further, so the
/// eight rows of an octet of a ds_read_b128, and the octet served with it
/// (which reads a chunk of the other parity), fall into different banks.
__device__ __forceinline__ int k_swizzle(int row) { return 2 * ((row >> 2) & 1); }

/// Chunk swizzle of an n-contiguous tile (rows of at least 16 chunks), for
/// ds_read_b64_tr_b16: k rows 0-3 in four 32-byte bank groups, rows 8 apart
/// in the other half of the banks.
__device__ __forceinline__ int n_swizzle(int row) { return 2 * (row & 3) + 8 * ((row >> 3) & 1); }

/// Workgroup ids are dealt round-robin over the 8 XCDs: position `id` of
/// `total` such that each XCD gets a run of consecutive positions, whatever
/// the total.
__device__ __forceinline__ int xcd_run(int id, int total) {
    constexpr int kXcds = 8;
    const int xcd = id % kXcds;
    const int each = total / kXcds;
    const int more = total % kXcds;
    return xcd * each + (xcd < more ? xcd : more) + id / kXcds;
}

/// Tile `position`: row tiles fastest within bands of four, so the tiles that
/// read the same columns of w, and then the same rows of x, are neighbours.
__device__ __forceinline__ void place_tile(int position, int tiles_m, int tiles_n, int& tm, int& tn) {
    constexpr int kBand = 4;
    const int band = position / (kBand * tiles_n);
    const int rows = tiles_m - band * kBand < kBand ? tiles_m - band * kBand : kBand;
    const int in_band = position - band * kBand * tiles_n;
    tm = band * kBand + in_band % rows;
    tn = in_band / rows;
}

struct TileArgs {
    const uint16_t* x;    // [M, K]
    const uint16_t* w;    // [K, N]
    const uint16_t* u;    // [M, ext]: bf16(x @ a), zero-padded
    const uint16_t* b;    // [rank, N]
    uint16_t* y;          // [M, N]
    float* part;          // split tiles: [tile - whole][slice][rows of the tile][columns]
    int64_t M;
    int64_t N;
    int64_t K;
    int64_t rank;
    int64_t ext;          // the rank as whole K-steps: a multiple of kBK
    int steps;            // K-steps of the adapter, then of x @ w
    int ext_steps;        // of the adapter
    float scale;
    int tiles_m;
    int tiles_n;
    int whole;            // the first tiles take a workgroup each; those after
    int slices;           // them take `slices`, each `slice_steps` K-steps
    int slice_steps;
};

/// A workgroup of kWM x kWN waves, each computing 16 kTM rows by 16 kTN
/// columns.
template <int kTM, int kTN, int kWM, int kWN, int kStages, int kPerSimd>
__global__ __launch_bounds__(kWM * kWN * 64) __attribute__((amdgpu_waves_per_eu(kPerSimd, kPerSimd)))
void lora_tile_kernel(TileArgs args) {
    constexpr int kWaves = kWM * kWN;
    constexpr int kBM = 16 * kTM * kWM;
    constexpr int kBN = 16 * kTN * kWN;
    constexpr int kXBytes = kBM * kBK * 2;
    constexpr int kWBytes = kBN * kBK * 2;
    constexpr int kStage = kXBytes + kWBytes;
    constexpr int kXPieces = kXBytes / 1024 / kWaves;  // DMA instructions per wave and K-step
    constexpr int kWPieces = kWBytes / 1024 / kWaves;
    constexpr int kPieces = kXPieces + kWPieces;
    constexpr int kOutRow = kTN * 32;                  // bytes of a wave's output row
    static_assert(kXPieces * kWaves * 1024 == kXBytes && kWPieces * kWaves * 1024 == kWBytes,
                  "whole DMA instructions per wave");
    static_assert(kWaves * 16 * kTM * kOutRow <= kStages * kStage, "output staging");
    __shared__ __attribute__((aligned(16))) uint8_t lds[kStages * kStage];

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / kWN;
    const int wn = wave % kWN;
    const int g = lane >> 4;
    const int jl = lane & 15;
    const int id = static_cast<int>(blockIdx.x);
    const bool split = id >= args.whole;
    const int split_tiles = args.tiles_m * args.tiles_n - args.whole;
    int position;
    int slice = 0;
    if (split) {
        // Slice by slice, so that neighbours read the same part of w or x.
        const int at = xcd_run(id - args.whole, split_tiles * args.slices);
        slice = at / split_tiles;
        position = args.whole + at % split_tiles;
    } else {
        position = xcd_run(id, args.whole);
    }
    int tm;
    int tn;
    place_tile(position, args.tiles_m, args.tiles_n, tm, tn);
    const int64_t m0 = static_cast<int64_t>(tm) * kBM;
    const int64_t n0 = static_cast<int64_t>(tn) * kBN;
    const int64_t M = args.M;
    const int64_t N = args.N;
    const int first = slice * args.slice_steps;
    const int last = split && first + args.slice_steps < args.steps ? first + args.slice_steps : args.steps;

    // x and u: a DMA instruction fills 16 rows; lane l -> row l / 4, physical
    // chunk l % 4. The rows of an instruction and the K-step travel in the
    // scalar offset.
    const int64_t rows_here = M - m0 < kBM ? M - m0 : kBM;
    const uint32_t x_row = static_cast<uint32_t>(args.K * 2);
    const uint32_t u_row = static_cast<uint32_t>(args.ext * 2);
    const i32x4_t xbuf = uniform(
        raw_buffer_words(args.x + m0 * args.K, static_cast<uint32_t>(rows_here) * x_row));
    const i32x4_t ubuf = uniform(
        raw_buffer_words(args.u + m0 * args.ext, static_cast<uint32_t>(rows_here) * u_row));
    const int x_chunk = (lane & 3) ^ k_swizzle(lane >> 2);
    const uint32_t x_lane = static_cast<uint32_t>(lane >> 2) * x_row + static_cast<uint32_t>(x_chunk * 16);
    const uint32_t u_lane = static_cast<uint32_t>(lane >> 2) * u_row + static_cast<uint32_t>(x_chunk * 16);
    // w and b: an instruction fills 512 / kBN rows.
    constexpr int kRowChunks = kBN / 8;
    constexpr int kRowsPerPiece = 64 / kRowChunks;
    const i32x4_t wbuf = uniform(raw_buffer_words(args.w, static_cast<uint32_t>(args.K * N * 2)));
    const i32x4_t bbuf = uniform(raw_buffer_words(args.b, static_cast<uint32_t>(args.rank * N * 2)));
    uint32_t w_lane[kWPieces];
#pragma unroll
    for (int i = 0; i < kWPieces; ++i) {
        const int row = (wave * kWPieces + i) * kRowsPerPiece + lane / kRowChunks;
        const int64_t col = n0 + 8 * ((lane % kRowChunks) ^ n_swizzle(row));
        w_lane[i] = col < N ? static_cast<uint32_t>((row * N + col) * 2) : kOutOfRange;
    }

    const uint32_t lds_addr = static_cast<uint32_t>(reinterpret_cast<size_t>((lds_u8_t*)lds));
    // Where K-step `step` comes from, for the copies of one step.
    struct Source {
        i32x4_t x;
        i32x4_t w;
        uint32_t x_off;   // lane offset, past the buffer for k past K
        uint32_t x_step;  // scalar offset of the K-step, and bytes per row
        uint32_t x_row;
        uint32_t w_step;
        uint32_t stage;   // LDS address
    };
    auto source = [&](int step, int slot) {
        // Uniform already; said so that the selected descriptors stay scalar.
        step = __builtin_amdgcn_readfirstlane(step);
        slot = __builtin_amdgcn_readfirstlane(slot);
        const bool ext = step < args.ext_steps;
        const int k0 = (ext ? step : step - args.ext_steps) * kBK;
        Source s;
        s.x = ext ? ubuf : xbuf;
        s.w = ext ? bbuf : wbuf;
        if (step >= last) {
            // Past the slice: an empty range, so every step issues the same
            // number of copies and nothing is read.
            s.x[2] = 0;
            s.w[2] = 0;
        }
        s.x = uniform(s.x);
        s.w = uniform(s.w);
        const uint32_t past = ext || k0 + 8 * x_chunk < args.K ? 0u : kOutOfRange;
        s.x_off = (ext ? u_lane : x_lane) | past;
        s.x_step = static_cast<uint32_t>(k0 * 2);
        s.x_row = ext ? u_row : x_row;
        s.w_step = static_cast<uint32_t>(k0) * static_cast<uint32_t>(N * 2);
        s.stage = lds_addr + static_cast<uint32_t>(slot * kStage);
        return s;
    };
    auto copy = [&](const Source& s, int i) {
        if (i < kXPieces) {
            const uint32_t piece = static_cast<uint32_t>(wave * kXPieces + i);
            dma16_m0(s.x, s.stage + piece * 1024, s.x_off, s.x_step + 16 * piece * s.x_row);
        } else {
            const uint32_t piece = static_cast<uint32_t>(wave * kWPieces + i - kXPieces);
            dma16_m0(s.w, s.stage + kXBytes + piece * 1024, w_lane[i - kXPieces], s.w_step);
        }
    };

    // Fragment addresses: x (B operand) row 16 (kTM wm + i) + lane % 16, chunk
    // lane / 16; w (A operand, transposed read) k rows 8 g + j / 4 (then + 4),
    // columns 4 (j % 4) .. +3 of column block kTN wn + jb.
    const int x_rd = (wm * kTM * 16 + jl) * (kBK * 2) + ((g ^ k_swizzle(jl)) << 4);
    int w_rd[kTN];
#pragma unroll
    for (int jb = 0; jb < kTN; ++jb) {
        const int row = 8 * g + (jl >> 2);
        const int chunk = 2 * (wn * kTN + jb) + ((jl & 3) >> 1);
        w_rd[jb] = kXBytes + row * (kBN * 2) + ((chunk ^ n_swizzle(row)) << 4) + (jl & 1) * 8;
    }

    f32x4_t acc[kTN][kTM];
#pragma unroll
    for (int jb = 0; jb < kTN; ++jb) {
#pragma unroll
        for (int i = 0; i < kTM; ++i) acc[jb][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }

    const int steps = last - first;
#pragma unroll
    for (int t = 0; t < kStages - 1; ++t) {
        const Source s = source(first + t, t);
#pragma unroll
        for (int i = 0; i < kPieces; ++i) copy(s, i);
    }
    bf16x8_t x0[kTM];
    bf16x8_t x1[kTM];
    bf16x8_t wf[kTN];
    auto read_x = [&](bf16x8_t (&xf)[kTM], const uint8_t* stage) {
#pragma unroll
        for (int i = 0; i < kTM; ++i) {
            xf[i] = *reinterpret_cast<const bf16x8_t*>(stage + x_rd + i * (16 * kBK * 2));
        }
    };
    auto read_w = [&](const uint8_t* stage, int jb) {
        return concat(lds_read_tr(stage, w_rd[jb]), lds_read_tr(stage, w_rd[jb] + 4 * kBN * 2));
    };
    // K-step kt + 1 has landed once at most the copies of the kStages - 3
    // steps after it are outstanding. The LDS reads of step kt - 1, whose slot
    // this step's copies fill, have returned in every wave that reaches the
    // barrier.
    auto arrive = [&]() {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((kStages - 3) * kPieces) & ~(15 << 8));
        bare_barrier();
    };
    // K-step 0 in LDS.
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((kStages - 2) * kPieces));
    bare_barrier();
    read_x(x0, lds);
#pragma unroll
    for (int jb = 0; jb < kTN; ++jb) wf[jb] = read_w(lds, jb);
    auto scale_adapter = [&]() {
#pragma unroll
        for (int jb = 0; jb < kTN; ++jb) {
#pragma unroll
            for (int i = 0; i < kTM; ++i) acc[jb][i] *= args.scale;
        }
    };
    int slot = 0;
    auto step = [&](int kt, bf16x8_t (&cur)[kTM], bf16x8_t (&nxt)[kTM]) {
        arrive();
        const int next = slot == kStages - 1 ? 0 : slot + 1;
        const uint8_t* stage = lds + next * kStage;
        const Source s = source(first + kt + kStages - 1, slot == 0 ? kStages - 1 : slot - 1);
        slot = next;
        read_x(nxt, stage);
#pragma unroll
        for (int jb = 0; jb < kTN; ++jb) {
#pragma unroll
            for (int i = 0; i < kTM; ++i) {
                acc[jb][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[jb], cur[i], acc[jb][i], 0, 0, 0);
            }
            wf[jb] = read_w(stage, jb);
            constexpr int kEach = (kPieces + kTN - 1) / kTN;
#pragma unroll
            for (int q = 0; q < kEach; ++q) {
                if (jb * kEach + q < kPieces) copy(s, jb * kEach + q);
            }
            // In this order: left to itself the compiler gathers the 128x256
            // tile's 32 MFMAs behind all the reads and copies (2000 x 4096 x
            // 4096 r64 83.9 us, 80.3 like this).
            if (kTN == 8 && jb < kTN - 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto final_step = [&](bf16x8_t (&cur)[kTM]) {
#pragma unroll
        for (int jb = 0; jb < kTN; ++jb) {
#pragma unroll
            for (int i = 0; i < kTM; ++i) {
                acc[jb][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[jb], cur[i], acc[jb][i], 0, 0, 0);
            }
        }
    };
    int kt = 0;
    // The adapter's K-steps of this slice (at most four), in a loop of their
    // own: tested for in the loop below, the scale took config 0's 128
    // accumulators out of the accumulation registers, and spilled.
    const int lead = args.ext_steps > first ? args.ext_steps - first : 0;
#pragma unroll 1
    for (; kt < lead && kt + 1 < steps; ++kt) {
        step(kt, x0, x1);
#pragma unroll
        for (int i = 0; i < kTM; ++i) x0[i] = x1[i];
    }
    if (lead > 0 && lead < steps) scale_adapter();
    for (; kt + 2 < steps; kt += 2) {
        step(kt, x0, x1);
        step(kt + 1, x1, x0);
    }
    if (kt + 1 < steps) {
        step(kt, x0, x1);
        final_step(x1);
    } else {
        final_step(x0);
    }
    if (lead >= steps) scale_adapter();  // a slice within the adapter

    // acc[jb][i] lane: row m0 + 16 (kTM wm + i) + lane % 16, columns
    // n0 + 16 (kTN wn + jb) + 4 g .. +3; N is a multiple of 8, so those four
    // are all inside or all outside.
    const int64_t row0 = m0 + wm * kTM * 16;
    const int64_t col0 = n0 + wn * kTN * 16;
    if (split) {
        float* dst = args.part + (static_cast<int64_t>(position - args.whole) * args.slices + slice) * (kBM * kBN);
#pragma unroll
        for (int i = 0; i < kTM; ++i) {
            const int row = wm * kTM * 16 + 16 * i + jl;
#pragma unroll
            for (int jb = 0; jb < kTN; ++jb) {
                const int col = wn * kTN * 16 + 16 * jb + 4 * g;
                *reinterpret_cast<f32x4_t*>(dst + row * kBN + col) = acc[jb][i];
            }
        }
    } else {
        // Through LDS, so that a store instruction writes whole row pieces of
        // the wave's tile: chunk c of row r at c ^ r (mod the row's chunks).
        constexpr int kChunks = kOutRow / 16;
        // Every wave has left the operand stages, and the copies past the
        // end (zeros) have landed.
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0) & ~(15 << 8));
        bare_barrier();
        uint8_t* out = lds + wave * (16 * kTM * kOutRow);
#pragma unroll
        for (int i = 0; i < kTM; ++i) {
            const int row = 16 * i + jl;
#pragma unroll
            for (int jb = 0; jb < kTN; ++jb) {
                const int chunk = 2 * jb + (g >> 1);
                uint2 packed;
                packed.x = f32x2_to_bf16x2_canon(acc[jb][i][0], acc[jb][i][1]);
                packed.y = f32x2_to_bf16x2_canon(acc[jb][i][2], acc[jb][i][3]);
                *reinterpret_cast<uint2*>(out + row * kOutRow + ((chunk ^ (row & (kChunks - 1))) << 4) +
                                          (g & 1) * 8) = packed;
            }
        }
        // Only this wave reads what it wrote, and its LDS operations complete
        // in order; the fence keeps the compiler from reordering them.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int c = lane % kChunks;
        const int64_t col = col0 + 8 * c;
        constexpr int kRows = 64 / kChunks;
#pragma unroll
        for (int s = 0; s < 16 * kTM / kRows; ++s) {
            const int row = kRows * s + lane / kChunks;
            const uint4 v =
                *reinterpret_cast<const uint4*>(out + row * kOutRow + ((c ^ (row & (kChunks - 1))) << 4));
            if (row0 + row < M && col < N) store_stream16(args.y + (row0 + row) * N + col, v);
        }
    }
}

/// The split tiles: y = bf16(sum of the slices' partials, in order), eight
/// outputs per thread; blockIdx.y is the tile.
__global__ __launch_bounds__(kDefaultBlockSize) void lora_tile_sum_kernel(TileArgs args, int bm, int bn) {
    const int at = static_cast<int>(blockIdx.x * kDefaultBlockSize + threadIdx.x) * 8;
    const int row = at / bn;
    const int col = at - row * bn;
    int tm;
    int tn;
    place_tile(args.whole + static_cast<int>(blockIdx.y), args.tiles_m, args.tiles_n, tm, tn);
    const int64_t m = static_cast<int64_t>(tm) * bm + row;
    const int64_t n = static_cast<int64_t>(tn) * bn + col;
    if (m >= args.M || n >= args.N) return;
    const int64_t size = static_cast<int64_t>(bm) * bn;
    const float* part = args.part + blockIdx.y * args.slices * size + at;
    f32x4_t lo = *reinterpret_cast<const f32x4_t*>(part);
    f32x4_t hi = *reinterpret_cast<const f32x4_t*>(part + 4);
#pragma unroll 4
    for (int s = 1; s < args.slices; ++s) {
        lo += *reinterpret_cast<const f32x4_t*>(part + s * size);
        hi += *reinterpret_cast<const f32x4_t*>(part + s * size + 4);
    }
    uint4 v;
    v.x = f32x2_to_bf16x2_canon(lo[0], lo[1]);
    v.y = f32x2_to_bf16x2_canon(lo[2], lo[3]);
    v.z = f32x2_to_bf16x2_canon(hi[0], hi[1]);
    v.w = f32x2_to_bf16x2_canon(hi[2], hi[3]);
    *reinterpret_cast<uint4*>(args.y + m * args.N + n) = v;
}

// ---------------------------------------------------------------------------
// x @ a.
// ---------------------------------------------------------------------------

constexpr int kDownWaves = 8;
constexpr int kDownThreads = kDownWaves * 64;

struct DownArgs {
    const uint16_t* x;  // [M, K]
    const uint16_t* a;  // [K, rank]
    uint16_t* u;        // [M, ext]
    float* xa_out;      // [M, rank] or null
    int64_t M;
    int64_t K;
    int rank;
    int ext;
    bool vector_a;      // rows of a are whole aligned 16-byte pieces
    bool pair_a;        // rows of a are whole aligned 4-byte pairs
};

/// kRB: 16-column blocks of a.
template <int kRB>
__global__ __launch_bounds__(kDownThreads) void lora_down_kernel(DownArgs args) {
    // Per wave: a's rows of one K-step ([32 k][16 kRB], read transposed); after
    // the loop the waves' accumulators ([wave][block][lane] float4).
    constexpr int kRowBytes = 32 * kRB;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kDownWaves * kBK * kRowBytes];
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4;
    const int jl = lane & 15;
    const int rank = args.rank;
    const int ext = args.ext;

    const int64_t m0 = static_cast<int64_t>(blockIdx.x) * 16;
    const int64_t rows_here = args.M - m0 < 16 ? args.M - m0 : 16;
    const __amdgpu_buffer_rsrc_t xbuf =
        make_buffer(args.x + m0 * args.K, static_cast<uint32_t>(rows_here * args.K * 2));
    const __amdgpu_buffer_rsrc_t abuf = make_buffer(args.a, static_cast<uint32_t>(args.K * rank * 2));
    uint8_t* mine = lds + wave * (kBK * kRowBytes);

    constexpr int kDepth = kRB <= 2 ? 6 : kRB == 4 ? 4 : 3;  // K-steps in flight per wave
    uint4 xv[kDepth];
    uint4 av[kDepth][kRB];
    auto load = [&](int s, int64_t k0) {
        const int64_t k = k0 + 8 * g;
        xv[s] = buffer_load16(
            xbuf, k < args.K ? static_cast<uint32_t>((jl * args.K + k) * 2) : kOutOfRange, 0);
#pragma unroll
        for (int i = 0; i < kRB; ++i) {
            const int piece = lane + 64 * i;
            const int64_t row = k0 + piece / (2 * kRB);
            const int col = piece % (2 * kRB) * 8;
            if (args.vector_a) {
                const uint32_t off = col < rank ? static_cast<uint32_t>((row * rank + col) * 2) : kOutOfRange;
                av[s][i] = buffer_load16(abuf, off, 0);  // rows past K: past the buffer
            } else if (args.pair_a) {
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t off = col + 2 * e < rank
                                             ? static_cast<uint32_t>((row * rank + col + 2 * e) * 2)
                                             : kOutOfRange;
                    h[e] = __builtin_amdgcn_raw_buffer_load_b32(abuf, off, 0, 0);
                }
                av[s][i] = make_uint4(h[0], h[1], h[2], h[3]);
            } else {
                uint32_t h[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t off =
                        col + e < rank ? static_cast<uint32_t>((row * rank + col + e) * 2) : kOutOfRange;
                    h[e] = buffer_load2(abuf, off, 0);
                }
                av[s][i] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                                      h[6] | (h[7] << 16));
            }
        }
    };
    f32x4_t acc[kRB];
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) acc[rb] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int s) {
        // Only this wave touches its part of LDS, and its LDS operations
        // complete in order.
#pragma unroll
        for (int i = 0; i < kRB; ++i) {
            *reinterpret_cast<uint4*>(mine + (lane + 64 * i) * 16) = av[s][i];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const bf16x8_t fx = __builtin_bit_cast(bf16x8_t, xv[s]);
        const int rd = (8 * g + (jl >> 2)) * kRowBytes + (jl & 3) * 8;
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) {
            const bf16x8_t fa = concat(lds_read_tr(mine, rd + rb * 32),
                                       lds_read_tr(mine, rd + rb * 32 + 4 * kRowBytes));
            acc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa, fx, acc[rb], 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    constexpr int64_t kStride = kDownWaves * kBK;
    const int64_t start = wave * kBK;
#pragma unroll
    for (int s = 0; s < kDepth; ++s) load(s, start + s * kStride);
    for (int64_t k0 = start; k0 < args.K; k0 += kDepth * kStride) {
#pragma unroll
        for (int s = 0; s < kDepth; ++s) {
            multiply(s);  // past K: zeros
            load(s, k0 + (s + kDepth) * kStride);
        }
    }
    __syncthreads();
    // acc[rb] lane: (x @ a)[row jl][16 rb + 4 g + t].
    float4* sums = reinterpret_cast<float4*>(lds);
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
        sums[(wave * kRB + rb) * 64 + lane] = make_float4(acc[rb][0], acc[rb][1], acc[rb][2], acc[rb][3]);
    }
    __syncthreads();
    for (int e = tid; e < kRB * 64; e += kDownThreads) {
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < kDownWaves; ++w) {
            const float4 p = sums[w * kRB * 64 + e];
            v[0] += p.x;
            v[1] += p.y;
            v[2] += p.z;
            v[3] += p.w;
        }
        const int64_t row = e & 15;
        const int j0 = 16 * (e >> 6) + 4 * ((e >> 4) & 3);
        if (row >= rows_here) continue;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (j0 + t >= rank) continue;
            if (args.xa_out != nullptr) args.xa_out[(m0 + row) * rank + j0 + t] = v[t];
            args.u[(m0 + row) * ext + j0 + t] = static_cast<uint16_t>(f32_to_bf16_bits(v[t]));
        }
    }
    const int pad = ext - rank;
    for (int e = tid; e < static_cast<int>(rows_here) * pad; e += kDownThreads) {
        args.u[(m0 + e / pad) * ext + rank + e % pad] = 0;
    }
}

// ---------------------------------------------------------------------------
// Host.
// ---------------------------------------------------------------------------

size_t align256(size_t bytes) { return (bytes + 255) / 256 * 256; }

int64_t ext_of(int64_t rank) { return ceil_div<int64_t>(rank, kBK) * kBK; }

struct Config {
    int bm;
    int bn;
};

constexpr Config kConfigs[] = {{128, 256}, {128, 128}, {64, 128}};

TilePlan make_plan(int config, int64_t whole, int64_t want, int64_t steps) {
    TilePlan p;
    p.config = config;
    p.whole = static_cast<int>(whole);
    p.slice_steps = static_cast<int>(ceil_div<int64_t>(steps, want));
    p.slices = static_cast<int>(ceil_div<int64_t>(steps, p.slice_steps));
    p.us = 0.0f;
    return p;
}

// What a K-step of one workgroup takes, in microseconds, alone on its CU and
// as its share of a CU that several fill (measured: 2000 x 4096 x 4096 with
// 128x256 tiles, 1000 and 4096 x 4096 x 4096 with 128x128, 100 and 2000 x
// 4096 x 4096 with 64x128), and the fixed part of a launch. Split tiles add
// the write and read of their fp32 partials and the launch that sums them.
constexpr float kStepAlone[] = {0.50f, 0.35f, 0.26f};
constexpr float kStepShared[] = {0.50f, 0.26f, 0.19f};
constexpr float kLaunchUs = 5.0f;
constexpr int kCus = 256;
constexpr int kMinSliceSteps = 4;

/// The fastest of: every tile one workgroup; every tile split; whole rounds
/// of one workgroup per CU and the tiles left over split (333 x 4096 x
/// 11008 r16, whole call: 60.8 us with 256 of the 258 tiles whole and the other
/// two in 8 slices, 71.6 with nothing split, where two CUs work twice as long).
/// (A call comes here twice, for the workspace and for the launch, so it is kept
/// to a few dozen candidates and 32-bit divisions: 0.3 us.)
TilePlan best_plan(int64_t M, int64_t N, int64_t K, int64_t rank) {
    constexpr int kSlices[] = {1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32};
    const int steps = static_cast<int>(ceil_div<int64_t>(K, kBK) + ext_of(rank) / kBK);
    TilePlan best;
    best.us = INFINITY;
    for (int c = 0; c < 3; ++c) {
        const int bm = kConfigs[c].bm;
        const int bn = kConfigs[c].bn;
        const int tiles = static_cast<int>(ceil_div<int64_t>(M, bm) * ceil_div<int64_t>(N, bn));
        const int rounds = tiles / kCus;
        const float partial_us = static_cast<float>(bm * bn) * 8.0f / 3e6f;
        // Every tile split (or none).
        for (const int want : kSlices) {
            if (want > 1 && (want * kMinSliceSteps > steps || tiles * want > 4 * kCus)) break;
            const int groups = tiles * want;
            const int slice_steps = ceil_div(steps, want);
            float us = kLaunchUs + static_cast<float>(ceil_div(groups, kCus) * slice_steps) *
                                       (groups <= kCus ? kStepAlone[c] : kStepShared[c]);
            if (want > 1) us += 4.0f + static_cast<float>(groups) * partial_us;
            if (us < best.us) {
                best = make_plan(c, want == 1 ? tiles : 0, want, steps);
                best.us = us;
            }
        }
        // Whole rounds, and the tiles left over split.
        const int whole = rounds * kCus;
        const int rest = tiles - whole;
        if (whole == 0 || rest == 0) continue;
        const float whole_us = kLaunchUs + static_cast<float>(rounds * steps) *
                                               (rounds == 1 ? kStepAlone[c] : kStepShared[c]);
        for (const int want : kSlices) {
            if (want == 1) continue;
            if (want * kMinSliceSteps > steps || rest * want > 2 * kCus) break;
            const int groups = rest * want;
            const float us = whole_us +
                             static_cast<float>(ceil_div(groups, kCus) * ceil_div(steps, want)) * kStepShared[c] +
                             4.0f + static_cast<float>(groups) * partial_us;
            if (us < best.us) {
                best = make_plan(c, whole, want, steps);
                best.us = us;
            }
        }
    }
    if (rank > 0) best.us += kLaunchUs + static_cast<float>(K * (16 + rank) * 2) / 6e4f;
    return best;
}

template <int kTM, int kTN, int kWM, int kWN, int kStages, int kPerSimd>
void launch_tile(const TileArgs& args, hipStream_t stream) {
    const int groups = args.whole + (args.tiles_m * args.tiles_n - args.whole) * args.slices;
    launch(lora_tile_kernel<kTM, kTN, kWM, kWN, kStages, kPerSimd>, dim3(static_cast<unsigned>(groups)),
           dim3(kWM * kWN * 64), 0, stream, args);
}

cf_status run_plan(const TilePlan& plan, const void* x, const void* w, const void* a, const void* b, void* y,
                   float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank, float scale, void* workspace,
                   hipStream_t stream) {
    const int64_t ext = ext_of(rank);
    uint8_t* p = static_cast<uint8_t*>(workspace);
    TileArgs args;
    args.x = static_cast<const uint16_t*>(x);
    args.w = static_cast<const uint16_t*>(w);
    args.u = reinterpret_cast<uint16_t*>(p);
    args.part = reinterpret_cast<float*>(p + align256(static_cast<size_t>(M * ext) * 2));
    args.b = static_cast<const uint16_t*>(b);
    args.y = static_cast<uint16_t*>(y);
    args.M = M;
    args.N = N;
    args.K = K;
    args.rank = rank;
    args.ext = ext;
    args.ext_steps = static_cast<int>(ext / kBK);
    args.steps = static_cast<int>(ceil_div<int64_t>(K, kBK)) + args.ext_steps;
    args.scale = scale;
    args.whole = plan.whole;
    args.slices = plan.slices;
    args.slice_steps = plan.slice_steps;
    const Config& c = kConfigs[plan.config];
    args.tiles_m = static_cast<int>(ceil_div<int64_t>(M, c.bm));
    args.tiles_n = static_cast<int>(ceil_div<int64_t>(N, c.bn));

    if (rank > 0) {
        DownArgs down;
        down.x = args.x;
        down.a = static_cast<const uint16_t*>(a);
        down.u = const_cast<uint16_t*>(args.u);
        down.xa_out = xa_out;
        down.M = M;
        down.K = K;
        down.rank = static_cast<int>(rank);
        down.ext = static_cast<int>(ext);
        down.vector_a = rank % 8 == 0 && host_aligned(a, 16);
        down.pair_a = rank % 2 == 0 && host_aligned(a, 4);
        const dim3 grid(static_cast<unsigned>(ceil_div<int64_t>(M, 16)));
        if (rank <= 16) {
            launch(lora_down_kernel<1>, grid, dim3(kDownThreads), 0, stream, down);
        } else if (rank <= 32) {
            launch(lora_down_kernel<2>, grid, dim3(kDownThreads), 0, stream, down);
        } else if (rank <= 64) {
            launch(lora_down_kernel<4>, grid, dim3(kDownThreads), 0, stream, down);
        } else {
            launch(lora_down_kernel<8>, grid, dim3(kDownThreads), 0, stream, down);
        }
    }
    if (plan.config == 0) {
        launch_tile<4, 8, 2, 2, 6, 1>(args, stream);
    } else if (plan.config == 1) {
        launch_tile<4, 4, 2, 2, 5, 2>(args, stream);
    } else {
        launch_tile<2, 4, 2, 2, 4, 3>(args, stream);
    }
    const int tiles = args.tiles_m * args.tiles_n - plan.whole;
    if (tiles > 0) {
        launch(lora_tile_sum_kernel,
               dim3(static_cast<unsigned>(c.bm * c.bn / 8 / kDefaultBlockSize), static_cast<unsigned>(tiles)),
               dim3(kDefaultBlockSize), 0, stream, args, c.bm, c.bn);
    }
    return check_launch("launching the tiled bf16 LoRA kernels", stream);
}

}  // namespace

bool lora_tile_shape(int64_t M, int64_t N, int64_t K, int64_t rank) {
    // Buffer offsets are 32-bit with an out-of-range marker at 2^31.
    const int64_t ext = ext_of(rank);
    return M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 && rank >= 0 && rank <= kTileMaxRank &&
           (K + kBK) * N * 2 < (1LL << 31) && 256 * K * 2 < (1LL << 31) && ext * N * 2 < (1LL << 31) &&
           ceil_div<int64_t>(M, 64) * ceil_div<int64_t>(N, 128) < (1LL << 24);
}

bool lora_tile_aligned(const void* x, const void* w, const void* a, const void* b, const void* y, int64_t rank) {
    return host_aligned(x, 16) && host_aligned(w, 16) && host_aligned(y, 16) &&
           (rank == 0 || (host_aligned(a, 2) && host_aligned(b, 16)));
}

TilePlan lora_tile_plan(int64_t M, int64_t N, int64_t K, int64_t rank) { return best_plan(M, N, K, rank); }

size_t lora_tile_workspace_bytes(const TilePlan& p, int64_t M, int64_t N, int64_t rank) {
    const Config& c = kConfigs[p.config];
    const int64_t tiles = ceil_div<int64_t>(M, c.bm) * ceil_div<int64_t>(N, c.bn);
    return align256(static_cast<size_t>(M * ext_of(rank)) * 2) +
           static_cast<size_t>((tiles - p.whole) * p.slices) * c.bm * c.bn * 4;
}

cf_status launch_lora_tile(const TilePlan& plan, const void* x, const void* w, const void* a, const void* b,
                           void* y, float* xa_out, int64_t M, int64_t N, int64_t K, int64_t rank, float scale,
                           void* workspace, hipStream_t stream) {
    return run_plan(plan, x, w, a, b, y, xa_out, M, N, K, rank, scale, workspace, stream);
}

}  // namespace cf
