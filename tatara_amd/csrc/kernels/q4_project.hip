// Affine 4-bit (group 64) projections either side of the attention family: the
// input projections of both layer kinds and the output projection back to the
// hidden width.  Weight format (MLX affine, bits 4): w[n][k] = scale[n][k/64] *
// nibble + bias[n][k/64], eight nibbles to a 32-bit word, low nibble first;
// scales and biases bf16.
//
//   attn_project, attn_project_ms{,_v2}   attention.metal:1-41, 1111-1222
//   gdn_project, gdn_project_ms{,_v2}     gdn.metal:1-47, 380-491
//   gdn_outproj, gdn_outproj_ms{,_v2}     gdn.metal:209-230, 492-551 (the out_projection
//                                         pipeline of both layer kinds, decode_step.cpp:697-733)
//   gdn_project_blk, attn_project_blk, outproj_blk   prefill_dense.metal:120-260
//
// Two evaluations:
//  * rows kernel (up to 16 input rows): the reference's own sequence of operations
//    (q4_dot.metal:9-41 - one lane of 32 per 16 consecutive inputs of a 512 block,
//    power-of-two pre-scaled inputs against masked nibbles, fused chains, the
//    adjacent-pairs tree), so every output is the reference's bit pattern.  A half
//    wave owns an output row; the weights are read once for all input rows.
//  * block product (more rows): both operands are written out once as f16 numbers that
//    hold them exactly, the affine terms as further columns, and multiplied as one
//    matrix product with fp32 sums - the same mathematics in another summation order.
#include <algorithm>
#include <type_traits>

#include "../tt_internal.h"
#include "block_product.h"
#include "lane_sums.h"
#include "rms_row.h"

namespace tt {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

constexpr uint32_t kQ4Block = 512;        // columns one pass of a 32-lane row group covers
constexpr uint32_t kQ4Group = 64;         // columns per {scale, bias}
constexpr uint32_t kQ4BatchRowsMax = 16;  // q4_dot.metal:49
constexpr uint32_t kMaxSegments = 4;

__device__ __forceinline__ float widen(uint16_t h) {
    return __uint_as_float(static_cast<uint32_t>(h) << 16);
}
__device__ __forceinline__ float widen_half(uint32_t word, uint32_t j) {
    return __uint_as_float((j & 1) ? (word & 0xFFFF0000u) : (word << 16));
}
// round to nearest even with subnormal results flushed to signed zero
__device__ __forceinline__ uint16_t store16(float v) {
    uint32_t b = __float_as_uint(v);
    if ((b & 0x7F800000u) == 0) b &= 0x80000000u;
    if ((b & 0x7F800000u) == 0x7F800000u) return static_cast<uint16_t>(b >> 16);
    const uint16_t h = static_cast<uint16_t>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
    return (h & 0x7F80u) ? h : static_cast<uint16_t>(h & 0x8000u);
}

// A projection = up to four weight matrices stacked along the output rows.
struct Q4Projection {
    const uint32_t* words[kMaxSegments];
    const uint16_t* scales[kMaxSegments];
    const uint16_t* biases[kMaxSegments];
    uint32_t first_row[kMaxSegments + 1];  // first output row of each matrix; [segments] = total
    uint32_t segments;
    uint32_t k_size;                       // input width, a multiple of 512
    const uint16_t* input;                 // [rows][input_stride]
    uint16_t* output;                      // [rows][output_stride]
    uint64_t input_stride, output_stride;
    uint32_t rows;                         // input rows in this dispatch
    uint32_t row_tile;                     // input rows one workgroup carries (<= 16)
    // the decode-wave kernel only:
    const uint16_t* norm_weight;           // not null: the input rows go through the RMS norm first
    const uint16_t* residual;              // not null: output = bf16(residual + bf16(projection)),
    uint64_t residual_stride;              //   [rows][residual_stride]; may be the output itself
    bool centred;                          // a block's rows: the exact small nibbles (centred_eight)
};

// The weight matrix that holds output row `n`, with n the same for every lane (matrices have
// multiples of 16 rows, so a workgroup's 8 or 16 rows share one): the operands are picked with
// selects on scalar registers.  Indexing the argument arrays with a per-lane value instead
// turns into vector loads from the argument block - a round trip to memory before the
// first weight can be requested.
struct Q4Matrix {
    const uint32_t* words;
    const uint16_t* scales;
    const uint16_t* biases;
    uint32_t first_row;
};
__device__ __forceinline__ Q4Matrix matrix_of_row(const Q4Projection& p, uint32_t n) {
    Q4Matrix m{p.words[0], p.scales[0], p.biases[0], 0};
#pragma unroll
    for (uint32_t s = 1; s < kMaxSegments; ++s) {
        const bool here = s < p.segments && n >= p.first_row[s];
        m.words = here ? p.words[s] : m.words;
        m.scales = here ? p.scales[s] : m.scales;
        m.biases = here ? p.biases[s] : m.biases;
        m.first_row = here ? p.first_row[s] : m.first_row;
    }
    return m;
}

// grid (ceil(out_rows / 8), ceil(rows / row_tile)) x 256: half wave h of a workgroup
// owns output row 8 * blockIdx.x + h for the tile's input rows.  kBlocks = k_size / 512:
// all of the row's nibbles, scales and biases are requested before the first is used, so
// one row keeps kBlocks loads per lane in flight instead of one.  The tile's x rows are
// the same for all eight output rows: they come in once with coalesced 16-byte loads,
// requested first, and are read back from LDS (every half wave fetching its own copy from
// global memory cost as much as streaming the weights).  LDS layout of one 512-column
// block of a row: the even 16-byte pieces, then the odd ones, so that the 32 lanes of a
// half wave read 512 contiguous bytes twice.  Where the tiles of the workgroups that share
// a compute unit do not fit its LDS (kStaged = false) x is read from global memory: there
// the workgroups per compute unit matter more than the x traffic.
// kEarly: the weights are requested before the first row's pieces are stored (see launch_rows).
// kRowsMax: input rows of a tile this instantiation takes at most.  A single row has one of its own:
// in sixteen rows' code its instructions lie a row's apart, and a kernel of a few us waits for each
// fresh cache line of them (gdn_project / attn_project / gdn_outproj of one row 8.0 / 7.0 / 6.4 ->
// 6.8 / 5.9 / 4.5 us; 31 and 57 KB of code -> 3 and 5).
template <uint32_t kBlocks, bool kStaged, bool kEarly = kStaged, uint32_t kRowsMax = kQ4BatchRowsMax>
__global__ __launch_bounds__(256) void q4_rows_kernel(Q4Projection p) {
    extern __shared__ __align__(16) uint8_t rows_lds[];   // [tile rows][kBlocks][1024]
    constexpr uint32_t kPiecesPerRow = kBlocks * 64;
    const uint32_t lane = threadIdx.x & 31;
    const uint32_t row_base = blockIdx.y * p.row_tile;
    const uint32_t tile_rows = min(p.row_tile, p.rows - row_base);
    auto slot_of = [&](uint32_t piece) {
        const uint32_t r = piece / kPiecesPerRow, c = piece % kPiecesPerRow;
        return (r * kPiecesPerRow + (c & ~63u) + ((c & 63u) >> 1) + (c & 1u) * 32) * 16;
    };
    auto piece_of = [&](uint32_t piece) {
        return *reinterpret_cast<const u32x4*>(
            p.input + static_cast<uint64_t>(row_base + piece / kPiecesPerRow) * p.input_stride +
            piece % kPiecesPerRow * 8);
    };
    // the first row's pieces are stored once the weights have been requested as well, so that
    // the two round trips overlap (a single row, the ordinary case, is all of x)
    constexpr uint32_t kFirst = kPiecesPerRow / 256;
    u32x4 first[kFirst];
    if constexpr (kEarly) {
#pragma unroll
        for (uint32_t j = 0; j < kFirst; ++j) first[j] = piece_of(threadIdx.x + j * 256);
    } else if constexpr (kStaged) {
        for (uint32_t piece = threadIdx.x; piece < tile_rows * kPiecesPerRow; piece += 256) {
            *reinterpret_cast<u32x4*>(rows_lds + slot_of(piece)) = piece_of(piece);
        }
    }
    // rows past the last one compute on the last row and store nothing
    const uint32_t n = min(blockIdx.x * 8 + (threadIdx.x >> 5), p.first_row[p.segments] - 1);
    const bool stores = blockIdx.x * 8 + (threadIdx.x >> 5) < p.first_row[p.segments];
    const Q4Matrix matrix = matrix_of_row(p, min(blockIdx.x * 8, p.first_row[p.segments] - 1));
    const uint32_t local = n - matrix.first_row;
    const uint32_t* words = matrix.words + static_cast<uint64_t>(local) * (kBlocks * 64);
    const uint16_t* scales = matrix.scales + static_cast<uint64_t>(local) * (kBlocks * 8);
    const uint16_t* biases = matrix.biases + static_cast<uint64_t>(local) * (kBlocks * 8);

    u32x2 packed[kBlocks];
    uint16_t scale_bits[kBlocks], bias_bits[kBlocks];
#pragma unroll
    for (uint32_t b = 0; b < kBlocks; ++b) {
        // four 16-bit words = this lane's 16 nibbles of block b
        packed[b] = *reinterpret_cast<const u32x2*>(words + b * 64 + lane * 2);
        scale_bits[b] = scales[b * 8 + (lane >> 2)];
        bias_bits[b] = biases[b * 8 + (lane >> 2)];
    }
    if constexpr (kEarly) {
#pragma unroll
        for (uint32_t j = 0; j < kFirst; ++j) {
            *reinterpret_cast<u32x4*>(rows_lds + slot_of(threadIdx.x + j * 256)) = first[j];
        }
        for (uint32_t piece = kPiecesPerRow + threadIdx.x; kRowsMax > 1 && piece < tile_rows * kPiecesPerRow;
             piece += 256) {
            *reinterpret_cast<u32x4*>(rows_lds + slot_of(piece)) = piece_of(piece);
        }
    }
    if (kStaged) __syncthreads();
    const uint16_t* x0 = p.input + static_cast<uint64_t>(row_base) * p.input_stride + lane * 16;
    float acc[kRowsMax];
#pragma unroll
    for (uint32_t r = 0; r < kRowsMax; ++r) acc[r] = 0.0f;
#pragma unroll
    for (uint32_t b = 0; b < kBlocks; ++b) {
        float wq[16];   // masked, never shifted
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t word = (i & 1) ? (packed[b][i >> 1] >> 16) : (packed[b][i >> 1] & 0xFFFFu);
            wq[i * 4] = static_cast<float>(word & 0x000Fu);
            wq[i * 4 + 1] = static_cast<float>(word & 0x00F0u);
            wq[i * 4 + 2] = static_cast<float>(word & 0x0F00u);
            wq[i * 4 + 3] = static_cast<float>(word & 0xF000u);
        }
        const float scale = widen(scale_bits[b]);
        const float bias = widen(bias_bits[b]);
        const uint8_t* xk = rows_lds + b * 1024 + lane * 16;
#pragma unroll
        for (uint32_t r = 0; r < kRowsMax; ++r) {
            if (kRowsMax == 1 || r < tile_rows) {
                u32x4 lo, hi;
                if (kStaged) {
                    lo = *reinterpret_cast<const u32x4*>(xk + r * (kPiecesPerRow * 16));
                    hi = *reinterpret_cast<const u32x4*>(xk + r * (kPiecesPerRow * 16) + 512);
                } else {
                    const u32x4* xr =
                        reinterpret_cast<const u32x4*>(x0 + b * kQ4Block + r * p.input_stride);
                    lo = xr[0];
                    hi = xr[1];
                }
                float sum = 0.0f, quant = 0.0f;
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    const uint32_t w0 = i < 2 ? lo[2 * i] : hi[2 * i - 4];
                    const uint32_t w1 = i < 2 ? lo[2 * i + 1] : hi[2 * i - 3];
                    const float a0 = widen_half(w0, 0), a1 = widen_half(w0, 1);
                    const float a2 = widen_half(w1, 0), a3 = widen_half(w1, 1);
                    sum += ((a0 + a1) + a2) + a3;
                    quant = fmaf(a0, wq[i * 4], quant);
                    quant = fmaf(a1 * 0.0625f, wq[i * 4 + 1], quant);
                    quant = fmaf(a2 * 0.00390625f, wq[i * 4 + 2], quant);
                    quant = fmaf(a3 * 0.000244140625f, wq[i * 4 + 3], quant);
                }
                acc[r] = fmaf(sum, bias, fmaf(scale, quant, acc[r]));
            }
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < kRowsMax; ++r) {
        if (kRowsMax == 1 || r < tile_rows) {
            const float total = half_wave_sum(acc[r]);
            if (lane == 0 && stores) {
                p.output[static_cast<uint64_t>(row_base + r) * p.output_stride + n] = store16(total);
            }
        }
    }
}

constexpr uint32_t kRowsStagedBytes = 128 * 1024;   // of the 160 KB of a compute unit

// 0 when the width has no instantiation
int32_t launch_rows(const Q4Projection& p, hipStream_t stream) {
    const uint32_t out_rows = p.first_row[p.segments];
    const dim3 grid((out_rows + 7) / 8, (p.rows + p.row_tile - 1) / p.row_tile);
    const uint32_t tile_rows = min(p.rows, p.row_tile);
    // as many workgroups as the grid puts on a compute unit (up to eight) must still fit
    const uint32_t resident = min(8u, (grid.x * grid.y + 255) / 256);
    const auto staged = [&](uint32_t row_bytes) {
        return tile_rows * row_bytes * resident <= kRowsStagedBytes;
    };
    switch (p.k_size / kQ4Block) {
    // LDS: the tile's x rows where they fit kRowsStagedBytes.  Requesting the weights before the
    // first row is stored hides a round trip from a single row, which is all of x (gdn_project
    // 7.2 -> 7.1 us, outproj 6.0 -> 5.8, and up to 13 rows of it by 2 to 4 %); the in-projections
    // of 2 .. 5 rows were 1 to 2 % slower so, 16 rows of outproj 3 %.
    case 4:
        if (staged(4096) && tile_rows > 1) {
            hipLaunchKernelGGL((q4_rows_kernel<4, true, false>), grid, dim3(256), tile_rows * 4096, stream, p);
        } else if (staged(4096)) {
            hipLaunchKernelGGL((q4_rows_kernel<4, true, true, 1>), grid, dim3(256), tile_rows * 4096, stream, p);
        } else {
            hipLaunchKernelGGL((q4_rows_kernel<4, false>), grid, dim3(256), 0, stream, p);
        }
        break;
    case 8:
        if (staged(8192) && tile_rows > 13) {
            hipLaunchKernelGGL((q4_rows_kernel<8, true, false>), grid, dim3(256), tile_rows * 8192, stream, p);
        } else if (staged(8192) && tile_rows == 1) {
            hipLaunchKernelGGL((q4_rows_kernel<8, true, true, 1>), grid, dim3(256), 8192, stream, p);
        } else if (staged(8192)) {
            hipLaunchKernelGGL((q4_rows_kernel<8, true>), grid, dim3(256), tile_rows * 8192, stream, p);
        } else {
            hipLaunchKernelGGL((q4_rows_kernel<8, false>), grid, dim3(256), 0, stream, p);
        }
        break;
    default: return TT_CMD_INVALID_DISPATCH_EXTENT;
    }
    return TT_OK;
}

// ----------------------------------------------------------- block product ---
//
// out[m][n] = sum_k x[m][k] (nibble - 8) scale[n][g] + sum_g (bias + 8 scale)[n][g] xs[m][g],
// xs[m][g] = sum of x over the 64 columns of group g.
//
// A scale has 8 significant bits and nibble - 8 (-8 .. 7) three or a power of two, so their
// product has at most 11: an f16 number, exactly.  So is x, of 8 bits.  Both are brought into
// f16's range by a power of two per row (an output row's largest of 8 |scale| and |bias| below
// 2^15, an input row's largest |x| below 2^9, so that its group sums stay below 2^15): an x that
// lies so far below the row's largest that f16 rounds it is off by 2^-33 of that one at most, a
// weight by 2^-39.  The affine terms are four further columns a group, {bias, 8 scale, bias,
// 8 scale} against {hi, hi, lo, lo} of the group sum in two f16 parts, 2^-23 of the sum at most
// from it: the largest of these roundings, about one of the fp32 sums' own.  One pass writes both
// operands so into the queue's workspace; the product is then a plain one (block_product.h) and the
// powers of two leave with the result.
//
// Why not unpack inside the product: a scale per 64 columns costs a product of its own from a
// zero accumulator and 64 fused adds a lane for every 32 products, and the unpacking is
// repeated for every 256 rows.  That kernel reached 28 % of the matrix unit's rate (gdn_project
// at 16384 / 2048 / 777 / 100 rows: 1178 / 189 / 103 / 38 us, outproj 359 / 65 / 46 / 36 us);
// this pass is bound by its writes (4.4 bytes per weight byte read).
constexpr uint32_t kAffineColumns = 4;               // per group
__host__ __device__ constexpr uint32_t unfolded_columns(uint32_t k_size) {
    return k_size + k_size / kQ4Group * kAffineColumns;
}
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;

struct Unfold {
    _Float16* weights;         // [out_rows][unfolded_columns]
    int32_t* weight_exponents; // [out_rows]: the row's values times 2^-exponent were written
    _Float16* rows;            // [x_rows][unfolded_columns]
    int32_t* row_exponents;    // [x_rows]
    uint32_t weight_rows;      // 0: the weights are there already
    uint32_t first_weight;     // the output row that row 0 of `weights` is
    uint32_t first_row, x_rows;
    bool short_rows;           // the rows' pieces in q4_short_kernel's order (unfolded_piece)
};

// the power of two that brings `largest` (a magnitude) to [2^(below - 1), 2^below)
__device__ __forceinline__ int32_t shift_below(float largest, int32_t below) {
    const int32_t field = static_cast<int32_t>(__float_as_uint(largest) >> 23);   // no sign
    return field == 0 ? (largest == 0.0f ? 0 : below + 125) : below + 126 - field;
}

// The columns of an unfolded row stand in an order of their own, the same in both operands (a
// product does not ask for one).  Of eight columns, in pairs: 0 and 4, 1 and 5, 2 and 6, 3 and 7 -
// a word's nibbles come apart so with one shift and one mask a pair.  For q4_short_kernel the rows
// of x also have the pieces of eight columns of every four units in the order 0, 4, 8 .., 1, 5,
// 9 ..: a unit then takes one word of every 16 bytes of a weight row, so that it can load whole 16
// bytes.  (Written in that order for the block product as well, both operands took 1 to
// 2 us longer at 2048 rows: a store's lanes no longer fall together.)
template <uint32_t kBlocks>
__device__ __forceinline__ uint32_t unfolded_piece(uint32_t piece) {
    constexpr uint32_t kSpan = kBlocks == 4 ? 64 : 128;   // pieces
    const uint32_t within = piece % kSpan;
    return piece - within + within % 4 * (kSpan / 4) + within / 4;
}
// Nibbles i and i + 4 of `word`, less 8, times the steps: the nibbles in the lowest four bits of f16
// 1024.0, or in the four above of 64.0, where they count units; less 1032 or 72 they are n - 8, exactly.
// Eight weights are a shift, four and-ors, four sums and four products.  (16 + n from one position and a
// fused multiply-add are 12 instructions instead of 13, gdn_project of 17 / 100 / 256 rows 12.65 / 20.2 / 36.4 us
// instead of 12.8 / 20.4 / 36.6, but the 24 steps it takes off must fit f16: the row's largest below 2^14,
// and a bit less of the small steps beside it.)
__device__ __forceinline__ uint32_t unfold_pair(uint32_t word, uint32_t i, f16x2 steps) {
    const bool lowest = i % 2 == 0;
    uint32_t base = lowest ? 0x64006400u : 0x54005400u;
    asm("" : "+v"(base));   // kept in a register: one v_and_or_b32 instead of two instructions
    const uint32_t pair = ((i < 2 ? word : word >> 8) & (lowest ? 0x000F000Fu : 0x00F000F0u)) | base;
    const _Float16 less = static_cast<_Float16>(lowest ? 1032.0f : 72.0f);
    return __builtin_bit_cast(uint32_t, (__builtin_bit_cast(f16x2, pair) - f16x2{less, less}) * steps);
}

// the largest of four values, one to a row of 16 lanes
__device__ __forceinline__ float wave_largest_of_rows(float v) {
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F)));   // lane ^ 16
    return fmaxf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)),
                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32)));
}

// grid ceil((weight_rows + x_rows) / 4) x 256: a wave per row.  Lanes meet through DPP, not through
// the LDS crossbar: with that, up to 30 round trips a row, 100 rows of 2048 / 4096 columns took 3.6 /
// 4.8 us instead of 3.3 / 4.2.
template <uint32_t kBlocks>   // k_size / 512
__global__ __launch_bounds__(256) void q4_unfold_kernel(Q4Projection p, Unfold u) {
    constexpr uint32_t kColumns = unfolded_columns(kBlocks * kQ4Block);
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row < u.weight_rows) {
        const Q4Matrix matrix = matrix_of_row(p, u.first_weight + row);
        const uint64_t local = u.first_weight + row - matrix.first_row;
        const uint32_t* words = matrix.words + local * (kBlocks * 64);
        const uint16_t* scales = matrix.scales + local * (kBlocks * 8);
        const uint16_t* biases = matrix.biases + local * (kBlocks * 8);
        uint32_t packed[kBlocks];
        float scale[kBlocks], bias[kBlocks];
        float largest = 0.0f;
#pragma unroll
        for (uint32_t b = 0; b < kBlocks; ++b) {
            // word `lane` of the block's 64: columns 8 lane .. 8 lane + 7, group lane / 8
            packed[b] = words[b * 64 + lane];
            scale[b] = widen(scales[b * 8 + (lane >> 3)]);
            bias[b] = widen(biases[b * 8 + (lane >> 3)]);
            largest = fmaxf(largest, fmaxf(8.0f * fabsf(scale[b]), fabsf(bias[b])));
        }
        // over the lanes of other groups of eight
        largest = fmaxf(largest, lane_dpp<0x128>(largest));   // row_ror:8
        largest = wave_largest_of_rows(largest);
        const int32_t shift = shift_below(largest, 15);
        if (lane == 0) u.weight_exponents[row] = -shift;
        _Float16* out = u.weights + static_cast<uint64_t>(row) * kColumns;
#pragma unroll
        for (uint32_t b = 0; b < kBlocks; ++b) {
            const _Float16 step = static_cast<_Float16>(ldexpf(scale[b], shift));
            const f16x2 steps = f16x2{step, step};
            u32x4 eight;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                eight[i] = unfold_pair(packed[b], i, steps);
            }
            *reinterpret_cast<u32x4*>(out + b * kQ4Block + lane * 8) = eight;
            if ((lane & 7) == 0) {
                const _Float16 first = static_cast<_Float16>(ldexpf(bias[b], shift));
                const _Float16 second = static_cast<_Float16>(ldexpf(scale[b], shift + 3));
                *reinterpret_cast<f16x4*>(out + kBlocks * kQ4Block +
                                          (b * 8 + (lane >> 3)) * kAffineColumns) =
                    f16x4{first, second, first, second};
            }
        }
    } else if (row - u.weight_rows < u.x_rows) {
        const uint32_t at = row - u.weight_rows;
        const uint16_t* x = p.input + static_cast<uint64_t>(u.first_row + at) * p.input_stride + lane * 8;
        u32x4 raw[kBlocks];
        uint32_t largest = 0;   // bf16 magnitudes order as their bits
#pragma unroll
        for (uint32_t b = 0; b < kBlocks; ++b) {
            raw[b] = *reinterpret_cast<const u32x4*>(x + b * kQ4Block);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                largest = max(largest, max(raw[b][i] & 0x7FFFu, (raw[b][i] >> 16) & 0x7FFFu));
            }
        }
        float magnitude = __uint_as_float(largest << 16);
        magnitude = fmaxf(magnitude, lane_dpp<0xB1>(magnitude));    // the steps of row_sum
        magnitude = fmaxf(magnitude, lane_dpp<0x4E>(magnitude));
        magnitude = fmaxf(magnitude, lane_dpp<0x141>(magnitude));
        magnitude = fmaxf(magnitude, lane_dpp<0x140>(magnitude));
        const int32_t shift = shift_below(wave_largest_of_rows(magnitude), 9);
        if (lane == 0) u.row_exponents[at] = -shift;
        _Float16* out = u.rows + static_cast<uint64_t>(at) * kColumns;
#pragma unroll
        for (uint32_t b = 0; b < kBlocks; ++b) {
            float value[8];
            float sum = 0.0f;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                value[2 * i] = ldexpf(widen_half(raw[b][i], 0), shift);
                value[2 * i + 1] = ldexpf(widen_half(raw[b][i], 1), shift);
                sum += value[2 * i] + value[2 * i + 1];
            }
            u32x4 eight;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                eight[i] = __builtin_bit_cast(uint32_t, f16x2{static_cast<_Float16>(value[i]),
                                                              static_cast<_Float16>(value[i + 4])});
            }
            const uint32_t piece = b * 64 + lane;
            *reinterpret_cast<u32x4*>(out + (u.short_rows ? unfolded_piece<kBlocks>(piece) : piece) * 8) = eight;
            sum += lane_dpp<0xB1>(sum);
            sum += lane_dpp<0x4E>(sum);
            sum += lane_dpp<0x141>(sum);
            if ((lane & 7) == 0) {
                const _Float16 high = static_cast<_Float16>(sum);
                const _Float16 low = static_cast<_Float16>(sum - static_cast<float>(high));
                *reinterpret_cast<f16x4*>(out + kBlocks * kQ4Block +
                                          (b * 8 + (lane >> 3)) * kAffineColumns) =
                    f16x4{high, high, low, low};
            }
        }
    }
}

template <typename Product>
__global__ __launch_bounds__(Product::kThreads) void q4_product_kernel(Unfold u, uint16_t* output,
                                                                      uint64_t output_stride,
                                                                      uint32_t columns,
                                                                      uint32_t out_rows, uint32_t runs) {
    const bool wide = ((reinterpret_cast<uintptr_t>(output) | (output_stride * 2)) & 7) == 0;
    Product::run(u.rows, u.weights, u.x_rows, columns, out_rows, runs,
                 [&](uint32_t m, uint32_t n, typename Product::Sums sums) {
                     typedef __attribute__((ext_vector_type(4))) int32_t Exponents;
                     const int32_t row_exponent = u.row_exponents[m];
                     const Exponents exponents = *reinterpret_cast<const Exponents*>(u.weight_exponents + n);
#pragma unroll
                     for (uint32_t j = 0; j < 4; ++j) {
                         sums[j] = ldexpf(sums[j], row_exponent + exponents[j]);
                     }
                     block_store(output + static_cast<uint64_t>(u.first_row + m) * output_stride, n,
                                 out_rows, wide, sums);
                 });
}

// ------------------------------------------------------------ short blocks ---
//
// The same product for blocks of few rows, with the weights unpacked where they are multiplied:
// only the rows of x are unfolded.  A workgroup of eight waves owns 32 kNWaves outputs and 16 kTm
// rows and walks the columns in units of 32 for each of its 8 / kNWaves waves along them; a wave multiplies 32
// outputs with all the rows over its 32 columns of every unit (as many partial sums an output, added
// up at the end), which lets every fragment of x feed two products and every unpacked fragment of
// weights kTm.  A lane's operand of one product is the eight nibbles of one word, and a lane's words of
// four units are 16 bytes of a weight row (unfolded_piece): everything a workgroup needs of the
// weights is requested at its start.  x comes through LDS as in block_product.h, a ring of units.
// Over 2048 columns two waves share the columns' work (as many workgroups as compute units, nearly);
// the 2048 outputs over 4096 columns are cut finer, in as many units of twice the columns.
template <uint32_t kTm_, uint32_t kBlocks_>   // kBlocks: k_size / 512
struct ShortProduct {
    static constexpr uint32_t kTm = kTm_, kBlocks = kBlocks_;
    static constexpr uint32_t kNWaves = kBlocks == 4 ? 2 : 1, kKWaves = 8 / kNWaves;
    static constexpr uint32_t kTileM = 16 * kTm, kTileN = 32 * kNWaves;
    static constexpr uint32_t kThreads = 512;
    static constexpr uint32_t kUnitColumns = 32 * kKWaves, kRowBytes = 2 * kUnitColumns;
    static constexpr uint32_t kUnitBytes = kTileM * kRowBytes;
    static constexpr uint32_t kRing = kBlocks == 4 || kTm == 2 ? 4 : kTm == 4 ? 4 : kTm == 6 ? 3 : 2;
    static constexpr uint32_t kExponentBytes = kTileN * 4;
    static constexpr uint32_t kLdsBytes = kRing * kUnitBytes + kExponentBytes;
    static constexpr uint32_t kTransfers = kUnitBytes / 1024 / 8;   // of a wave and unit
    static_assert(kTm % 2 == 0 && kLdsBytes <= 160 * 1024);
    // the partial sums of all eight waves take the ring's place
    static_assert(8 * kTm * 2 * 1024 <= kRing * kUnitBytes);
    // Waves to a SIMD: 128 registers each where that costs no spills, for a second workgroup where two fit the LDS
    // (64 rows over 4096 columns fill it alone, and are faster so all the same: outproj_blk of 129 / 256 rows 18.0 /
    // 19.8 us, with 256 registers 18.5 / 20.4).
    static constexpr uint32_t kWavesPerSimd = kTm <= 4 ? 4 : 2;
};

typedef u32x4 u32x4_pairs __attribute__((aligned(4)));   // scales and biases: see check_block_operands

// grid (out_rows / kTileN, ceil(x_rows / kTileM))
template <typename Product>
__global__ __launch_bounds__(512, Product::kWavesPerSimd) void q4_short_kernel(Q4Projection p, Unfold u) {
    constexpr uint32_t kTm = Product::kTm, kBlocks = Product::kBlocks;
    constexpr uint32_t kGroups = kBlocks * 8;
    constexpr uint32_t kUnitColumns = Product::kUnitColumns;
    constexpr uint32_t kAffineUnits = kGroups * kAffineColumns / kUnitColumns;
    constexpr uint32_t kSpans = kBlocks * kQ4Block / kUnitColumns / 4;   // of four units, 16 bytes a lane
    static_assert(kAffineUnits == 1 && kSpans == 4);
    constexpr uint32_t kUnits = kSpans * 4 + kAffineUnits;
    constexpr uint32_t kRowBytes = unfolded_columns(kBlocks * kQ4Block) * 2;
    constexpr uint32_t kTransfers = Product::kTransfers;
    constexpr uint32_t kRing = Product::kRing;
    constexpr uint32_t kPieces = kUnitColumns / 8;   // of a unit's row
    typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
    extern __shared__ __align__(16) uint8_t short_lds[];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t i16 = lane & 15, g = lane >> 4;
    const uint32_t nw = wave % Product::kNWaves, kh = wave / Product::kNWaves;
    const uint32_t first_out = blockIdx.x * Product::kTileN;
    const uint32_t m0 = blockIdx.y * Product::kTileM;
    const uint32_t lds_base = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)short_lds));

    // In a row of the ring, one row's unit, the 16-byte piece c sits in slot c ^ (row & 15), so
    // that the sixteen rows of a fragment read fall on different banks.
    const uint8_t* x = reinterpret_cast<const uint8_t*>(u.rows);
    uint32_t x_offset[kTransfers];
#pragma unroll
    for (uint32_t t = 0; t < kTransfers; ++t) {
        const uint32_t row = (wave * kTransfers + t) * (64 / kPieces) + lane / kPieces;
        x_offset[t] = min(m0 + row, u.x_rows - 1) * kRowBytes + (lane % kPieces ^ (row & 15)) * 16;
    }
    const auto request = [&](uint32_t unit) __attribute__((always_inline)) {
        // the affine columns first: their operand is not kept
        const uint32_t column = unit < kAffineUnits ? kBlocks * kQ4Block : (unit - kAffineUnits) * kUnitColumns;
#pragma unroll
        for (uint32_t t = 0; t < kTransfers; ++t) {
            block_transfer(x + column * 2, x_offset[t],
                           lds_base + unit % kRing * Product::kUnitBytes +
                               (wave * kTransfers + t) * 1024);
        }
    };

    // Scales and biases: of all the row's groups for its exponent (a quarter by each g), those of the
    // affine operand.
    u32x4 words[2][kSpans];
    u32x4 scale_bits[2][kBlocks / 4], bias_bits[2][kBlocks / 4];
    uint32_t affine_scale[2], affine_bias[2];
    const uint32_t* word_rows[2];
#pragma unroll
    for (uint32_t tn = 0; tn < 2; ++tn) {
        const uint32_t n = first_out + nw * 32 + tn * 16;   // every matrix has a multiple of 16 rows
        const Q4Matrix matrix = matrix_of_row(p, n);
        const uint64_t local = n + i16 - matrix.first_row;
        word_rows[tn] = matrix.words + local * (kBlocks * 64) + (4 * kh + g) * 4;
        const uint16_t* scales = matrix.scales + local * kGroups;
        const uint16_t* biases = matrix.biases + local * kGroups;
#pragma unroll
        for (uint32_t i = 0; i < kBlocks / 4; ++i) {
            scale_bits[tn][i] = *reinterpret_cast<const u32x4_pairs*>(scales + g * (kGroups / 4) + i * 8);
            bias_bits[tn][i] = *reinterpret_cast<const u32x4_pairs*>(biases + g * (kGroups / 4) + i * 8);
        }
        affine_scale[tn] = *reinterpret_cast<const uint32_t*>(scales + kh * 8 + g * 2);
        affine_bias[tn] = *reinterpret_cast<const uint32_t*>(biases + kh * 8 + g * 2);
    }
#pragma unroll
    for (uint32_t unit = 0; unit < kRing - 1; ++unit) request(unit);
#pragma unroll
    for (uint32_t span = 0; span < kSpans; ++span) {
#pragma unroll
        for (uint32_t tn = 0; tn < 2; ++tn) {
            words[tn][span] = *reinterpret_cast<const u32x4*>(word_rows[tn] + span * (kUnitColumns / 2));
        }
    }

    int32_t shift[2];
#pragma unroll
    for (uint32_t tn = 0; tn < 2; ++tn) {
        float largest = 0.0f;
#pragma unroll
        for (uint32_t i = 0; i < kBlocks; ++i) {
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                largest = fmaxf(largest, 8.0f * fabsf(widen_half(scale_bits[tn][i >> 2][i & 3], j)));
                largest = fmaxf(largest, fabsf(widen_half(bias_bits[tn][i >> 2][i & 3], j)));
            }
        }
        largest = fmaxf(largest, __shfl_xor(largest, 16));
        largest = fmaxf(largest, __shfl_xor(largest, 32));
        shift[tn] = shift_below(largest, 15);
        if (kh == 0 && g == 0) {
            *reinterpret_cast<int32_t*>(short_lds + kRing * Product::kUnitBytes +
                                        (nw * 32 + tn * 16 + i16) * 4) = -shift[tn];
        }
    }
    // the step of span s: of its groups the one of number 2 kh + (g >> 1), all held by lane group s
    f16x2 steps[2][kSpans];
#pragma unroll
    for (uint32_t tn = 0; tn < 2; ++tn) {
        const u32x4 held = scale_bits[tn][kBlocks == 4 ? 0 : kh >> 2];
        const uint32_t at = kh & 3;
        const uint32_t mine = at == 0 ? held[0] : at == 1 ? held[1] : at == 2 ? held[2] : held[3];
#pragma unroll
        for (uint32_t span = 0; span < kSpans; ++span) {
            const uint32_t pair =
                static_cast<uint32_t>(__shfl(static_cast<int>(mine), span * 16 + i16));
            const _Float16 step = static_cast<_Float16>(ldexpf(widen_half(pair, g >> 1), shift[tn]));
            steps[tn][span] = f16x2{step, step};
        }
    }

    f32x4 acc[2][kTm];
#pragma unroll
    for (uint32_t tn = 0; tn < 2; ++tn) {
#pragma unroll
        for (uint32_t tm = 0; tm < kTm; ++tm) acc[tn][tm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const uint32_t fragment = i16 * Product::kRowBytes + ((4 * kh + g) ^ i16) * 16;
    const auto step = [&](uint32_t unit, const f16x8 (&w)[2]) __attribute__((always_inline)) {
        const uint8_t* at = short_lds + unit % kRing * Product::kUnitBytes + fragment;
#pragma unroll
        for (uint32_t tm = 0; tm < kTm; ++tm) {
            const f16x8 rows = *reinterpret_cast<const f16x8*>(at + tm * 16 * Product::kRowBytes);
#pragma unroll
            for (uint32_t tn = 0; tn < 2; ++tn) {
                acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[tn], rows, acc[tn][tm], 0, 0, 0);
            }
        }
    };
    // Unit `unit` has landed, mine, then everybody's, and nobody reads the one before it: the unit
    // after the last requested takes its place.  (At most kRing - 2 units were requested after
    // `unit`; whatever else is in flight only makes the wait longer.)
    const auto arrive = [&](uint32_t unit) __attribute__((always_inline)) {
        if (unit + kRing - 1 <= kUnits) {
            __builtin_amdgcn_s_waitcnt(block_vmcnt((kRing - 2) * kTransfers));
        } else {
            __builtin_amdgcn_s_waitcnt(block_vmcnt(0));
        }
        __syncthreads();
        if (unit + kRing - 1 < kUnits) request(unit + kRing - 1);
    };
    const auto affine = [&](f16x8 (&w)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t tn = 0; tn < 2; ++tn) {
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                const _Float16 first =
                    static_cast<_Float16>(ldexpf(widen_half(affine_bias[tn], j), shift[tn]));
                const _Float16 second =
                    static_cast<_Float16>(ldexpf(widen_half(affine_scale[tn], j), shift[tn] + 3));
                w[tn][4 * j] = w[tn][4 * j + 2] = first;
                w[tn][4 * j + 1] = w[tn][4 * j + 3] = second;
            }
        }
    };
    // the operand of a unit: affine columns, or a word of the span it is of
    const auto unpack = [&](uint32_t unit, f16x8 (&w)[2]) __attribute__((always_inline)) {
        if (unit < kAffineUnits) {
            affine(w);
            return;
        }
        const uint32_t span = (unit - kAffineUnits) / 4, j = (unit - kAffineUnits) % 4;
#pragma unroll
        for (uint32_t tn = 0; tn < 2; ++tn) {
            u32x4 eight;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                eight[i] = unfold_pair(words[tn][span][j], i, steps[tn][span]);
            }
            w[tn] = __builtin_bit_cast(f16x8, eight);
        }
    };
    f16x8 w[2][2];
    unpack(0, w[0]);
#pragma unroll
    for (uint32_t unit = 0; unit < kUnits; ++unit) {
        arrive(unit);
        if (unit + 1 < kUnits) unpack(unit + 1, w[(unit + 1) & 1]);   // beside the products
        step(unit, w[unit & 1]);
    }

    // the partial sums of every output, in the ring's place: [kh][nw][tm][tn][lane]
    __syncthreads();
    f32x4* partial = reinterpret_cast<f32x4*>(short_lds) + lane;
    const auto place = [&](uint32_t part, uint32_t tm, uint32_t tn) {
        return (((part * Product::kNWaves + nw) * kTm + tm) * 2 + tn) * 64;
    };
#pragma unroll
    for (uint32_t tm = 0; tm < kTm; ++tm) {
#pragma unroll
        for (uint32_t tn = 0; tn < 2; ++tn) partial[place(kh, tm, tn)] = acc[tn][tm];
    }
    __syncthreads();
    const bool wide = ((reinterpret_cast<uintptr_t>(p.output) | (p.output_stride * 2)) & 7) == 0;
    const uint32_t out_rows = p.first_row[p.segments];
    // of the 2 kTm fragments of its outputs a wave finishes every kKWaves-th
#pragma unroll
    for (uint32_t f = 0; f < 2 * kTm; f += Product::kKWaves) {
        if (f + kh >= 2 * kTm) break;
        const uint32_t tm = (f + kh) >> 1, tn = (f + kh) & 1;
        f32x4 sums = partial[place(0, tm, tn)];
#pragma unroll
        for (uint32_t part = 1; part < Product::kKWaves; ++part) sums += partial[place(part, tm, tn)];
        const uint32_t m = m0 + tm * 16 + i16;
        if (m >= u.x_rows) continue;
        typedef __attribute__((ext_vector_type(4))) int32_t Exponents;
        const uint32_t column = nw * 32 + tn * 16 + g * 4;
        const Exponents exponents = *reinterpret_cast<const Exponents*>(
            short_lds + kRing * Product::kUnitBytes + column * 4);
        const int32_t row_exponent = u.row_exponents[m];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) sums[j] = ldexpf(sums[j], row_exponent + exponents[j]);
        block_store(p.output + static_cast<uint64_t>(u.first_row + m) * p.output_stride, first_out + column,
                    out_rows, wide, sums);
    }
}

// What the pass assumes of its operands beyond their sizes: 16-byte pieces of x (and of the
// nibble words and 4-byte pairs of scales and biases, which every block call has been held to).
int32_t check_block_operands(const Q4Projection& p) {
    uintptr_t wide = reinterpret_cast<uintptr_t>(p.input), narrow = 0;
    for (uint32_t s = 0; s < p.segments; ++s) {
        wide |= reinterpret_cast<uintptr_t>(p.words[s]);
        narrow |= reinterpret_cast<uintptr_t>(p.scales[s]) | reinterpret_cast<uintptr_t>(p.biases[s]);
    }
    if ((wide & 15) != 0 || (narrow & 3) != 0 || ((p.input_stride * 2) & 15) != 0) {
        return TT_CMD_INVALID_BUFFER_OFFSET;
    }
    if (static_cast<uint64_t>(p.rows) * p.input_stride * 2 >= (1ull << 32)) {
        return TT_CMD_INVALID_DISPATCH_EXTENT;
    }
    return TT_OK;
}

// The workspace of a block: the unfolded weights of the largest projection and the unfolded
// rows of 16384 tokens at the hidden width (8192 at the attention width); a longer block goes
// through in slices of that many rows.  In a smaller workspace (device memory was short when the
// queue was made) the weights go through in slices as well, half of it for either.
constexpr uint64_t kUnfoldedWeightBytes =
    static_cast<uint64_t>(kGdnProjectionRows) * unfolded_columns(kHidden) * 2;
constexpr uint64_t kUnfoldedRowBytes = 16384ull * unfolded_columns(kHidden) * 2;
constexpr uint64_t kWeightExponentBytes = (kGdnProjectionRows * 4 + 255) / 256 * 256;
constexpr uint64_t kRowExponentBytes = 16384ull * 4;
constexpr uint64_t kUnfoldWorkspaceBytes =
    kUnfoldedWeightBytes + kUnfoldedRowBytes + kWeightExponentBytes + kRowExponentBytes;
static_assert(kUnfoldedWeightBytes % 256 == 0 && kUnfoldedRowBytes % 256 == 0, "aligned parts");
static_assert(static_cast<uint64_t>(kHidden) * unfolded_columns(kGdnValueValues) <=
                  static_cast<uint64_t>(kGdnProjectionRows) * unfolded_columns(kHidden),
              "the output projection's weights fit as well");

// The row tile of a short block with the shortest estimate, and that estimate: ns of a launch, a
// fixed part and one per workgroup of a compute unit, fitted to 17 .. 777 rows (128 rows over 4096 columns, 23 us
// a workgroup, are never the shortest).  gdn_project_blk / attn_project_blk / outproj_blk with unfolding,
// weights written out and unpacked in the product:
//   17 rows   29.5 / 26.4 / 25.0 and 12.8 / 12.7 / 14.7 us     384 rows  48.0 / 37.0 / 27.4 and 44.3 / 36.5 / 25.4
//   100 rows  32.3 / 30.6 / 25.9 and 20.5 / 20.0 / 15.4        400 rows  47.8 / 41.9 / 27.2 and 50.0 / 36.3 / 30.4
//   256 rows  38.1 / 35.1 / 25.9 and 36.2 / 28.9 / 20.1        448 rows  47.8 / 42.2 / 27.1 and 50.5 / 36.8 / 30.9
//   320 rows  44.3 / 36.6 / 27.8 and 37.2 / 29.4 / 24.7        512 rows  48.9 / 45.6 / 27.1 and 57.1 / 43.7 / 31.3
// What bounds it: at 100 rows of gdn_project the x rows' unfolding and two launches 5.5 us, the weights'
// arrival 3, the products and the barrier of each unit 7 (4 of them on the matrix unit), the partial sums 2.
struct ShortChoice {
    uint32_t tm;
    uint64_t ns;
};
inline ShortChoice choose_short_tile(uint32_t rows, uint32_t k_size, uint32_t out_rows, uint32_t compute_units) {
    struct Cost {
        uint32_t tm, fixed[2], each[2];   // over 2048 and 4096 columns
    };
    static constexpr Cost kCosts[] = {
        {2, {3200, 1500}, {5200, 8500}},
        {4, {3500, 0}, {7000, 13500}},
        {6, {500, 0}, {12600, 18000}},
        {8, {1800, 0}, {14200, 0}},
    };
    const uint32_t deep = k_size > kHidden ? 1 : 0;
    ShortChoice best{0, ~0ull};
    for (const Cost& c : kCosts) {
        if (c.each[deep] == 0) continue;
        const uint64_t groups = static_cast<uint64_t>((rows + 16 * c.tm - 1) / (16 * c.tm)) * (out_rows / (deep ? 32 : 64));
        const uint64_t ns = c.fixed[deep] + (groups + compute_units - 1) / compute_units * c.each[deep];
        if (ns < best.ns) best = ShortChoice{c.tm, ns};
    }
    return best;
}
// The tile of a short block if its weights are unpacked in the product, 0 if they are written out first: what that
// takes, 5 bytes a ns, is spared where each row tile unpacks its own.  Estimates of products that do not
// fill their rounds are too long, those of one round too short (30.4 us with the writing measured as 38 with
// x's unfolding, 46.0 as 48): hence a line through both against the sum.
inline uint32_t short_tile(uint32_t rows, uint32_t k_size, uint32_t out_rows, uint32_t compute_units) {
    const uint32_t columns = unfolded_columns(k_size);
    const uint64_t unfolded = block_tile<_Float16>(rows, columns, out_rows, compute_units).ns +
                              static_cast<uint64_t>(out_rows) * columns * 2 / 5000;
    const ShortChoice brief = choose_short_tile(rows, k_size, out_rows, compute_units);
    return brief.ns < (unfolded + 6000) * 6 / 7 ? brief.tm : 0;
}
// use(product) of a short block's tile
template <uint32_t kBlocks, typename Use>
void short_product(uint32_t tm, Use use) {
    if constexpr (kBlocks == 4) {
        if (tm == 8) return use(ShortProduct<8, kBlocks>{});
    }
    switch (tm) {
    case 2: return use(ShortProduct<2, kBlocks>{});
    case 4: return use(ShortProduct<4, kBlocks>{});
    default: return use(ShortProduct<6, kBlocks>{});
    }
}
template <uint32_t kBlocks>
void launch_short(const Q4Projection& p, const Unfold& u, uint32_t tm, hipStream_t stream) {
    hipLaunchKernelGGL(q4_unfold_kernel<kBlocks>, dim3((u.x_rows + 3) / 4), dim3(256), 0, stream, p, u);
    short_product<kBlocks>(tm, [&](auto product) {
        typedef decltype(product) Product;
        hipLaunchKernelGGL(q4_short_kernel<Product>,
                           dim3(p.first_row[p.segments] / Product::kTileN,
                                (u.x_rows + Product::kTileM - 1) / Product::kTileM),
                           dim3(Product::kThreads), Product::kLdsBytes, stream, p, u);
    });
}

typedef BlockTiles<_Float16> Q4Tiles;
int32_t launch_block(const Q4Projection& p, hipStream_t stream) {
    const StreamWorkspace workspace = stream_workspace(stream);
    const uint32_t columns = unfolded_columns(p.k_size);
    const uint32_t out_rows = p.first_row[p.segments];
    const bool whole = workspace.bytes >= kUnfoldWorkspaceBytes;
    constexpr uint64_t kExponentBytes = kWeightExponentBytes + kRowExponentBytes;
    const uint64_t unfolded_bytes = whole ? kUnfoldedWeightBytes + kUnfoldedRowBytes
                                          : (std::max(workspace.bytes, kExponentBytes) - kExponentBytes) / 512 * 512;
    const uint64_t weight_bytes = whole ? kUnfoldedWeightBytes : unfolded_bytes / 2;
    // whole tiles of either operand, as many as there are exponents for
    const auto slice_of = [&](uint64_t bytes, uint32_t most) {
        return static_cast<uint32_t>(std::min<uint64_t>(bytes / 2 / columns / 256 * 256, most));
    };
    const uint32_t weight_slice = whole ? out_rows : slice_of(weight_bytes, kGdnProjectionRows);
    const uint32_t slice = slice_of(unfolded_bytes - weight_bytes, 16384);
    // a queue (almost) without workspace: the rows kernel takes any number of rows
    if (workspace.base == nullptr || workspace.compute_units == 0 || weight_slice == 0 || slice == 0) {
        return launch_rows(p, stream);
    }
    Unfold u{};
    u.weights = reinterpret_cast<_Float16*>(workspace.base);
    u.rows = reinterpret_cast<_Float16*>(workspace.base + weight_bytes);
    u.weight_exponents = reinterpret_cast<int32_t*>(workspace.base + unfolded_bytes);
    u.row_exponents = reinterpret_cast<int32_t*>(
        reinterpret_cast<uint8_t*>(u.weight_exponents) + kWeightExponentBytes);
    const uint32_t tm = short_tile(p.rows, p.k_size, out_rows, workspace.compute_units);
    if (tm != 0) {
        u.short_rows = true;
        for (; u.first_row < p.rows; u.first_row += u.x_rows) {
            u.x_rows = std::min(slice, p.rows - u.first_row);
            if (p.k_size == 4 * kQ4Block) {
                launch_short<4>(p, u, tm, stream);
            } else {
                launch_short<8>(p, u, tm, stream);
            }
        }
        return TT_OK;
    }
    for (; u.first_weight < out_rows; u.first_weight += weight_slice) {
        const uint32_t columns_out = std::min(weight_slice, out_rows - u.first_weight);
        u.weight_rows = columns_out;
        for (u.first_row = 0; u.first_row < p.rows; u.first_row += u.x_rows) {
            u.x_rows = std::min(slice, p.rows - u.first_row);
            const dim3 grid((u.weight_rows + u.x_rows + 3) / 4);
            if (p.k_size == 4 * kQ4Block) {
                hipLaunchKernelGGL(q4_unfold_kernel<4>, grid, dim3(256), 0, stream, p, u);
            } else {
                hipLaunchKernelGGL(q4_unfold_kernel<8>, grid, dim3(256), 0, stream, p, u);
            }
            u.weight_rows = 0;
            Q4Tiles::choose(u.x_rows, columns, columns_out, workspace.compute_units, [&](auto product) {
                typedef decltype(product) Product;
                const BlockLaunch launch =
                    block_launch<Product>(u.x_rows, columns, columns_out, workspace.compute_units);
                hipLaunchKernelGGL(q4_product_kernel<Product>, dim3(launch.workgroups), dim3(Product::kThreads),
                                   Product::kLdsBytes, stream, u, p.output + u.first_weight, p.output_stride,
                                   columns, columns_out, launch.runs);
            });
        }
    }
    return TT_OK;
}

// ------------------------------------------------------- decode-wave kernel ---
//
// The same mathematics as the block product for 2..16 input rows (a decode wave), sized for
// latency: a workgroup owns 16 output rows and all input rows, its waves split K in slices
// of 512 columns (eight groups each), every operand of a slice is requested before the
// first is used, and the slices are summed through LDS in a fixed order.  Per group two
// v_mfma_f32_16x16x32_bf16 multiply the x rows with the nibbles as bf16 16 + nibble (lane g
// of a row owns the group's columns 16 g .. 16 g + 15) and two more, against a ones operand, give
// the group sums of x; then acc += scale[n] * products + bias[n] * sums in fp32.  The
// result has n along its columns, so a lane needs one scale and one bias per group, and
// reads all eight of a slice with two 16-byte loads.

constexpr float kNibbleOffset = 16.0f;   // nibbles enter the matrix unit as 16 + nibble

// The eight nibbles of `word` as the bf16 numbers 16 + nibble, in pairs 0 and 4, 1 and 5, 2 and 6, 3
// and 7: a nibble dropped into mantissa bits 3..6 of bf16 16.0 (0x4180), where it counts units, a
// shift, a mask and an or for two.  The offset leaves the products as 16 * (sum of x) too much, which the
// caller takes out of the bias term; 16 is the smallest offset that keeps all sixteen values in one
// binade, and keeps the fp32 partial sums about three times as large as the plain ones.
__device__ __forceinline__ bf16x8 offset_eight(uint32_t word) {
    uint32_t sixteens = 0x41804180u;
    asm("" : "+v"(sixteens));   // kept in a register: one v_and_or_b32 instead of two instructions
    u32x4 out;
    out[0] = ((word << 3) & 0x00780078u) | sixteens;
    out[1] = ((word >> 1) & 0x00780078u) | sixteens;
    out[2] = ((word >> 5) & 0x00780078u) | sixteens;
    out[3] = ((word >> 9) & 0x00780078u) | sixteens;
    return __builtin_bit_cast(bf16x8, out);
}
// eight values of x in that order
__device__ __forceinline__ u32x4 paired_eight(u32x4 x) {
    return u32x4{__builtin_amdgcn_perm(x[2], x[0], 0x05040100u), __builtin_amdgcn_perm(x[2], x[0], 0x07060302u),
                 __builtin_amdgcn_perm(x[3], x[1], 0x05040100u), __builtin_amdgcn_perm(x[3], x[1], 0x07060302u)};
}

// The eight nibbles of `word` less 8, as bf16, for a block of 2..16 rows.  A block used to be
// evaluated in the reference's own order, and its fp32 sums may be no further from the exact ones
// than there: the nibbles stay small (16 + nibble makes the partial sums three times as large), and
// the groups of a slice, whose products come from the matrix unit in fp32, are added up in 64 bits.
// Rms left where the exact result is zero (rows of N(0, 1), scales 0.5 .. 0.9) over 2048 / 4096
// columns: reference's order 6.5e-6 / 11.6e-6, this 4.1e-6 / 5.8e-6, a decode wave's form 22.5e-6 /
// 31.9e-6.
// Time against the decode wave's form, 12 rows: gdn_project 9.0 -> 9.2 us, outproj 6.3 -> 6.6 us.
__device__ __forceinline__ bf16x8 centred_eight(uint32_t word) {
    const uint32_t twos = word ^ 0x88888888u;   // nibble - 8 as four bits of two's complement
    bf16x8 out;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        out[i] = static_cast<__bf16>(static_cast<float>(static_cast<int32_t>(twos << (28 - 4 * i)) >> 28));
    }
    return out;
}

// bytes between the x rows staged in LDS: 16 more than a row, so that the sixteen lanes of
// a fragment read (one row each, the same columns) fall on different banks
template <uint32_t kWaves>
constexpr uint32_t kWaveRowBytes = kWaves * 1024 + 16;

// kWaves = k_size / 512; kRowsMax: the rows this instantiation takes at most; kCentred: a block's
// rows, see centred_eight
template <uint32_t kWaves, bool kNorm = false, bool kResidual = false, uint32_t kRowsMax = kQ4BatchRowsMax,
          bool kCentred = false>
__global__ __launch_bounds__(64 * kWaves) void q4_wave_kernel(Q4Projection p) {
    // [rows][kWaveRowBytes] of x, then the waves' partial results
    extern __shared__ __align__(16) uint8_t wave_lds[];
    constexpr uint32_t kThreads = 64 * kWaves;
    constexpr uint32_t kPiecesPerRow = kWaves * 64;          // 16-byte pieces of an x row
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t i16 = lane & 15, g = lane >> 4;
    const uint32_t n = blockIdx.x * 16 + i16;   // every matrix has a multiple of 16 rows
    const Q4Matrix matrix = matrix_of_row(p, blockIdx.x * 16);
    const uint64_t local = n - matrix.first_row;
    const uint32_t first_group = wave * 8;
    const uint32_t* words = matrix.words + local * (kWaves * 64) + first_group * 8 + 2 * g;
    const uint16_t* scales = matrix.scales + local * (kWaves * 8) + first_group;
    const uint16_t* biases = matrix.biases + local * (kWaves * 8) + first_group;

    // The x rows are the same for every workgroup: they come in once with coalesced 16-byte
    // loads (requested first, so that storing them does not wait for the weights) and are
    // read back from LDS as fragments; each lane loading its own 32 bytes per group from
    // global memory cost as much as streaming the weights.
    float* partial = reinterpret_cast<float*>(wave_lds + p.rows * kWaveRowBytes<kWaves>);
    u32x2 q[8];
    u32x4 scale_bits, bias_bits;
    auto request_weights = [&]() {
#pragma unroll
        for (uint32_t group = 0; group < 8; ++group) {
            q[group] = *reinterpret_cast<const u32x2*>(words + group * 8);
        }
        scale_bits = *reinterpret_cast<const u32x4*>(scales);
        bias_bits = *reinterpret_cast<const u32x4*>(biases);
    };
    // as the nibbles of a word come apart
    const auto in_order = [](u32x4 eight) { return kCentred ? eight : paired_eight(eight); };
    if constexpr (kNorm) {
        // The rows go through the RMS norm on their way into LDS, bit for bit as the norm
        // operator does it with one thread per four values: a thread here holds eight
        // values of a row, the slices of that operator's threads 2 t and 2 t + 1, whose
        // sum is the first step of its 32-lane tree; the other four steps run over the 16
        // lanes of a row of this wave, and the sixteen sums of a row of x meet in the same
        // zero-padded 32-slot tree.
        static_assert(kWaves == 4, "one 16-byte piece of a 2048-wide row per thread");
        float* stage = partial;   // [rows][16], before the partial results need the space
        u32x4 raw[kQ4BatchRowsMax];
#pragma unroll
        for (uint32_t r = 0; r < kQ4BatchRowsMax; ++r) {
            if (r < p.rows) {
                raw[r] = *reinterpret_cast<const u32x4*>(
                    p.input + static_cast<uint64_t>(r) * p.input_stride + threadIdx.x * 8);
            }
        }
        const u32x4 weight = *reinterpret_cast<const u32x4*>(p.norm_weight + threadIdx.x * 8);
        request_weights();   // in flight while the rows are normed
#pragma unroll
        for (uint32_t r = 0; r < kQ4BatchRowsMax; ++r) {
            if (r < p.rows) {
                const float slices = rms_slice_squares(raw[r][0], raw[r][1]) +
                                     rms_slice_squares(raw[r][2], raw[r][3]);
                const float sixteen = row_sum(slices);
                if ((threadIdx.x & 15) == 0) stage[r * 16 + (threadIdx.x >> 4)] = sixteen;
            }
        }
        __syncthreads();
        float inverse[kQ4BatchRowsMax];
#pragma unroll
        for (uint32_t r = 0; r < kQ4BatchRowsMax; ++r) {
            if (r < p.rows) {
                const float slot = (lane & 31) < 16 ? stage[r * 16 + (lane & 15)] : 0.0f;
                inverse[r] = rms_inverse(half_wave_sum(slot), kWaves * kQ4Block);
            }
        }
        __syncthreads();   // the stage is read before the partial results overwrite it
#pragma unroll
        for (uint32_t r = 0; r < kQ4BatchRowsMax; ++r) {
            if (r < p.rows) {
                u32x4 normed;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) normed[j] = rms_scale_pair(raw[r][j], weight[j], inverse[r]);
                *reinterpret_cast<u32x4*>(wave_lds + r * kWaveRowBytes<kWaves> + threadIdx.x * 16) = in_order(normed);
            }
        }
    } else {
        // One piece of each row per thread.  Over 2048 columns the weights are requested before the
        // first piece is stored, so that the two round trips overlap (rows past the last repeat it:
        // no branch between the requests, where what is in flight would be waited for): gdn_project
        // of 4 / 8 / 12 / 16 rows 8.24 / 8.92 / 10.16 / 12.04 -> 8.14 / 8.70 / 9.37 / 10.66 us.  Over
        // 4096, half a workgroup to a compute unit, the weights first cost 0.1 .. 0.2 us of 6 .. 7.
        static_assert(kPiecesPerRow == kThreads, "a row is one piece per thread");
        if constexpr (kWaves == 4) {
            u32x4 raw[kRowsMax];
#pragma unroll
            for (uint32_t r = 0; r < kRowsMax; ++r) {
                raw[r] = *reinterpret_cast<const u32x4*>(
                    p.input + static_cast<uint64_t>(min(r, p.rows - 1)) * p.input_stride + threadIdx.x * 8);
            }
            request_weights();
#pragma unroll
            for (uint32_t r = 0; r < kRowsMax; ++r) {
                *reinterpret_cast<u32x4*>(wave_lds + min(r, p.rows - 1) * kWaveRowBytes<kWaves> +
                                          threadIdx.x * 16) = in_order(raw[r]);
            }
        } else {
            for (uint32_t first = 0; first < p.rows; first += 4) {
                u32x4 staged[4];
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    staged[j] = *reinterpret_cast<const u32x4*>(
                        p.input + static_cast<uint64_t>(min(first + j, p.rows - 1)) * p.input_stride +
                        threadIdx.x * 8);
                }
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    *reinterpret_cast<u32x4*>(wave_lds + min(first + j, p.rows - 1) * kWaveRowBytes<kWaves> +
                                              threadIdx.x * 16) = in_order(staged[j]);
                }
            }
            request_weights();
        }
    }
    __syncthreads();

    const uint8_t* x_row = wave_lds + min(i16, p.rows - 1) * kWaveRowBytes<kWaves> +
                           first_group * (kQ4Group * 2) + 32 * g;
    bf16x8 eight_ones;
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) eight_ones[j] = static_cast<__bf16>(1.0f);
    const f32x4 zero = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 acc = zero;
    [[maybe_unused]] double wide[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (uint32_t group = 0; group < 8; ++group) {
        const u32x4 x_low = *reinterpret_cast<const u32x4*>(x_row + group * (kQ4Group * 2));
        const u32x4 x_high = *reinterpret_cast<const u32x4*>(x_row + group * (kQ4Group * 2) + 16);
        f32x4 products = zero, sums = zero;
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j) {
            const bf16x8 xf = __builtin_bit_cast(bf16x8, j == 0 ? x_low : x_high);
            const bf16x8 qf = kCentred ? centred_eight(q[group][j]) : offset_eight(q[group][j]);
            products = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, qf, products, 0, 0, 0);
            sums = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, eight_ones, sums, 0, 0, 0);
        }
        const float scale = widen_half(scale_bits[group >> 1], group & 1);
        // scale * (products + kBack sums) + bias * sums
        constexpr float kBack = kCentred ? 8.0f : -kNibbleOffset;
        const float bias = fmaf(kBack, scale, widen_half(bias_bits[group >> 1], group & 1));
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            if constexpr (kCentred) {
                wide[i] += fmaf(scale, products[i], bias * sums[i]);
            } else {
                acc[i] = fmaf(bias, sums[i], fmaf(scale, products[i], acc[i]));
            }
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        partial[(wave * 4 + i) * 64 + lane] = kCentred ? static_cast<float>(wide[i]) : acc[i];
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        std::conditional_t<kCentred, double, float> sum = partial[i * 64 + lane];
#pragma unroll
        for (uint32_t w = 1; w < kWaves; ++w) sum += partial[(w * 4 + i) * 64 + lane];
        const float total = static_cast<float>(sum);
        const uint32_t m = 4 * g + i;   // the result has the input rows along its rows
        if (m < p.rows) {
            uint16_t result = store16(total);
            if constexpr (kResidual) {
                // the residual sum of the step that follows (moe.metal:1-46), on the rounded projection
                const uint16_t before = p.residual[static_cast<uint64_t>(m) * p.residual_stride + n];
                result = rms_store16(rms_widen(rms_fz16(before)) + rms_widen(rms_fz16(result)));
            }
            p.output[static_cast<uint64_t>(m) * p.output_stride + n] = result;
        }
    }
}

template <uint32_t kWaves>
constexpr uint32_t wave_lds_bytes(uint32_t rows) {
    return rows * kWaveRowBytes<kWaves> + kWaves * 4 * 64 * 4;
}

// The instantiation for 2048 columns that requests the fewest rows of x, repeats included.
template <bool kCentred>
auto wave_kernel_for(uint32_t rows) {
    return rows <= 4    ? q4_wave_kernel<4, false, false, 4, kCentred>
           : rows <= 8  ? q4_wave_kernel<4, false, false, 8, kCentred>
           : rows <= 12 ? q4_wave_kernel<4, false, false, 12, kCentred>
                        : q4_wave_kernel<4, false, false, 16, kCentred>;
}

int32_t launch_wave(const Q4Projection& p, hipStream_t stream) {
    const uint32_t out_rows = p.first_row[p.segments];
    switch (p.k_size / kQ4Block) {
    case 4:
        if (p.residual != nullptr) return TT_CMD_INVALID_DISPATCH_EXTENT;
        if (p.norm_weight != nullptr) {
            hipLaunchKernelGGL((q4_wave_kernel<4, true, false>), dim3(out_rows / 16), dim3(256),
                               wave_lds_bytes<4>(p.rows), stream, p);
        } else {
            hipLaunchKernelGGL(p.centred ? wave_kernel_for<true>(p.rows) : wave_kernel_for<false>(p.rows),
                               dim3(out_rows / 16), dim3(256), wave_lds_bytes<4>(p.rows), stream, p);
        }
        break;
    case 8:
        if (p.norm_weight != nullptr) return TT_CMD_INVALID_DISPATCH_EXTENT;
        if (p.residual != nullptr) {
            hipLaunchKernelGGL((q4_wave_kernel<8, false, true>), dim3(out_rows / 16), dim3(512),
                               wave_lds_bytes<8>(p.rows), stream, p);
        } else {
            hipLaunchKernelGGL((p.centred ? q4_wave_kernel<8, false, false, 16, true> : q4_wave_kernel<8>),
                               dim3(out_rows / 16), dim3(512), wave_lds_bytes<8>(p.rows), stream, p);
        }
        break;
    default: return TT_CMD_INVALID_DISPATCH_EXTENT;
    }
    return TT_OK;
}

// Binds `count` weight matrices from buffer slots first, first+3, ...: words, scales,
// biases of each, sized for its rows.
void bind_segments(Args& a, Q4Projection& p, uint32_t first_slot, const uint32_t* rows,
                   uint32_t count, uint32_t k_size) {
    p.segments = count;
    p.k_size = k_size;
    p.first_row[0] = 0;
    for (uint32_t s = 0; s < count; ++s) {
        const uint32_t slot = first_slot + 3 * s;
        p.words[s] = a.buffer<const uint32_t>(slot, static_cast<uint64_t>(rows[s]) * (k_size / 8) * 4);
        p.scales[s] =
            a.buffer<const uint16_t>(slot + 1, static_cast<uint64_t>(rows[s]) * (k_size / kQ4Group) * 2);
        p.biases[s] =
            a.buffer<const uint16_t>(slot + 2, static_cast<uint64_t>(rows[s]) * (k_size / kQ4Group) * 2);
        p.first_row[s + 1] = p.first_row[s] + rows[s];
    }
}

constexpr uint32_t kMaxBatchRows = 16;              // rows of a decode wave (decode_step.cpp:554)
constexpr uint32_t kProjectionRowThreads = 128;     // decode_geometry.h:147
constexpr uint32_t kOutProjectionRowThreads = 64;   // decode_geometry.h:148

// One projection operator family: its weight matrices (slots 1, 4, 7, ...), input
// width, the slot of the output and the threads per group of the reference's grid
// (one 32-lane group per output row).
struct Family {
    uint32_t segment_rows[kMaxSegments];
    uint32_t segments;
    uint32_t k_size;
    uint32_t out_slot;
    uint32_t threads;
    constexpr uint32_t out_rows() const {
        uint32_t total = 0;
        for (uint32_t s = 0; s < segments; ++s) total += segment_rows[s];
        return total;
    }
    constexpr uint64_t groups() const {
        const uint32_t per_group = threads / 32;
        return (out_rows() + per_group - 1) / per_group;
    }
};
constexpr Family kAttnProject{{kAttnQGateRows, kAttnVRowOffset - kAttnQGateRows,
                               kAttnProjectionRows - kAttnVRowOffset, 0},
                              3, kHidden, 10, kProjectionRowThreads};
constexpr Family kGdnProject{{kGdnConvChannels, kGdnValueValues, kGdnValueHeads, kGdnValueHeads},
                             4, kHidden, 13, kProjectionRowThreads};
constexpr Family kOutProject{{kHidden, 0, 0, 0}, 1, kGdnValueValues, 4, kOutProjectionRowThreads};
static_assert(kAttnProject.out_rows() == kAttnProjectionRows && kAttnProject.groups() == 2304);
static_assert(kGdnProject.out_rows() == kGdnProjectionRows && kGdnProject.groups() == 3088);
static_assert(kOutProject.out_rows() == kHidden && kOutProject.groups() == 1024);

// Binds input, weights and output once rows / strides / tiling are known, checks the
// reference's grid (groups, tiles) x threads, and launches.
int32_t finish(Args& a, const Grid& g, hipStream_t stream, bool validate_only, const Family& f,
               Q4Projection& p, uint32_t k_size, uint64_t tiles, bool wave_kernel = false) {
    const uint32_t out_rows = f.out_rows();
    a.require(p.output_stride >= out_rows, TT_CMD_INVALID_BUFFER);
    a.require(grid_is(g, f.groups(), tiles, 1, f.threads, 1, 1), TT_CMD_INVALID_DISPATCH_EXTENT);
    if (a.status != TT_OK) return a.status;
    p.input_stride = k_size;
    p.input = a.buffer<const uint16_t>(0, static_cast<uint64_t>(p.rows) * k_size * 2);
    bind_segments(a, p, 1, f.segment_rows, f.segments, k_size);
    p.output = a.buffer<uint16_t>(
        f.out_slot, (static_cast<uint64_t>(p.rows - 1) * p.output_stride + out_rows) * 2);
    if (a.status != TT_OK) return a.status;
    // a handful of rows is a weight-streaming problem: the exact rows kernel; a block
    // is a matrix product: MFMA
    const bool block = !wave_kernel && p.rows > kQ4BatchRowsMax;
    if (block) {
        const int32_t status = check_block_operands(p);
        if (status != TT_OK) return status;
    }
    if (validate_only) return TT_OK;
    if (wave_kernel) return launch_wave(p, stream);
    return block ? launch_block(p, stream) : launch_rows(p, stream);
}

// one input row; grid (groups) x threads
int32_t project_single(const Bindings& b, const Grid& g, hipStream_t stream, bool validate_only,
                       const Family& f) {
    Args a(b);
    Q4Projection p{};
    p.rows = p.row_tile = 1;
    p.output_stride = f.out_rows();
    return finish(a, g, stream, validate_only, f, p, f.k_size, 1);
}

// rows of a decode wave: c[out+1] rows (1..16), then the output row stride where the
// operator has one, then the row tile; grid (groups, ceil(rows / tile)) x threads
enum class WaveExtra { None, NormedInput, ResidualOutput };

int32_t project_tiled(const Bindings& b, const Grid& g, hipStream_t stream, bool validate_only,
                      const Family& f, bool strided_output, bool wave_kernel = false,
                      WaveExtra extra = WaveExtra::None) {
    Args a(b);
    Q4Projection p{};
    p.rows = a.constant(f.out_slot + 1);
    p.output_stride = strided_output ? a.constant(f.out_slot + 2) : f.out_rows();
    p.row_tile = a.constant(f.out_slot + (strided_output ? 3 : 2));
    a.require(p.rows >= 1 && p.rows <= kMaxBatchRows && p.row_tile >= 1 &&
                  p.row_tile <= kQ4BatchRowsMax,
              TT_CMD_INVALID_DISPATCH_EXTENT);
    // the buffer after the operator's last constant: the norm weight of the input rows, or
    // the rows the projection is added to (same row stride as the output)
    const uint32_t extra_slot = f.out_slot + (strided_output ? 4 : 3);
    if (extra == WaveExtra::NormedInput) {
        p.norm_weight = a.buffer<const uint16_t>(extra_slot, static_cast<uint64_t>(f.k_size) * 2);
    } else if (extra == WaveExtra::ResidualOutput && a.status == TT_OK) {
        p.residual_stride = p.output_stride;
        p.residual = a.buffer<const uint16_t>(
            extra_slot, (static_cast<uint64_t>(p.rows - 1) * p.residual_stride + f.out_rows()) * 2);
    }
    if (a.status != TT_OK) return a.status;
    return finish(a, g, stream, validate_only, f, p, f.k_size,
                  (p.rows + p.row_tile - 1) / p.row_tile, wave_kernel);
}

// a block of consecutive tokens: c[out+1] rows, then the input width where the
// operator takes one; grid (groups) x threads.  wave_kernel: at most 16 rows, on q4_wave_kernel
int32_t project_block(const Bindings& b, const Grid& g, hipStream_t stream, bool validate_only,
                      const Family& f, bool variable_width, bool wave_kernel = false) {
    Args a(b);
    Q4Projection p{};
    p.rows = a.constant(f.out_slot + 1);
    const uint32_t k_size = variable_width ? a.constant(f.out_slot + 2) : f.k_size;
    // the two input widths of the model: hidden (2048) and the attention / value width (4096)
    a.require(p.rows >= 1 && (k_size == kHidden || k_size == kGdnValueValues) &&
                  (!wave_kernel || p.rows <= kMaxBatchRows),
              TT_CMD_INVALID_DISPATCH_EXTENT);
    if (a.status != TT_OK) return a.status;
    p.row_tile = kQ4BatchRowsMax;
    p.output_stride = f.out_rows();
    p.centred = wave_kernel;
    return finish(a, g, stream, validate_only, f, p, k_size, 1, wave_kernel);
}

// attn_project: b0 input[2048], b1-3 query+gate (8192 rows), b4-6 key (512), b7-9 value
// (512), b10 projection[9216]; grid 2304 x 128 (decode_step.cpp:705-711).
int32_t op_attn_project(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_single(b, g, s, v, kAttnProject);
}
// attn_project_ms{,_v2}: + c11 rows, c12 row tile; grid (2304, ceil(rows/tile)) x 128
// (decode_step.cpp:1213-1229).
int32_t op_attn_project_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kAttnProject, false);
}
// attn_project_blk: + c11 block rows; grid 2304 x 128 (prefill_step.cpp:1428-1446).
int32_t op_attn_project_blk(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_block(b, g, s, v, kAttnProject, false);
}
// gdn_project: b0 input[2048], b1-3 qkv (8192 rows), b4-6 z (4096), b7-9 b (32), b10-12 a
// (32), b13 projection[12352]; grid 3088 x 128 (decode_step.cpp:657-664).
int32_t op_gdn_project(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_single(b, g, s, v, kGdnProject);
}
// gdn_project_ms{,_v2}: + c14 rows, c15 row tile (decode_step.cpp:1117-1130).
int32_t op_gdn_project_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kGdnProject, false);
}
// gdn_project_blk: + c14 block rows (prefill_step.cpp:1909-1926).
int32_t op_gdn_project_blk(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_block(b, g, s, v, kGdnProject, false);
}
// gdn_outproj: b0 input[4096], b1-3 weights (2048 rows), b4 output[2048]; grid 1024 x 64
// (decode_step.cpp:697-701, 729-733: the out_projection pipeline of both layer kinds).
int32_t op_gdn_outproj(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_single(b, g, s, v, kOutProject);
}
// gdn_outproj_ms{,_v2}: + c5 rows, c6 output row stride, c7 row tile (decode_step.cpp:1196-1206).
int32_t op_gdn_outproj_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kOutProject, true);
}
// attn_project_mfma_ms, gdn_project_mfma_ms, gdn_outproj_mfma_ms (no reference counterpart):
// the bindings and grids of the _ms forms, evaluated on the matrix unit by q4_wave_kernel -
// the same mathematics in another summation order, for decode waves of several lanes.
int32_t op_attn_project_mfma_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kAttnProject, false, true);
}
int32_t op_gdn_project_mfma_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kGdnProject, false, true);
}
int32_t op_gdn_outproj_mfma_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kOutProject, true, true);
}
// attn_project_rms_mfma_ms, gdn_project_rms_mfma_ms (no reference counterpart): the _mfma_ms
// forms on rows that have not been normed yet, + b13 / b16 the norm weight [2048]: every
// workgroup norms the rows while it stages them (rms_only_ms's bits), which takes the norm
// dispatch out of a decode layer.
int32_t op_attn_project_rms_mfma_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kAttnProject, false, true, WaveExtra::NormedInput);
}
int32_t op_gdn_project_rms_mfma_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kGdnProject, false, true, WaveExtra::NormedInput);
}
// gdn_outproj_residual_mfma_ms (no reference counterpart): gdn_outproj_mfma_ms + b8 the rows
// the projection is added to, [rows][c6]: output = bf16(residual + bf16(projection)), the sum
// residual_rms would form next (moe.metal:1-46); the output may be the residual buffer itself.
int32_t op_gdn_outproj_residual_mfma_ms(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_tiled(b, g, s, v, kOutProject, true, true, WaveExtra::ResidualOutput);
}
// outproj_blk: + c5 block rows, c6 input width (prefill_step.cpp:2063-2078).
int32_t op_outproj_blk(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_block(b, g, s, v, kOutProject, true);
}
// attn_project_mfma_blk, gdn_project_mfma_blk, outproj_mfma_blk (no reference counterpart): the
// bindings and grids of the _blk forms for at most 16 rows, evaluated on the matrix unit with fp32
// sums no further from the exact ones than the reference's order (centred_eight); the _blk forms
// themselves keep that order, and its bits, up to 16 rows.
int32_t op_attn_project_mfma_blk(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_block(b, g, s, v, kAttnProject, false, true);
}
int32_t op_gdn_project_mfma_blk(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_block(b, g, s, v, kGdnProject, false, true);
}
int32_t op_outproj_mfma_blk(const Bindings& b, const Grid& g, hipStream_t s, bool v) {
    return project_block(b, g, s, v, kOutProject, true, true);
}

}  // namespace

uint64_t q4_workspace_bytes() { return kUnfoldWorkspaceBytes; }

#if !defined(__HIP_DEVICE_COMPILE__)  // host-side table of launchers
uint32_t q4_block_tile(uint32_t rows, uint32_t k_size, uint32_t out_rows, uint32_t compute_units) {
    const uint32_t tm = short_tile(rows, k_size, out_rows, compute_units);
    if (tm != 0) return kShortBlockTiles + tm;
    const uint32_t columns = unfolded_columns(k_size);
    const uint32_t slice = std::min<uint64_t>(kUnfoldedRowBytes / 2 / columns / 256 * 256, 16384);
    return static_cast<uint32_t>(block_tile<_Float16>(std::min(rows, slice), columns, out_rows, compute_units).tile);
}

bool prepare_q4_kernels() {
    const auto allow = [](auto product) {
        typedef decltype(product) Product;
        return hipFuncSetAttribute(reinterpret_cast<const void*>(q4_product_kernel<Product>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                   Product::kLdsBytes) == hipSuccess;
    };
    const auto allow_wave = [](void (*kernel)(Q4Projection), uint32_t bytes) {
        return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
    };
    const auto allow_rows = [&](uint32_t rows) {
        return allow_wave(wave_kernel_for<false>(rows), wave_lds_bytes<4>(rows)) &&
               allow_wave(wave_kernel_for<true>(rows), wave_lds_bytes<4>(rows));
    };
    bool short_allowed = true;
    const auto allow_short = [&](auto product) {
        typedef decltype(product) Product;
        short_allowed = short_allowed &&
                        hipFuncSetAttribute(reinterpret_cast<const void*>(q4_short_kernel<Product>),
                                            hipFuncAttributeMaxDynamicSharedMemorySize,
                                            Product::kLdsBytes) == hipSuccess;
    };
    for (const uint32_t tm : {2u, 4u, 6u, 8u}) short_product<4>(tm, allow_short);
    for (const uint32_t tm : {2u, 4u, 6u}) short_product<8>(tm, allow_short);
    return short_allowed && Q4Tiles::each(allow) &&
           allow_wave(q4_rows_kernel<4, true, false>, kRowsStagedBytes) &&
           allow_wave(q4_rows_kernel<8, true>, kRowsStagedBytes) &&
           allow_wave(q4_rows_kernel<8, true, false>, kRowsStagedBytes) &&
           allow_rows(4) && allow_rows(8) && allow_rows(12) && allow_rows(16) &&
           allow_wave(q4_wave_kernel<8>, wave_lds_bytes<8>(16)) &&
           allow_wave(q4_wave_kernel<8, false, false, 16, true>, wave_lds_bytes<8>(16)) &&
           hipFuncSetAttribute(reinterpret_cast<const void*>(q4_wave_kernel<4, true, false>),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               wave_lds_bytes<4>(kQ4BatchRowsMax)) == hipSuccess &&
           hipFuncSetAttribute(reinterpret_cast<const void*>(q4_wave_kernel<8, false, true>),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               wave_lds_bytes<8>(kQ4BatchRowsMax)) == hipSuccess;
}

const KernelDesc kQ4ProjectKernels[] = {
    {"attn_project", op_attn_project},
    {"attn_project_ms", op_attn_project_ms},
    {"attn_project_ms_v2", op_attn_project_ms},
    {"attn_project_blk", op_attn_project_blk},
    {"gdn_project", op_gdn_project},
    {"gdn_project_ms", op_gdn_project_ms},
    {"gdn_project_ms_v2", op_gdn_project_ms},
    {"gdn_project_blk", op_gdn_project_blk},
    {"gdn_outproj", op_gdn_outproj},
    {"gdn_outproj_ms", op_gdn_outproj_ms},
    {"gdn_outproj_ms_v2", op_gdn_outproj_ms},
    {"outproj_blk", op_outproj_blk},
    {"attn_project_mfma_ms", op_attn_project_mfma_ms},
    {"gdn_project_mfma_ms", op_gdn_project_mfma_ms},
    {"gdn_outproj_mfma_ms", op_gdn_outproj_mfma_ms},
    {"attn_project_rms_mfma_ms", op_attn_project_rms_mfma_ms},
    {"gdn_project_rms_mfma_ms", op_gdn_project_rms_mfma_ms},
    {"gdn_outproj_residual_mfma_ms", op_gdn_outproj_residual_mfma_ms},
    {"attn_project_mfma_blk", op_attn_project_mfma_blk},
    {"gdn_project_mfma_blk", op_gdn_project_mfma_blk},
    {"outproj_mfma_blk", op_outproj_mfma_blk},
};
const uint32_t kQ4ProjectKernelCount = sizeof(kQ4ProjectKernels) / sizeof(kQ4ProjectKernels[0]);
#endif

}  // namespace tt
