// C[m][n] = sum_k X[m][k] W[n][k] on the matrix unit for blocks of rows: both operands 16-bit
// floats (bf16 or f16) with k contiguous, sums in fp32, and the way a tile of sums leaves is the
// caller's.  One persistent workgroup of kWavesM x kWavesN waves owns tiles of kTileM x kTileN
// and walks K in units of 64 columns, two steps of 32 each:
//   * both operands go from global memory straight into LDS (16 bytes per lane and
//     transfer, whole 128-byte lines of a row, no registers), a ring of kRing units.  The
//     transfers are issued as assembly, so that the only waits are the ones written below
//     (M0 is used for nothing else in these kernels).  A ring row is one row's 128 bytes of
//     the unit; 16-byte piece p of row r sits in slot p ^ (r & 7), with which the 16-byte
//     fragment reads of a wave (sixteen consecutive rows, one piece per quarter wave) were
//     measured free of bank conflicts.
//   * a wave multiplies its part of the tile as products of 16 x 16 x 32, W as the left
//     operand: a lane then holds four consecutive n of one m per product.  The fragments of a
//     step are read into registers while the step before it is multiplied; one barrier per
//     unit.
//   * the first units of a workgroup's next tile are requested before it converts and
//     stores the sums of this one.
// m and n past the end are clamped on the way in; the caller does not store them.
#pragma once

#include <algorithm>
#include <type_traits>

#include "../tt_internal.h"

namespace tt {
namespace {

// lane l's 16 bytes at base + offset land at lds_address + 16 l
__device__ __forceinline__ void block_transfer(const uint8_t* base, uint32_t offset,
                                               uint32_t lds_address) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_address)), "v"(offset), "s"(base)
                 : "memory");
}

// the rounds of tiles dealt in runs (block_launch); of the first, the workgroups mod 8 and by 8
constexpr uint32_t kWholeRounds = 1, kLastRound = 2, kRunsMore = 2, kRunsShare = 5;

// s_waitcnt until at most `left` (< 64) transfers are in flight
constexpr uint32_t block_vmcnt(uint32_t left) { return 0x0F70u | (left & 15u) | ((left >> 4) << 14); }

// two sums to a packed bf16 pair: hardware round to nearest even, then results below the
// normal range flushed to signed zero
__device__ __forceinline__ uint32_t block_pack(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float Pair;
    typedef __attribute__((ext_vector_type(2))) __bf16 Rounded;
    const uint32_t pair = __builtin_bit_cast(uint32_t, __builtin_convertvector(Pair{a, b}, Rounded));
    const uint32_t keep = ((pair & 0x00007F80u) ? 0x0000FFFFu : 0x00008000u) |
                          ((pair & 0x7F800000u) ? 0xFFFF0000u : 0x80000000u);
    return pair & keep;
}

// four results as bf16 at columns n .. n + 3 of an output row of `out_dim`; wide: 8-byte aligned
template <typename Sums>
__device__ __forceinline__ void block_store(uint16_t* out_row, uint32_t n, uint32_t out_dim,
                                            bool wide, Sums v) {
    typedef __attribute__((ext_vector_type(2))) uint32_t Four;
    const Four four = Four{block_pack(v[0], v[1]), block_pack(v[2], v[3])};
    if (wide && n + 4 <= out_dim) {
        *reinterpret_cast<Four*>(out_row + n) = four;
    } else {
        for (uint32_t j = 0; j < 4 && n + j < out_dim; ++j) {
            out_row[n + j] = static_cast<uint16_t>(four[j >> 1] >> (16 * (j & 1)));
        }
    }
}

template <typename Element, uint32_t kTileM_, uint32_t kTileN_, uint32_t kWavesM, uint32_t kWavesN,
          uint32_t kRing = 2>
struct BlockProduct {
    static constexpr uint32_t kTileM = kTileM_, kTileN = kTileN_;
    static constexpr uint32_t kWaves = kWavesM * kWavesN;
    static constexpr uint32_t kThreads = 64 * kWaves;
    static constexpr uint32_t kUnitColumns = 64;
    static constexpr uint32_t kRowBytes = kUnitColumns * 2;
    static constexpr uint32_t kXUnitBytes = kTileM * kRowBytes;
    static constexpr uint32_t kUnitBytes = (kTileM + kTileN) * kRowBytes;
    static constexpr uint32_t kLdsBytes = kRing * kUnitBytes;
    static constexpr uint32_t kWaveM = kTileM / kWavesM, kWaveN = kTileN / kWavesN;
    static constexpr uint32_t kTm = kWaveM / 16, kTn = kWaveN / 16;
    static_assert(kLdsBytes <= 160 * 1024, "the ring fits a compute unit");
    // A unit is kTileM + kTileN rows in transfers of eight.  Where both operands' divide among the
    // waves, a wave has its share of either, known when this is compiled (the 256 x 256 tile took 2 %
    // longer without that); other tiles deal them in runs of both, and what is over repeats the last.
    static constexpr uint32_t kXTransfers = kTileM / 8, kAllTransfers = (kTileM + kTileN) / 8;
    static constexpr bool kEvenShares = kXTransfers % kWaves == 0 && kAllTransfers % kWaves == 0;
    static constexpr uint32_t kTransfers = (kAllTransfers + kWaves - 1) / kWaves;   // of a wave
    static_assert(kXTransfers * 8 == kTileM && kAllTransfers * 8 == kTileM + kTileN &&
                      kTm * 16 * kWavesM == kTileM && kTn * 16 * kWavesN == kTileN,
                  "whole transfers and fragments");

    static constexpr uint32_t vmcnt(uint32_t left) { return block_vmcnt(left); }
    static_assert((kRing - 2) * kTransfers < 64, "what vmcnt counts");

    typedef __attribute__((ext_vector_type(8))) Element Elements;
    typedef __attribute__((ext_vector_type(4))) float Sums;
    // A step's fragments.  Tall waves keep one set of x fragments, each replaced by the next
    // step's as soon as its products have been issued (two sets would not fit the registers);
    // for one or two fragments that would be a wait at the end of every step.
    static constexpr bool kTwoSetsOfX = kTm <= 2;
    struct Fragments {
        Elements w[kTn], x[kTwoSetsOfX ? kTm : 1];
    };

    static __device__ __forceinline__ Sums product(Elements w, Elements x, Sums sums) {
        if constexpr (std::is_same<Element, _Float16>::value) {
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(w, x, sums, 0, 0, 0);
        } else {
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, sums, 0, 0, 0);
        }
    }

    // x [rows][in_dim], weights [out_dim][in_dim], in_dim a multiple of 64; 16-byte aligned and
    // each smaller than 4 GiB.  runs: the rounds dealt in runs, block_launch's.  store(m, n, sums) gets the
    // sums of row m, columns n .. n + 3.
    template <typename Store>
    static __device__ __forceinline__ void run(const void* x, const void* weights, uint32_t rows,
                                               uint32_t in_dim, uint32_t out_dim, uint32_t runs, Store store) {
        extern __shared__ __align__(16) uint8_t block_lds[];
        // one wait for all arguments: fetched where each is used, a short product waits three times
        const uint32_t workgroups = gridDim.x;
        asm volatile("" ::"s"(x), "s"(weights), "s"(workgroups));
        const uint32_t lane = threadIdx.x & 63;
        const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const uint32_t i16 = lane & 15, g = lane >> 4;
        const uint32_t units = in_dim / kUnitColumns;
        const uint32_t n_tiles = (out_dim + kTileN - 1) / kTileN;
        const uint32_t m_tiles = (rows + kTileM - 1) / kTileM;
        const uint32_t tiles = n_tiles * m_tiles;
        const uint32_t lds_base = static_cast<uint32_t>(
            reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)block_lds));
        const uint32_t wave_n = wave % kWavesN, wave_m = wave / kWavesN;

        // staging roles: transfer t fills rows 8 t .. 8 t + 7, those of x and then those of the
        // weights; lane l lands in row + (l >> 3), slot l & 7, so it fetches piece (l & 7) ^ (l >> 3)
        // of that row
        const uint8_t* x_base = reinterpret_cast<const uint8_t*>(x);
        const uint8_t* w_base = reinterpret_cast<const uint8_t*>(weights);
        const uint32_t piece = ((lane & 7) ^ (lane >> 3)) * 16;
        const uint32_t row_bytes = in_dim * 2;
        // Tiles are numbered along bands of eight tile rows, down a band's columns first, so that
        // a run of consecutive numbers is a compact patch (32 of them: eight rows x four columns,
        // twelve operand panels for 32 tiles).
        auto place = [&](uint32_t tile, uint32_t& m0, uint32_t& n0) {
            const uint32_t band = tile / (8 * n_tiles);
            const uint32_t band_rows = min(8u, m_tiles - 8 * band);
            const uint32_t within = tile - band * 8 * n_tiles;
            m0 = (8 * band + within % band_rows) * kTileM;
            n0 = (within / band_rows) * kTileN;
        };
        // This wave's transfer `index` of `unit`.  Lane offsets are bytes from the tile's first row
        // of its operand, clamped to the last row that is there (both carry `piece`).
        constexpr uint32_t kXShare = kEvenShares ? kXTransfers / kWaves : 0, kWShare = kTransfers - kXShare;
        const uint32_t lane_offset = (lane >> 3) * row_bytes + piece;
        const uint32_t x_lane = lane_offset + 8 * kXShare * wave * row_bytes;
        const uint32_t w_lane = lane_offset + 8 * kWShare * wave * row_bytes;
        uint32_t x_last = 0, w_last = 0;
        const uint8_t *x_tile = nullptr, *w_tile = nullptr;   // the tile the requests go to
        auto aim = [&](uint32_t tile) {
            uint32_t m0, n0;
            place(tile, m0, n0);
            x_tile = x_base + static_cast<uint64_t>(m0) * row_bytes;
            w_tile = w_base + static_cast<uint64_t>(n0) * row_bytes;
            x_last = (rows - 1 - m0) * row_bytes + piece;
            w_last = (out_dim - 1 - n0) * row_bytes + piece;
        };
        auto request_one = [&](uint32_t unit, uint32_t index) __attribute__((always_inline)) {
            const uint32_t to = lds_base + (unit % kRing) * kUnitBytes;
            if constexpr (!kEvenShares) {
                const uint32_t t = min(kTransfers * wave + index, kAllTransfers - 1);
                const bool of_x = t < kXTransfers;
                const uint32_t first = (of_x ? t : t - kXTransfers) * 8 * row_bytes;
                block_transfer((of_x ? x_tile : w_tile) + unit * kRowBytes,
                               min(lane_offset + first, of_x ? x_last : w_last), to + t * 8 * kRowBytes);
            } else if (index < kXShare) {
                block_transfer(x_tile + unit * kRowBytes, min(x_lane + 8 * index * row_bytes, x_last),
                               to + (8 * kXShare * wave + 8 * index) * kRowBytes);
            } else {
                const uint32_t j = index - kXShare;
                block_transfer(w_tile + unit * kRowBytes, min(w_lane + 8 * j * row_bytes, w_last),
                               to + kXUnitBytes + (8 * kWShare * wave + 8 * j) * kRowBytes);
            }
        };
        auto request = [&](uint32_t unit) {
#pragma unroll
            for (uint32_t index = 0; index < kTransfers; ++index) request_one(unit, index);
        };

        // fragment of (row, step of the unit): piece 4 step + g, stored at slot piece ^ (row & 7)
        const uint32_t frag_row = i16 * kRowBytes;
        const uint32_t frag_piece[2] = {(g ^ (i16 & 7)) * 16, ((4 + g) ^ (i16 & 7)) * 16};
        const uint32_t x_frag = kWaveM * wave_m * kRowBytes + frag_row;
        const uint32_t w_frag = kXUnitBytes + kWaveN * wave_n * kRowBytes + frag_row;
        Sums acc[kTn][kTm];

        Elements x_only[kTwoSetsOfX ? 1 : kTm];
        auto x_of = [&](Fragments& f, uint32_t tm) __attribute__((always_inline)) -> Elements& {
            return kTwoSetsOfX ? f.x[kTwoSetsOfX ? tm : 0] : x_only[kTwoSetsOfX ? 0 : tm];
        };
        auto read_weights = [&](uint32_t unit, uint32_t step, uint32_t tn, Fragments& f)
                                __attribute__((always_inline)) {
            f.w[tn] = *reinterpret_cast<const Elements*>(block_lds + (unit % kRing) * kUnitBytes +
                                                         frag_piece[step] + w_frag + tn * 16 * kRowBytes);
        };
        auto read_x = [&](uint32_t unit, uint32_t step, uint32_t tm, Fragments& f)
                          __attribute__((always_inline)) {
            x_of(f, tm) = *reinterpret_cast<const Elements*>(block_lds + (unit % kRing) * kUnitBytes +
                                                             frag_piece[step] + x_frag + tm * 16 * kRowBytes);
        };
        // One step: multiply, and between the products read the fragments of the step after it
        // and (requests) send the transfers of a unit off, a few at a time: reads and transfers
        // that are issued together keep the matrix unit waiting until the last of them has gone
        // out.  The order is pinned: left alone the scheduler sinks each read to the product
        // that needs it, a step later.
        auto multiply = [&](Fragments& now, auto reads, uint32_t unit, uint32_t step, Fragments& next,
                            auto requests, uint32_t requested) __attribute__((always_inline)) {
            constexpr bool kRead = decltype(reads)::value, kRequest = decltype(requests)::value;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t tm = 0; tm < kTm; ++tm) {
                if constexpr (kRead) {
#pragma unroll
                    for (uint32_t i = tm * kTn / kTm; i < (tm + 1) * kTn / kTm; ++i) {
                        read_weights(unit, step, i, next);
                    }
                    if (kTwoSetsOfX) {
                        read_x(unit, step, tm, next);
                    } else if (tm > 0) {
                        read_x(unit, step, tm - 1, next);
                    }
                }
                if constexpr (kRequest) {
#pragma unroll
                    for (uint32_t i = tm * kTransfers / kTm; i < (tm + 1) * kTransfers / kTm; ++i) {
                        request_one(requested, i);
                    }
                }
#pragma unroll
                for (uint32_t tn = 0; tn < kTn; ++tn) {
                    acc[tn][tm] = product(now.w[tn], x_of(now, tm), acc[tn][tm]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (kRead && !kTwoSetsOfX) read_x(unit, step, kTm - 1, next);
        };
        using std::bool_constant;
        // first step of `unit` (its fragments are in `first`): read the second step's while
        // multiplying; the unit was published a step ago, so nothing to wait for
        auto first_step = [&](uint32_t unit, Fragments& first, Fragments& second)
                              __attribute__((always_inline)) {
            multiply(first, bool_constant<true>{}, unit, 1, second, bool_constant<false>{}, 0);
        };
        // second step of `unit`: the next unit has landed - mine, then everybody's -, and nobody
        // reads this one any more (its last fragments are in `second`), so the unit kRing further
        // on goes into its place; read the next unit's first fragments while multiplying
        auto second_step = [&](uint32_t unit, Fragments& second, Fragments& first_of_next,
                               auto with_request) __attribute__((always_inline)) {
            if constexpr (decltype(with_request)::value) {
                __builtin_amdgcn_s_waitcnt(vmcnt((kRing - 2) * kTransfers));
            } else {
                __builtin_amdgcn_s_waitcnt(vmcnt(0));
            }
            __syncthreads();
            multiply(second, bool_constant<true>{}, unit + 1, 0, first_of_next, with_request, unit + kRing);
        };

        // Workgroup b of the dispatch order runs on XCD b mod 8, each XCD with an L2 of its own.  Dealt
        // in runs, the workgroups of an XCD (b / 8 = 0, 1, ...) take consecutive tiles of a round - the
        // operand panels a patch shares are then fetched into one L2 once instead of into several;
        // otherwise a workgroup takes the tile of its number (see block_launch).
        const auto in_runs = [&](uint32_t share, uint32_t more) {   // of a round of 8 share + more tiles
            const uint32_t xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
            return at < share + (xcd < more ? 1 : 0) ? xcd * share + min(xcd, more) + at : tiles;
        };
        const auto of_round = [&](uint32_t first) {
            const uint32_t left = tiles - min(first, tiles);
            if ((runs & (left >= workgroups ? kWholeRounds : kLastRound)) == 0) return first + blockIdx.x;
            const uint32_t count = min(workgroups, left);
            return first + in_runs(count / 8, count % 8);
        };
        // (the first round without of_round's work, of which a short product would wait for every instruction)
        uint32_t round = 0, tile = blockIdx.x;
        if (runs & kWholeRounds) {
            asm volatile("");   // a branch
            tile = in_runs(runs >> kRunsShare, runs >> kRunsMore & 7);
        }
        if (tile >= tiles) return;
        aim(tile);
        const uint32_t ahead = min(kRing, units);
        for (uint32_t unit = 0; unit < ahead; ++unit) request(unit);
        while (true) {
#pragma unroll
            for (uint32_t tn = 0; tn < kTn; ++tn) {
#pragma unroll
                for (uint32_t tm = 0; tm < kTm; ++tm) acc[tn][tm] = Sums{0.0f, 0.0f, 0.0f, 0.0f};
            }
            // unit 0 has landed (the second unit may be in flight; so may the stores of the tile
            // before, and reads and writes do not retire in one order: wait for everything)
            __builtin_amdgcn_s_waitcnt(vmcnt(0));
            __syncthreads();
            Fragments a, b;
#pragma unroll
            for (uint32_t tn = 0; tn < kTn; ++tn) read_weights(0, 0, tn, a);
#pragma unroll
            for (uint32_t tm = 0; tm < kTm; ++tm) read_x(0, 0, tm, a);
            uint32_t unit = 0;
            for (; unit + kRing < units; ++unit) {
                first_step(unit, a, b);
                second_step(unit, b, a, bool_constant<true>{});
            }
            for (; unit + 1 < units; ++unit) {   // nothing left to request
                first_step(unit, a, b);
                second_step(unit, b, a, bool_constant<false>{});
            }
            first_step(unit, a, b);
            multiply(b, bool_constant<false>{}, 0, 0, a, bool_constant<false>{}, 0);

            uint32_t m0, n0;
            place(tile, m0, n0);
            round += workgroups;
            const uint32_t next_tile = of_round(round);
            __syncthreads();   // nobody reads the stages any more
            if (next_tile < tiles) {
                aim(next_tile);
                for (uint32_t unit = 0; unit < ahead; ++unit) request(unit);
            }
            // the lane holds columns n0 + kWaveN wave_n + 16 tn + 4 g + j of row
            // m0 + kWaveM wave_m + 16 tm + i16
#pragma unroll
            for (uint32_t tm = 0; tm < kTm; ++tm) {
                const uint32_t m = m0 + kWaveM * wave_m + 16 * tm + i16;
                if (m >= rows) continue;
#pragma unroll
                for (uint32_t tn = 0; tn < kTn; ++tn) {
                    const uint32_t n = n0 + kWaveN * wave_n + 16 * tn + 4 * g;
                    if (n < out_dim) store(m, n, acc[tn][tm]);
                }
            }
            if (next_tile >= tiles) break;
            tile = next_tile;
        }
    }
};

enum class BlockTile { Large, Even, Deep, Tall, Small, Least, Wide, Seven, Five };

struct BlockCost {
    BlockTile tile;
    uint32_t m, n, single_unit, single_tile, both_unit, both_tile;
};
struct BlockChoice {
    BlockTile tile;
    uint32_t m, n;
    uint64_t ns;
};

// The tile with the shortest estimate.  A compute unit takes ceil(tiles / compute_units) tiles,
// two at a time where two workgroups fit it: `single` is the time of one tile alone on it, `both`
// of two side by side, as ns per 64 columns and ns per tile (fitted to the products below and to
// others of 33 .. 16384 rows, 2048 .. 12352 outputs and K = 2176 and 4352).
inline uint64_t block_ns(const BlockCost& c, uint32_t rows, uint32_t in_dim, uint32_t out_dim,
                         uint32_t compute_units) {
    const uint64_t units = in_dim / 64;
    const uint64_t tiles = static_cast<uint64_t>((rows + c.m - 1) / c.m) * ((out_dim + c.n - 1) / c.n);
    const uint64_t each = (tiles + compute_units - 1) / compute_units;
    const uint64_t time = each / 2 * (c.both_unit * units + c.both_tile) +
                          each % 2 * (c.single_unit * units + c.single_tile);
    // Compute units that the last round leaves idle make the others faster (they share the
    // power and the L2): one round of 256 x 256 tiles over K = 4096 takes 77 / 94 / 105 us with 64 /
    // 208 / 256 of them, two over K = 2048 104 with 392, three 159 with 576.  Fitted, the share of
    // the last round's walk that is saved is the idle share by 1 / (rounds + 2), or by a third for
    // a 128 x 128 tile left over behind pairs.
    const uint64_t idle = c.single_unit * units * (each * compute_units - tiles) / compute_units;
    if (c.n >= 256) return time - idle / (each + 2);
    return c.tile == BlockTile::Even && each > 1 && each % 2 == 1 ? time - idle / 3 : time;
}
inline BlockChoice choose_block_tile(uint32_t rows, uint32_t in_dim, uint32_t out_dim,
                                     uint32_t compute_units) {
    static constexpr BlockCost kCosts[] = {
        {BlockTile::Large, 256, 256, 1480, 8800, 2960, 17600},
        {BlockTile::Even, 128, 128, 600, 2000, 920, 4000},
        {BlockTile::Deep, 128, 128, 520, 2000, 1040, 4000},
        {BlockTile::Tall, 128, 64, 330, 1500, 630, 3000},
        {BlockTile::Small, 64, 64, 200, 1000, 400, 2000},
        {BlockTile::Least, 32, 64, 155, 1000, 275, 1500},
    };
    BlockChoice best{BlockTile::Large, 0, 0, ~0ull};
    for (const BlockCost& c : kCosts) {
        const uint64_t ns = block_ns(c, rows, in_dim, out_dim, compute_units);
        if (ns < best.ns) best = BlockChoice{c.tile, c.m, c.n, ns};
    }
    return best;
}
// Where 256 x 256 leaves a round short (or 128 x 128 takes its place for that) another height or a
// wider tile may fill the rounds better.  Taken where its estimate is 3 % shorter, which is what
// the estimates are good for, down to 1024 columns: they were fitted to 2048 and more, and below that
// are 5 % beside the pairs of 128 x 128 (1647 x 1152 x 7237, 3.3 % shorter as 224 x 256, took 50.6 us instead of
// 48.9).  One round of 224 x 256 over
// a long K is none: more compute units at once run at a lower clock, bf16 6000 x 4096 x 2048 96 us instead of
// 93, 2401 x 5120 x 4294 135 instead of 130.5, 11294 x 3520 x 1049 98.5 instead of 95.5, 2550 x 3648 x 4203 97.5
// instead of 99.5 (f16 operands of unfolded 4-bit weights, 5450 x 4352 x 2048 with their unfolding, 107
// instead of 111: not for these).
inline BlockChoice refine_block_tile(BlockChoice choice, uint32_t rows, uint32_t in_dim, uint32_t out_dim,
                                     uint32_t compute_units, bool bf16) {
    static constexpr BlockCost kCosts[] = {
        {BlockTile::Wide, 256, 288, 1800, 10500, 3600, 21000},
        {BlockTile::Seven, 224, 256, 1370, 8000, 2740, 16000},
        {BlockTile::Five, 160, 256, 1130, 5000, 2260, 10000},
    };
    if (in_dim < 1024) return choice;
    uint64_t bar = choice.ns - choice.ns * (in_dim < 2048 && choice.tile == BlockTile::Even ? 5 : 3) / 100;
    for (const BlockCost& c : kCosts) {
        const uint64_t tiles = static_cast<uint64_t>((rows + c.m - 1) / c.m) * ((out_dim + c.n - 1) / c.n);
        if (bf16 && c.tile == BlockTile::Seven && in_dim >= 3072 && tiles <= compute_units) continue;
        const uint64_t ns = block_ns(c, rows, in_dim, out_dim, compute_units);
        if (ns < bar) {
            choice = BlockChoice{c.tile, c.m, c.n, ns};
            bar = ns;
        }
    }
    return choice;
}
template <typename Element>
BlockChoice block_tile(uint32_t rows, uint32_t in_dim, uint32_t out_dim, uint32_t compute_units) {
    return refine_block_tile(choose_block_tile(rows, in_dim, out_dim, compute_units), rows, in_dim, out_dim,
                             compute_units, std::is_same<Element, __bf16>::value);
}
// The tiles a block product is launched with.  What bounds one is how the products of the two
// to four waves of a SIMD fill each other's waits, and the power (Large, 8192 x 4352 x 2048: matrix unit
// busy 64 % of the cycles, LDS reads 24 %, clock 1.9 GHz); units of
// 32 columns in a deeper ring, with a barrier each, were 6 to 20 % slower.  Measured, f16 operands:
//   Large  16384 x 2176 x 12352 / 9216, 8192 x 4352 x 2048: 763 / 553 / 110 us = 1.15 / 1.19 /
//          1.33 PFLOP/s.  Eight waves of 128 x 64: sixteen of 64 x 64 read a third more and were 2
//          to 5 % slower at every size (785 / 575 / 114; bf16 operands, 16384 x 2048 x 12352 /
//          9216 and 16384 x 4096 x 2048: 697 / 502 / 197 against 729 / 529 / 204)
//   Wide   2048 x 2176 x 9216, one round of 256 tiles: 71 us; Even 91, Large 112; 8192 rows 290, Large 313
//   Seven  2048 x 2176 x 12352: 109 us; Large 112, Wide 127; 3000 x 2176 x 9216 112, Large 119, Even 125
//   Five   777 x 2048 x 12352, one round of 245 tiles: 39.5 us; 4096 x 2176 x 12352 217, Large 243
//   Even   300 x 2048 x 12352: 26 us; Tall 33
//   Deep   2048 x 4352 x 2048: 38 us; Even 48, Large 81
//   Tall   100 x 2176 x 12352: 13.5 us; Deep 17, Small 20 (as 64 x 128, 19)
//          777 x 4352 x 2048: 24 us; Deep 30, Even 43
//   Small  300 x 4352 x 2048: 15 us; Least 20, Tall 22, Deep 29
//   Least  100 x 4352 x 2048: 11 us; Small 14, Tall 19, Deep 27
template <typename Element>
struct BlockTiles {
    typedef BlockProduct<Element, 256, 256, 2, 4> Large;      // the most products per byte fetched
    typedef BlockProduct<Element, 128, 128, 2, 4> Even;       // two a compute unit hide each other's waits
    typedef BlockProduct<Element, 128, 128, 2, 4, 4> Deep;    // one a compute unit, two units further ahead
    typedef BlockProduct<Element, 128, 64, 4, 2, 3> Tall;
    typedef BlockProduct<Element, 64, 64, 2, 2, 4> Small;
    typedef BlockProduct<Element, 32, 64, 2, 2, 4> Least;
    // where 256 x 256 leaves a round short: other heights and a wider one
    typedef BlockProduct<Element, 256, 288, 4, 2> Wide;
    typedef BlockProduct<Element, 224, 256, 2, 4> Seven;
    typedef BlockProduct<Element, 160, 256, 2, 4, 3> Five;

    // the tile a call takes, as use(product) of a value of its type
    template <typename Use>
    static auto choose(uint32_t rows, uint32_t in_dim, uint32_t out_dim, uint32_t compute_units, Use use) {
        switch (block_tile<Element>(rows, in_dim, out_dim, compute_units).tile) {
        case BlockTile::Even: return use(Even{});
        case BlockTile::Deep: return use(Deep{});
        case BlockTile::Tall: return use(Tall{});
        case BlockTile::Small: return use(Small{});
        case BlockTile::Least: return use(Least{});
        case BlockTile::Wide: return use(Wide{});
        case BlockTile::Seven: return use(Seven{});
        case BlockTile::Five: return use(Five{});
        default: return use(Large{});
        }
    }
    // use(product) of every tile, as long as it says true
    template <typename Use>
    static bool each(Use use) {
        return use(Large{}) && use(Even{}) && use(Deep{}) && use(Tall{}) && use(Small{}) && use(Least{}) &&
               use(Wide{}) && use(Seven{}) && use(Five{});
    }
};

// A launch: its workgroups, a persistent one per place on the device or one per tile, and the rounds of
// tiles that an XCD's workgroups take in runs.  Tiles are numbered down bands of eight tile rows (place):
// in a whole band the tile of a workgroup's own number gives an XCD one row of tiles, a good share by
// itself, in a lower band the rows shift from column to column.  So every round goes in runs where there is
// one lower band of many tiles, or a wide product over a long K (less wide below three whole bands);
// otherwise whole rounds of a multiple of eight workgroups do.  In runs and without, bf16, us:
//   777 x 2048 x 12352, one round of 5 x 49 tiles, 39.5 and 49.5     776 x 256 x 1119 (13 x 18) 5.5 and 5.1
//   1000 x 2048 x 9216 (7 x 36) 39.5 and 53                          3380 x 960 x 1083 (27 x 9) 18.7 and 17.3
//   300 x 2048 x 12352 (5 x 193) 25 and 32.5                         3144 x 1408 x 1189 (25 x 10) 21.5 and 21.0
//   2500 x 2048 x 9216 (20 x 72) 108 and 111                         11448 x 640 x 533 (90 x 5) 22.7 and 21.6
//   956 x 2304 x 572 (15 x 9) 10.3 and 10.8                          4431 x 3776 x 104 (70 x 2) 13.8 and 13.2
//   331 x 64 x 8988 (3 x 71) 5.0 and 5.4                             74 x 256 x 1023 (3 x 16) 3.85 and 3.70
struct BlockLaunch {
    uint32_t workgroups, runs;
};
template <typename Product>
BlockLaunch block_launch(uint32_t rows, uint32_t in_dim, uint32_t out_dim, uint32_t compute_units) {
    const uint32_t per_unit = 160 * 1024 / Product::kLdsBytes;
    const uint32_t m_tiles = (rows + Product::kTileM - 1) / Product::kTileM;
    const uint32_t n_tiles = (out_dim + Product::kTileN - 1) / Product::kTileN;
    const uint32_t places = compute_units * (per_unit < 2 ? per_unit : 2);
    const uint32_t workgroups = std::min(m_tiles * n_tiles, places);
    const bool low = m_tiles < 8 && m_tiles * n_tiles >= 128 && (in_dim >= 256 || Product::kTileN >= 128);
    const bool wide = m_tiles >= 8 && n_tiles >= (m_tiles < 24 ? 9 : 16) && in_dim >= 1024;
    const uint32_t rounds = low || wide ? kWholeRounds | kLastRound : workgroups % 8 == 0 ? kWholeRounds : 0;
    return {workgroups, rounds | workgroups % 8 << kRunsMore | workgroups / 8 << kRunsShare};
}

}  // namespace
}  // namespace tt
