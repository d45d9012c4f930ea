// Where a launch changes kernel by size: the rules that host tests check, in plain C++.  Times are microseconds of the
// launch alone on MI355X, buffers rotated.
#pragma once

#include <stdint.h>

namespace cq {

// The kernel of a transposed quantize whose runs are 16-byte aligned on both sides: the register kernel, the tile kernel
// with one step of columns per tile, or with 128 bytes of codes per row and tile.  `whole_tiles`, `steps`: how many tiles of
// either kind the launch has, batches included; `step_cols`: 64, or 128 for a fused abs-max over blocks of 128.
//
// From 1024 whole tiles on (two rounds of resident workgroups) those win.  Below:
// * Steps of 64 columns write a line of codes in pieces (of 16 bytes for 2-bit codes), the next piece of a line coming a
//   column of tiles later, so with many rows the line has left the L2 before it is full.  Fused abs-max, 2 bits of bf16
//   (steps, whole tiles, register kernel): [4096, 4096] 12.2, 14.6, 14.5, [8192, 2048] 13.7, 14.9, 14.8, [16384, 1024] 17.9,
//   15.0, 15.0, [14336, 2048] 24.8, 18.3, 23.4, [14336, 4096] 47.2, 31.7, 36.5; 4 bits [6144, 4096] 17.2, 14.5, 19.0,
//   [12288, 2048] 22.3, 15.4, 19.3, [14336, 1024] 14.5, 12.3, 14.5, [2048, 4096] 8.1, 9.8, 10.8, [1024, 28672] 18.9,
//   20.4, 23.2.
// * Given scales read them between the steps: 2 bits of bf16 [4096, 4096] 13.8, 19.8, 16.4, [8192, 2048] 17.0, 20.3, 15.9,
//   [14336, 1024] 13.9, 20.1, 15.7, [14336, 4096] 54, 44.2, 35.5; 4 bits [8192, 2048] 19.0, 17.0, 15.8, [14336, 1024] 17.4,
//   15.5, 15.8; wider codes and f32 gain from whole tiles all the same: 8 bits [6144, 2048] 13.8, 12.4, 15.9, 4 bits of f32
//   [12288, 1024] 19.7, 15.6, 17.2.
// * A step of 128 columns writes 32 bytes and more: 4 bits of bf16 [1056, 16384] 14.5, 16.8, 19.2, [14336, 2048] 22.0, 22.2, 23.1.
enum class TransposedTile { kRegisters, kStep, kWhole };
inline TransposedTile transposed_tile(uint32_t bits, uint32_t float_bytes, bool given_scales, uint64_t rows, uint64_t whole_tiles,
                                      uint64_t steps, uint32_t step_cols) {
    if (whole_tiles >= 1024) return TransposedTile::kWhole;
    if (step_cols == 128) return TransposedTile::kStep;
    const bool registers_keep_up = given_scales && float_bytes == 2 && bits < 8;
    const bool few_rows = !given_scales && rows <= 1280;
    if (!registers_keep_up && !few_rows && whole_tiles >= 512) return TransposedTile::kWhole;
    if (rows <= (given_scales ? 6144 : 8192) || steps <= 1536 || whole_tiles < 256) return TransposedTile::kStep;
    return given_scales ? TransposedTile::kRegisters : TransposedTile::kWhole;
}

// Whether the codes of whole tiles of a transposed quantize leave through plain stores instead of streaming ones (tiles of one
// step always take plain ones: their runs, shorter than a line, have to meet their neighbours' in the L2).
//
// After plain stores the codes are in the caches for the kernel that reads them next; the launch itself pays for that, and
// below 51 MiB moved that reader finds much of them there either way (streaming -> plain; the launch alone, with a re-pack
// behind it, with a dequantize behind it): 4 bits of bf16 [4096, 4096] 8 MB 11.8 -> 12.8, 17.3 -> 18.1, 23.2 -> 23.1; [4096,
// 5120] 10 MB 14.2 -> 15.2, 20.9 -> 21.6, 32.5 -> 28.9; [8192, 4096] 17 MB 21.6 -> 21.5, 29.2 -> 29.2, 42.9 -> 38.7; [14336,
// 4096] 29 MB 32.2 -> 33.4, 46.7 -> 42.9, 65.6 -> 59.3; 8 bits [4096, 4096] 17 MB 12.5 -> 13.6, 20.4 -> 20.6, 25.9 -> 24.0;
// [14336, 4096] 59 MB 38.4 -> 39.0, 58.9 -> 57.2, 79.9 -> 68.5; [16384, 8192] 134 MB 87.1 -> 86.8, 140 -> 140, 167 -> 153.
// Once codes and scales come near the 256 MB of the Infinity Cache they push themselves out, blocks of 32 (whose launches are
// the fastest) first: 8 bits [24576, 8192] 201 + 25 MB 127 -> 135, [28672, 8192] 235 + 29 MB 143 -> 175, 233 -> 255, 279 ->
// 259; 4 bits [28672, 8192] 117 + 29 MB 114 -> 119, 162 -> 158, 235 -> 226, [28672, 12288] 176 + 44 MB 174 -> 216, 353 -> 333;
// 2 bits [28672, 16384] 117 + 59 MB 204 -> 234.  Blocks of 64: 8 bits [28672, 8192] 235 + 15 MB 140 -> 145, 238 -> 226, 276 ->
// 252, [28672, 16384] 470 + 29 MB 298 -> 363, 504 -> 577.
inline bool transposed_codes_stay(uint64_t float_bytes, uint64_t code_bytes, uint64_t scale_bytes, uint32_t block) {
    const uint64_t kept = code_bytes + scale_bytes;
    return float_bytes + kept >= (51ull << 20) && kept <= (block <= 32 ? 152ull << 20 : 240ull << 20);
}

// Whether the tiles of a re-pack leave through plain stores instead of streaming ones.  `whole_lines`: the output's rows start on
// lines of 128 bytes.
//
// Rows that do not, cut a tile's runs into parts of lines, which have to meet their neighbours' in the L2 before they leave
// (streaming -> plain, us): 4 bits [4096, 14400] 17.8 -> 15.6, [1024, 117472] 51 -> 29, [8192, 28704] 103 -> 51.  Whole lines
// gain from plain stores only in the middle: 4 bits 8 MB 4.7 -> 5.7, 29 MB 13.3 -> 15.4, 34 MB 16.1 -> 16.6, 67 MB 29.9 -> 26.8,
// 84 MB 33.8 -> 31.9; 8 bits 17 MB 6.8 -> 7.9, 46 MB 19.1 -> 18.2, 67 MB 26.5 -> 24.9, 235 MB 84.9 -> 90.7.  Above, a quantize
// that left the codes in the caches and the output push each other out: 4 bits 117 MB 45.7 -> 41.9 alone, but both launches
// 158 -> 176; 8 bits 134 MB both 128 -> 135.
inline bool repack_stays(uint64_t bytes, bool whole_lines) {
    return !whole_lines || (bytes >= (32ull << 20) && bytes <= (96ull << 20));
}

// Whether a quantize with one scale per tensor keeps the tensor on the chip between its abs-max and its codes (one read and
// one launch, cq_kernels_resident.hpp) instead of reading it twice in two.  Small tensors gain the launch; from 8 chunks per lane
// on (16 MiB) the larger kernel's phases, with idle registers between them, cost more than a second read that the
// L2s and the Infinity Cache serve, until that read comes from memory again.  Narrower codes have less to write, and the arithmetic
// of the one pass, which nothing overlaps with, counts for more.  Two passes -> one, us: 8 bits of bf16 8 MiB 6.5 -> 6.3, 16 MiB
// 8.7 -> 8.1, 17 MiB 9.6 -> 9.6, 24 MiB 10.8 -> 10.9, 32 MiB 12.6 -> 12.7, 48 MiB 18.8 -> 17.3; of f32 16 MiB 8.0 -> 7.8, 32 MiB
// 11.4 -> 11.7, 48 MiB 17.4 -> 15.7; 4 bits of bf16 16 MiB 8.6 -> 8.2, 24 MiB 10.8 -> 11.1, 48 MiB 17.8 -> 17.9, 60 MiB 22.1 -> 21.4;
// e4m3 of f16 48 MiB 20.3 -> 20.1.
//
// Two bits of 16-bit floats have the least to write and lose until 128 MiB: bf16 56 MiB 20.0 -> 21.8, 80 MiB 26.9 -> 28.5, 112 MiB even, 128
// MiB 0.97 of the two.
//
// Captured launches need one more in front, which marks their slots: of 8 bits from 72 MiB on for 16-bit floats (f16 to e4m3 64 MiB 24.9 ->
// 26.3, 72 MiB 1.02 of the two; bf16 72 MiB 0.92), from 60 for f32 (64 MiB 26.1 -> 24.6), of narrower codes from 120 MiB (f16, 4 bits 100
// MiB 34.7 -> 36.2, 120 MiB 0.99) and 96 for f32 (2 bits 100 MiB 35.5 -> 32.7), not for two bits of 16-bit floats (f16 200 MiB 63.7 -> 68.0).
//
// What is beyond the chip's 128 MiB is read twice here too, by fewer waves than the two passes have, which cost more than the one read
// saves: past 384 MiB (captured 448) with a byte of codes for two of a tensor, past 768 MiB with one for four (8 bits of bf16 384 MiB 174 ->
// 154, 400 MiB 1.01 of the two, captured 448 MiB 177 -> 169, 4 GiB 1770 -> 1990; of f32 512 MiB 201 -> 171, 1 GiB 378 -> 377; 4 bits of bf16
// 512 MiB 201 -> 178, 1 GiB 380 -> 387).
inline bool quantize_stays_resident(uint64_t chunks, int bits, int float_bytes, bool captured) {
    constexpr uint64_t kMiB = 1 << 16;
    const bool f32 = float_bytes == 4;
    if (chunks > (bits == 8 && !f32 ? (captured ? 448 : 384) : 768) * kMiB) return false;
    if (captured) return bits == 8 ? chunks >= (f32 ? 60 : 72) * kMiB : f32 ? chunks >= 96 * kMiB : bits == 4 && chunks >= 120 * kMiB;
    return chunks <= 16 * kMiB || chunks >= (bits == 8 ? 48 : bits == 2 && !f32 ? 128 : 56) * kMiB;
}

inline uint32_t pow2_at_least(uint64_t v, uint32_t cap) {
    uint32_t p = 1;
    while (p < v && p < cap) p <<= 1;
    return p;
}

// Abs-max along an outer axis of a contiguous [outer, len, inner] tensor (cq_kernels_reduce.hip): the plan of slices and a fold, or
// one launch of tiles whose workgroups walk the whole axis, or a lane or wave per output (the kernel for any strides).  "->" below is from the former to the latter.
struct ReduceColumns {
    uint64_t outer, len, inner;  // elements
    uint64_t per_chunk;          // elements of a 16-byte chunk
    bool ragged;                 // rows that are not whole aligned chunks
    uint64_t tiles;              // workgroups of the plan's tiles before it cuts the axis; 0: the plan is a lane per chunk of columns
    bool long_axis;              // the plan wants slices, whatever the bytes of their partials
    uint64_t wanted, slices;     // slices that the plan wants, and what the workspace holds
};
// Chunk columns per tile of the one launch: a line of 128 bytes is eight of them, but fewer tiles than half of the compute units
// leave the others idle: 605 columns 4 (bf16 [1036, 4835] 4, 8: 8.3, 9.9), 832 - 2048 columns 8 ([4093, 11008] 4, 8, 16: 38.5,
// 19.1, 26.2), more 16 ([752, 19680] 4, 8, 16: 12.3, 11.1, 9.0).
constexpr uint32_t kWidestReduceTile = 16;
struct ReduceTile {
    uint32_t cw;
    uint64_t col_tiles;
};
inline ReduceTile reduce_tile(const ReduceColumns& c) {
    const uint64_t chunks = (c.inner + c.per_chunk - 1) / c.per_chunk, cols = c.outer * chunks;
    const uint32_t cw = pow2_at_least(chunks, cols >= 2200 ? kWidestReduceTile : cols >= 800 ? 8 : 4);
    return {cw, (chunks + cw - 1) / cw};
}

// Whether the workgroups of the one launch (512 lanes, four loads a lane in a trip) send out the next trip's loads before the last one's are
// folded (us, without -> with it): tiles of 16 columns with two to four trips, [404, 23360] 6.3 -> 5.7, [254, 33600] level, and of 8, which read whole lines where
// rows are whole lines, [829, 6976] 6.1 -> 5.5; half lines lose, [509, 10464] 5.4 -> 5.5.  More trips as long as no compute unit has a second tile, [666, 18112]
// 7.7 -> 6.9 ([602, 32896], 257 tiles, 9.7 -> 10.3), of 8 columns while every third has none: [1041, 9088] 6.5 -> 6.2 ([1134, 16384] 8.8 -> 9.3, [1082, 11776] 8.35 ->
// 8.5).  Not where there is nothing to load ahead, for ragged rows ([558, 9249] 6.95 -> 7.3, [5, 738, 3761] 10.15 -> 10.4), for narrower tiles, whose launches are small
// ([1116, 2307] 8.25 -> 8.6, f32 [1134, 115] 5.8 -> 6.1), nor past 896 tiles ([5, 138, 25216] 7.6 -> 8.3) or 1536 rows (bf16 [4093, 11008] 18.0 -> 18.7, [3726, 16384]
// 22.2 -> 24.2).  Over 1900 launches that it takes 1.03 times as fast on the mean, 0.97 at the least.
inline bool reduce_loads_ahead(const ReduceColumns& c, const ReduceTile& tile) {
    if (c.ragged || tile.cw < 8 || c.len > 1536) return false;
    const uint64_t tiles = c.outer * tile.col_tiles, trip = 4 * 512 / tile.cw;
    if (c.len <= trip || tiles > 896) return false;
    if (tile.cw == 8 && c.inner % (8 * c.per_chunk) != 0) return false;
    return c.len <= 4 * trip || tiles <= (tile.cw == 8 ? 160 : 256);
}

enum class ReduceWay { kPerOutput, kPlan, kOneLaunch };
inline ReduceWay reduce_way(const ReduceColumns& c) {
    const uint64_t cols = c.outer * ((c.inner + c.per_chunk - 1) / c.per_chunk), tiles = c.outer * reduce_tile(c).col_tiles;
    const bool f32 = c.per_chunk == 4;
    // Ragged rows, few elements per output: a workgroup per tile is mostly idle lanes and costs a large launch 1.5 ns each, a lane per
    // output 0.1 us per element of the axis, 0.2 of f32, or 1 ns per thousand elements of the tensor (tiles -> per output: f16 [34978, 9, 23]
    // 53.8 -> 5.9, [13557, 2, 125] 15.2 -> 6.1, bf16 [10812, 76, 11] 23.1 -> 10.2; [4485, 225, 11] 13.2 -> 22.9, f32 [7362, 85, 9] 10.6 -> 18.9, bf16 [3905, 8, 431] 9.4 ->
    // 14.6).  Below four elements (twelve in rows of less than 32 that are not f32) also against a lane per chunk, whose loads and
    // stores overlap and are not aligned (f16 [155, 2, 949] 2.7 -> 2.3, [620, 12, 11] 3.5 -> 2.9, f32 [200000, 3, 5] 5.7 -> 4.9), as
    // long as the launch is small (f32 [3038, 1, 365] 4.0 -> 4.7, [166490, 1, 11] 5.1 -> 6.6).
    if (c.ragged && !c.long_axis && c.len < 256) {
        if (c.len * (f32 ? 100 : 50) + 100 < c.tiles && c.outer * c.len * c.inner < c.tiles * 1800) return ReduceWay::kPerOutput;
        if (f32 ? c.len <= 4 && c.inner < 8 : c.inner < 32 ? c.len <= 12 : c.len <= 4 && c.outer * c.inner * c.len <= (1u << 19))
            return ReduceWay::kPerOutput;
    }
    // From 256 elements on an output has a wave, which for few of them ends before the tiles' 8 columns a lane have met (bf16
    // [631, 47] 4.0 -> 3.3, [325, 11] 3.4 -> 2.6, [901, 423] 3.6 -> 4.1; of f32, with 4, [452, 47] 2.2 -> 3.1).
    if (c.ragged && !f32 && c.len >= 256 && c.len <= 768 && c.outer * c.inner <= 1280) return ReduceWay::kPerOutput;
    // Without room for half of the slices, the columns alone are too few lanes (bf16 [43625, 2348] 4160 -> 158, [20000, 4097] 2133 -> 85,
    // [2000, 301] 36.5 -> 5.8, [4096, 4096] 394 -> 17.9).
    if (c.wanted > 2 * c.slices) return ReduceWay::kOneLaunch;
    // Tiles that want two slices and have room for one: they are wide, and few rows each (bf16 [2, 155, 128] 2.7 -> 2.9).
    if (c.slices < c.wanted && c.tiles != 0 && !c.ragged) return ReduceWay::kPlan;
    // An axis that is too short for slices is short for the plan's wider tiles too (f16 [15, 832] 1.8 -> 2.4, bf16 [20, 1640] 2.2 -> 2.5,
    // f16 [8, 24256] 2.0 -> 2.4, bf16 [212, 14, 799] 2.6 -> 4.5), except where a lane per ragged chunk would walk it (f32
    // [15, 11951] 2.7 -> 2.3).
    if (!c.long_axis && !(c.ragged && c.tiles == 0 && c.len > 8 && tiles <= 512)) return ReduceWay::kPlan;
    // A tile's lanes walk the whole axis, so its workgroup lasts len * cw / (4 * 512) loads' latency; a second launch costs about 4
    // us.  (Without a fold where the partials' bytes allowed one slice only, as in the first two.)
    //   f16 [115, 21256] 14.6 -> 4.1, bf16 [60, 30000] 8.7 -> 3.5, [337, 19272] 10.7 -> 6.2, [600, 8448] 10.5 -> 5.7, [1041, 9088]
    //   11.0 -> 6.8, [1036, 4835] 11.8 -> 8.3, f16 [391, 296] 6.3 -> 3.8, f32 [250, 32000] 9.9 -> 7.2, [83, 1184] 8.9 -> 3.0
    // Past 1280 rows the walk costs more than the fold (bf16 [2443, 4469] 12.2 -> 14.4, f32 [1468, 29424] 31.4 -> 33.9).
    if (tiles > 2048) return ReduceWay::kPlan;
    bool one = c.len <= 1280 && cols * c.len <= (1ull << 21);
    // Slices of few ragged rows cost more than those of whole chunks: f32 [1283, 115] 5.5 -> 3.0, [1748, 5] 5.0 -> 2.5, [2213, 61] 5.0 ->
    // 3.5, bf16 [1557, 1751] 8.5 -> 6.8, [1524, 9] 5.6 -> 4.1; f16 [2160, 73] 5.6 -> 6.5, f32 [2442, 501] 6.6 -> 9.0.
    if (c.ragged && c.len <= (f32 ? 2304 : 1920) && cols * c.len <= (1u << 19)) one = true;
    // Where rows are whole lines no tile reads half of one, and the walk may be longer, as long as the compute units without
    // a tile are few: they count for nothing in the one launch and read with the others in the plan's.  Calls in a row on
    // rotated buffers: 104 tiles bf16 [1600, 6656] 10.7 -> 9.7, [2048, 6656] 11.2 -> 11.0, [3000, 6656] 13.2 -> 15.1, f32 [1600, 3328] 9.1 ->
    // 9.2, [2048, 3328] 9.6 -> 10.7; 128 bf16 [2560, 8192] 13.7 -> 12.9, [3726, 8192] 15.5 -> 17.7, f32 [2400, 4096] 12.3 -> 12.0, [3000,
    // 4096] 13.4 -> 14.2; 144 and 160 [3000, 9216] 15.2 -> 15.1, [2400, 10240] 14.6 -> 14.8, [3000, 10240] 15.5 -> 17.5; 172 and more
    // [4093, 11008] 19.8 -> 18.3, f32 [4093, 5504] 18.5 -> 18.1, bf16 [4093, 14336] 24.2 -> 22.1, [3726, 16384] 27.0 -> 22.4; a second round
    // of a few, 274, [1281, 17536] 14.0 -> 12.0, [1600, 17536] 14.4 -> 14.9, [2560, 17536] 19.5 -> 21.3.
    // Tiles of 16 columns are twice the work each: up to 256 of them bf16 [2048, 20480] 18.2 -> 17.2, [2048, 32768] 26.4 -> 21.6; 272 [500, 34816]
    // 11.6 -> 10.0, [900, 34816] 15.1 -> 16.0; 384 [900, 49152] 19.5 -> 17.7; 512 [900, 65536] 24.7 -> 21.5.
    const uint32_t cw = reduce_tile(c).cw;
    if (!c.ragged && c.inner % (8 * c.per_chunk) == 0 && cw >= 8) {
        const uint64_t longest = cw == 8 ? (tiles < 128 ? 1700 : tiles < 171 ? 2400 : tiles <= 256 ? 4096 : 1400)
                                         : (tiles <= 256 ? 2048 : tiles <= 320 ? 768 : tiles < 512 ? 1152 : 2048);
        one = c.len <= longest && cols * c.len <= (1u << 23);
    }
    return one ? ReduceWay::kOneLaunch : ReduceWay::kPlan;
}

// A product with several vectors (cq_kernels_gemv_batch.hip): how many row groups share a workgroup's x, and how many waves share a
// row (kG x kS).  x comes from the L2 once per workgroup, so
// row groups together save L2 traffic; a launch wants a workgroup per compute unit and eight waves in each; and since
// the arithmetic bounds it, it ends with the compute unit that has the most row groups: with 600 of them, 1 x 4 leaves at most
// three on one, 2 x 4 four.  Measured on MI355X, us, kG x kS:
// * up to 256 groups, one to a compute unit: 1 x 8 as long as its LDS fits one (1 x 4, 1 x 8: e4m3 bytes, 112 groups, 9088 columns,
//   16 vectors 16.5, 11.7; 4 bits, 193 groups, 12288 columns, 12 vectors 13.6, 11.9; six stages 115 groups, 5 vectors 3.95, 3.69), but where
//   it leaves a compute unit one workgroup not for up to four stages, which are one round either way (4 bits, 148 groups, 10 units, 5 vectors
//   3.16, 3.52; 8 bits, 226 groups, 32 units, 12 vectors 2.92, 3.24), nor for the one round that it saves of 9 to 12 (117 groups, 91 units, 8
//   vectors 5.6, 5.9).
// * up to 512: 1 x 8 while two workgroups of it fit a compute unit's LDS, 80 KiB each; past that 1 x 4, but 2 x 4 for the widest x
//   (1 x 4, 2 x 4: 4 bits, 503 groups, 16 vectors 10.2, 7.4; 494 groups, 5 vectors 26.8, 29.2).
// * up to 1024: 4 x 2 for a wide x (2 x 4, 4 x 2: 4 bits, 990 groups, 16 vectors 9.1, 6.6; 661 groups, 12 vectors 9.2, 7.0), else 1 x 4 up to
//   768 (2 x 4, 1 x 4: 589 groups, 3 vectors 35.5, 28.9; 727 groups, 4 vectors 25.7, 22.1), 2 x 4 above (896 groups, 8 vectors 11.5, 12.7).
// * up to 1536: 1 x 4 for a narrow x, 2 x 4 for a middling one (4 x 2, 2 x 4, 1 x 4: 1416 groups, 2 vectors 79.7, 62.0, 58.4; 8 bits, 1306
//   groups, 16 vectors 155, 132, 146), not for rows of a few stages (1274 groups, 44 units 8.6, 9.2, 9.2) nor for e4m3 and e5m2 bytes,
//   which wait for memory (1200 groups, 7 vectors 29.4, 32.6, 34.7).
// * else 4 x 2 (4-bit bf16 [28672, 8192], 16 vectors 4 x 2, 2 x 4, 1 x 4 37.7, 49.6, 64.5).
enum class GemvShape { k1x8, k1x4, k2x4, k4x2 };
// `x`: bytes of a stage of x; lds_of_eight: of a workgroup of 1 x 8; `units` of a row, eight to a stage; `bytes`: e4m3 and e5m2
inline GemvShape gemv_batch_shape(uint32_t groups, uint32_t x, uint32_t lds_of_eight, uint32_t units, bool bytes) {
    const bool wide = x >= 6 * 1024;
    const uint32_t stages = (units + 7) / 8;
    const bool eight = (stages > 4 && stages <= 8) || stages > 12 || lds_of_eight <= 80 * 1024;
    if (groups <= 256) return eight && lds_of_eight <= 160 * 1024 ? GemvShape::k1x8 : GemvShape::k1x4;
    if (groups <= 512) return lds_of_eight <= 80 * 1024 ? GemvShape::k1x8 : lds_of_eight > 160 * 1024 ? GemvShape::k2x4 : GemvShape::k1x4;
    if (groups <= 1024 && !wide) return groups <= 768 ? GemvShape::k1x4 : GemvShape::k2x4;
    if (groups > 1024 && groups <= 1536 && !wide && units >= 48 && !bytes) return x <= 2 * 1024 ? GemvShape::k1x4 : GemvShape::k2x4;
    return GemvShape::k4x2;
}

// Whether such a product streams its codes past the caches: rows of whole lines of 128 bytes, and long rows of parts of them for twelve vectors and more where
// most compute units have one workgroup: its eight waves read a row's stages side by side, so that the parts of a line are asked for together, and x
// takes more of the caches (plain loads -> streaming, us, 16 vectors: 8 bits [3507, 10944] 19.4 -> 16.7, [3449, 16736] 28.2 -> 24.8, e2m1 bytes [3522,
// 22400] 30.0 -> 25.8; on the mean of 16 products 1.06 times as fast, of 34 with fewer vectors level, of rows of 7 to 9 kB or less 0.95, of up to 160
// groups 0.94).
inline bool gemv_batch_streams(bool whole_lines, uint32_t groups, uint64_t row_bytes, uint32_t vectors) {
    return whole_lines || (groups > 176 && groups <= 256 && row_bytes >= 9000 && vectors >= 12);
}

// A product with one to four vectors by gemv_quads_kernel (cq_kernels_gemv_quads.hip), whose workgroups, one per compute unit, take four
// rows a wave from x in LDS: whether it does, its workgroups and waves, and how many waves share four rows.  With `work`, the most steps (16
// units of four rows) that a workgroup has, us before (gemv_stream_kernel, gemv_batch_kernel) -> with it:
// * Several vectors: against the units that the busiest compute unit goes through there, in groups of 16 rows and stages of eight units.  Under
//   0.7 of them always ([1163, 23392] 8 bits, 2 vectors 26.4 -> 12.5, [4444, 10272] 4 bits of bf16, 4 16.1 -> 11.6, [4115, 5120] 7.7 -> 7.1;
//   0.79 [2856, 4864] 5.7 -> 5.9, 0.83 [3454, 1920] 4.05 -> 4.18), from work 64 on under 0.8 ([9559, 1952] f16 8 bits, 3 vectors
//   0.83 6.75 -> 7.45), from 128 on under 0.92 ([14336, 4096] 0.88, 8 bits 14.4 -> 13.3,
//   e4m3 13.6 -> 12.4; 1.0 [16384, 5120] 8 bits 17.0 -> 18.2, [15872, 1280] e4m3 6.1 -> 6.6), and where fields of 4 bits fill the chip (from work 128, of
//   f16 from 64) as long as it is any less ([23373, 10080] 0.96 40.4 -> 38.1, [21782, 7552] 26.3 -> 22.9; at work 112 0.88 [14336, 4096] 10.2 -> 10.5).
//   Not where waves are left without rows that the other has a round of for each: 4 bits, two four-row groups of three or four steps
//   on a compute unit (2 vectors [1693, 1920] 3.68 -> 3.83, 4 [1362, 1920] 3.68 -> 3.90; two steps [1024, 2048] 3.66 -> 3.36, five [1085, 2080] 4.31 -> 3.88), and
//   short rows of 8 bits in five groups of four rows for eight waves or pairs of waves ([5120, 1024] 2 vectors 4.33 -> 4.58, e4m3 3.98 -> 4.50,
//   [4608, 3456] 3 6.85 -> 7.65; 8 bits [5120, 3072] 4 7.15 -> 6.68, e4m3 [4736, 5504] 3 8.94 -> 8.34).
//   Rows of whole lines, which gemv_batch_kernel streams: 4 bits of bf16 and e2m1 bytes gain 1.05 times on the mean where others gain 1.15, and
//   lose with three and four vectors on two groups of four, six or eight steps (e2m1 bytes [2048, 4096] 4.80 -> 5.17; five and seven, and two vectors, 1.05 times as
//   fast), on more of up to six ([5120, 2048] 3 4.87 -> 5.21, [19754, 1024] 6.51 -> 6.97), fields on nine and more of work 64 to 128, and on three of long rows with
//   more than two vectors ([9435, 5120] 3 10.3 -> 11.0, [2863, 14080] 4 10.2 -> 11.3; six groups 1.04), and from work 128 on where they leave one or two of
//   sixteen waves without a group, 14 and 15 (0.97 on the mean of 237, [14336, 8192] 4 18.6 -> 19.9, [14336, 14336] 28.1 -> 30.1; [11008, 11008] 1.04 and [28672, 8192] 1.05).
//   e4m3 and e5m2, where the other is nearer to memory's rate: not in two groups of four steps ([2048, 1024] 3.53 -> 3.82), from 0.8 of the units on not for very short
//   and very long rows ([28672, 2048] 12.3 -> 13.2, [14336, 14336] 34.8 -> 37.4; [28672, 4096] 1.15, [28672, 11008] 1.25 times as fast, long ones in eight to
//   thirteen groups 1.09, [9728, 23936] 46.7 -> 39.8) nor where a wave or two have four rows
//   ([25344, 1664] 10.5 -> 11.4, [6784, 7040] 11.3 -> 12.2): all waves in other rows ask the same channels.
// * One vector, 4 bits of f16: the digits pair up without being shifted together (x is permuted on its way into LDS;
//   [18484, 6912] 23.3 -> 17.5, [7455, 2240] 7.3 -> 5.7), except in the smallest launches that fill the other's strips as well ([1514, 1280] 3.21 -> 3.42,
//   [1814, 1792] 3.35 -> 3.70; work 9 [2347, 1408] 3.85 -> 3.64, 12 [3425, 1344] 4.13 -> 3.74) or have four steps ([1024, 2048] 3.43 -> 3.64; eight [1024, 4096] 1.04).
// * One vector of e4m3 and e5m2 bytes, which leave time beside the arithmetic: from work 64 on ([9472, 18176] 32.6 -> 30.2, [4352, 24448] 28.9 ->
//   22.8; [5888, 1664] 5.3 -> 5.7), but up to 128 not with three to six groups of four rows on a compute unit, whose waves, two to four to a group, start and
//   end more often than they step ([4736, 4352] 7.46 -> 8.23, [5120, 4096] 6.60 -> 7.37, [3968, 4992] 6.27 -> 6.79; two [2048, 14592] 1.17 and eight [8576, 3328] 1.07
//   times as fast), and up to 512 not with six or ten in few strips ([9856, 1664] 6.03 -> 7.35, 0.96 and 0.98 times as fast on the mean of 99; nine and eleven 1.03, 1.05).  The waves go through their rows in step, so they ask the same channels of memory at a time where those rows lie apart by
//   the wrong distances: a compute unit's share a multiple of 2^18 bytes ([8192, 8192] 14.5 -> 15.3, [16384, 8192] 24.7 -> 27.2, [24576, 8192] 35.0 -> 42.3),
//   and others ([14336, 11008] 31.1 -> 34.7, [28672, 10624] 51 -> 55; [28672, 10496] 52 -> 50, [20480, 11008] 42.5 -> 38.4).  From work 512 on, where the other
//   kernel is near memory's rate, only where that one's strips and workgroups are filled badly ([5120, 28672] 32.5 -> 26.5, [6144, 24576] 29.1 -> 26.5) or eight
//   and more waves share four rows, or four of up to eleven groups ([9216, 16128] 30.1 -> 26.7, [11008, 14336] 30.5 -> 28.1; 1.03 times as fast on the mean of 229; the
//   others of four waves and fewer 0.99).
// * Else one vector is bound by the same instructions either way, and it takes the launch where the other's strips of 64 units and workgroups
//   of 8 or 16 rows are filled badly: four-row steps of 16 units under 0.72 of what its busiest compute unit goes through ([4524, 16512] 18.2
//   -> 14.6, [1024, 28672] 14.9 -> 8.4, [25471, 2240] 14.4 -> 11.8, [2675, 4672] 6.1 -> 5.6; 0.77 [6867, 3584] 6.7 -> 7.3), not in the
//   smallest launches ([3011, 1408] 3.8 -> 4.0); 8 bits and e2m1 bytes, with fewer steps in a row, under 0.55 up to work 48 (0.62 [2774, 2432] 5.05 -> 5.30, 0.66
//   [2583, 3360] 5.38 -> 5.63, e2m1 0.62 [4120, 4320] 6.49 -> 6.71; 0.5 [1024, 8192] 6.49 -> 5.28).
//   Of eight waves with a group each not for five groups or nine, of bf16 ([4708, 1152] 8 bits 4.62 -> 5.21, [4959, 3072] 4 bits 5.59 -> 6.13; seven 1.07, ten
//   1.03 times as fast).
// Eight waves where there is little for sixteen to do: work 28 [7455, 2240] f16 5.7, 6.1 of 16; 64 [16115, 1920] 7.9, 7.3; 96 [4352, 24448]
// 30, 22.8.  Shares of four rows are the fewest steps for the busiest wave, a quarter of one for each sum of its lanes.
//
// Over 3400 launches from [1024, 1024] to [28672, 28672] that it takes it is 1.18 times as fast as the others on the mean; 2 % are more than 2.5 % slower, e4m3 the
// most ([13568, 9984] 4 vectors 24.8 -> 27.3, one [4224, 6656] 9.1 -> 10.0).
struct QuadsSplit {
    uint32_t grid, waves, shares_log2, lds;  // grid 0: the other kernels
};
// rows of `units` units of `values` values; `fields4`: fields of 4 bits; `f16`: x is; `bytes`: e4m3 and e5m2
inline QuadsSplit quads_split(uint32_t rows, uint32_t units, uint32_t values, uint32_t vectors, bool fields4, bool f16, bool bytes) {
    constexpr uint32_t kComputeUnits = 256, kMostQuads = 64, kMostLds = 160 * 1024;
    constexpr QuadsSplit kNo = {0, 0, 0, 0};
    const uint64_t x_bytes = (static_cast<uint64_t>(units) + 15) / 16 * 16 * values * 2 * (vectors > 2 ? 4 : vectors);
    if (vectors > 4 || x_bytes > kMostLds) return kNo;
    const uint32_t quads = rows / 4 + (rows % 4 != 0), steps = (units + 15) / 16;
    QuadsSplit q = {quads < kComputeUnits ? quads : kComputeUnits, 16, 0, 0};
    while ((quads + q.grid - 1) / q.grid > kMostQuads) q.grid *= 2;
    const uint32_t each = (quads + q.grid - 1) / q.grid;
    const uint64_t work = static_cast<uint64_t>(quads + kComputeUnits - 1) / kComputeUnits * steps;
    const bool lines = units % 8 == 0;  // rows of whole lines of 128 bytes
    bool full = false;                  // the other kernels go through little more
    if (vectors > 1) {
        const uint32_t stage = (vectors * 16 * values + 1023) / 1024 * 1024, groups = rows / 16 + (rows % 16 != 0);
        const GemvShape shape = gemv_batch_shape(groups, stage, 16 * (stage + 2560), units, bytes);
        const uint32_t together = shape == GemvShape::k4x2 ? 4 : shape == GemvShape::k2x4 ? 2 : 1;
        const uint64_t busiest = static_cast<uint64_t>((groups + together - 1) / together + kComputeUnits - 1) / kComputeUnits * together * 16 * ((units + 7) / 8) * 8;
        const uint32_t most = work < 64 ? 70 : !fields4 ? (work < 128 ? 80 : 92) : f16 || work >= 128 ? 99 : 85;
        if (work * 64 * 100 >= busiest * most) return kNo;
        const auto at_least = [&](uint32_t percent) { return work * 64 * 100 >= busiest * percent; };  // ... of what the other goes through
        if (values == 32) {
            if (each > 1 && steps > 2 && work <= 8) return kNo;
            if (lines && !(fields4 && f16) && (each == 2 ? vectors > 2 && steps > 2 && steps <= 8 && steps % 2 == 0 : each >= 5 && steps <= 6 && work < 64)) return kNo;
            if (lines && fields4 && !f16 && work >= 64 && work < 128 && at_least(75) && (each >= 9 || (each == 3 && vectors > 2 && steps < 32))) return kNo;
            if (lines && !(fields4 && f16) && work >= 128 && at_least(85) && (each == 14 || each == 15)) return kNo;
        } else if (each == 5 && work < (bytes ? 96 : 48)) {
            return kNo;
        }
        full = at_least(80);
        if (bytes && ((each == 2 && steps == 4) || (full && !at_least(90) && (steps < 10 || (steps >= 50 && (each < 8 || each >= 14)))))) return kNo;
    } else {
        const uint32_t group = static_cast<uint64_t>(units) * values >= 16384 ? 16 : 8, groups = rows / group + (rows % group != 0);
        const uint64_t stream = static_cast<uint64_t>((units + 63) / 64) * 64 * group * ((groups + kComputeUnits - 1) / kComputeUnits);
        const auto at_least = [&](uint32_t percent) { return work * 64 * 100 >= stream * percent; };  // ... of what the other goes through
        if (bytes) {
            const bool apart_by_2_18 = static_cast<uint64_t>(rows) * units % (1u << 22) == 0;  // 256 shares of units of 16 bytes
            if (work < 64 || (work < 128 && each > 2 && each <= 6) || (at_least(85) && (apart_by_2_18 || (work < 512 && (each == 6 || each == 10))))) return kNo;
            full = work >= 512 && at_least(85);
        } else if (fields4 && f16) {
            if (work <= 8 && (at_least(72) || (each == 1 && steps <= 4))) return kNo;
        } else {
            if (work < 24 || at_least(72) || (!fields4 && work < 48 && at_least(55))) return kNo;
        }
    }
    if (work < (vectors > 1 ? 32 : 48)) q.waves = 8;
    uint64_t least = ~0ull;
    for (uint32_t l = 0; (1u << l) <= q.waves; l++) {
        const uint64_t slots = q.waves >> l, cost = (each + slots - 1) / slots * (4 * ((static_cast<uint64_t>(steps) + (1u << l) - 1) >> l) + 1);
        if (cost < least) q.shares_log2 = l, least = cost;
    }
    if (vectors > 1 ? bytes && (q.shares_log2 == 0 || (q.shares_log2 == 1 && full))
                    : bytes ? full && q.shares_log2 < (each < 12 ? 2u : 3u) : !f16 && q.shares_log2 == 0 && (each == 5 || each == 9)) return kNo;
    const uint64_t lds = x_bytes + (each << q.shares_log2) * 64;
    if (lds > kMostLds) return kNo;
    q.lds = static_cast<uint32_t>(lds);
    return q;
}

// Blocks over two dimensions, scale computed in the launch: whether quantize_block_tiles_kernel takes it (cq_kernels_rows.hip; per_lane 0:
// no), its lanes along the row, and how many chunks of a block's column each lane would hold in a workgroup of 256.  Blocks of a few rows are one chunk a lane, and a large launch of those waits for its many
// small workgroups to be dispatched (1.1 - 1.7 ns each): from kWideTileChunks on their tiles are wider, two or four chunks a lane.
// quantize_blocks_kernel, one chunk, wider, us: 8 x 128 bf16 [736, 7808] 6.2, 7.2, 3.9, 8 x 32 [8880, 4800] 24.3, 37.2, 20.0, 16 x 64 f16
// [67136, 2048] 73.7, 112, 61.6, f32 [17392, 1728] 29.2, 33.0, 23.9.  Where blocks have four rows, or rows no room for 64 lanes, that is
// the first of them's: 8 x 32 f16 [103208, 320] 29.2, 42.9, 4 x 128 bf16 [44832, 768] 26.9, 38.1, f32 [2984, 9344] 25.1, 29.9 (but [7864, 4864]
// 53, 40); smaller ones of f32 are faster here, [30360, 256] 19.6, 9.0, unless the tiles are less than three quarters full ([310176, 80] 38.8, 43.4).
constexpr uint64_t kWideTileChunks = 5u << 17;
struct BlockTiles {
    uint32_t per_lane, tj_log2, cpb_log2;
};
// blocks of `br` rows by `cpb` chunks, `rows` rows of `row_chunks`
inline BlockTiles block_tiles_of(bool f32, uint32_t br, uint32_t cpb, uint64_t rows, uint32_t row_chunks) {
    constexpr uint32_t kLanes = 256;
    constexpr BlockTiles kNo = {0, 0, 0};
    if (br == 0 || cpb == 0 || (br & (br - 1)) != 0 || (cpb & (cpb - 1)) != 0 || cpb > 64 || rows / br > 65535) return kNo;
    uint32_t cpb_log2 = 0, tj_log2 = 0;
    while ((1u << cpb_log2) < cpb) cpb_log2++;
    while ((1u << tj_log2) < cpb || tj_log2 < 4 || (br << tj_log2) < kLanes) tj_log2++;
    const uint64_t chunks = rows * row_chunks;
    if (chunks >= kWideTileChunks && (br << tj_log2) == kLanes)
        while (tj_log2 < 6 && (br << tj_log2) < 4 * kLanes && row_chunks >= (2u << tj_log2)) tj_log2++;
    if (tj_log2 > 6 || row_chunks < (1u << tj_log2) || (br << tj_log2) > 4096) return kNo;
    const uint32_t per_lane = (br << tj_log2) / kLanes;
    const bool filled = row_chunks * 4 >= ((row_chunks + (1u << tj_log2) - 1) >> tj_log2 << tj_log2) * 3;
    if (per_lane == 1 && chunks >= (f32 && filled ? 6u << 20 : 3u << 18)) return kNo;
    return {per_lane, tj_log2, cpb_log2};
}

// Quantize and dequantize lane by lane (cq_kernels_flat_launch.hpp): tiles of one step, a chunk per lane, for launches of fewer chunks.  There a tile of four steps is a few
// workgroups' serial work, every step with a walk of its own over the levels.  Quantize and dequantize, us, tiles of several steps
// and of one: f16 [16, 8, 3, 128] behind permuted dimensions 8.3 and 5.2, 120 tokens 9.5 and 6.7, 250 (512 000 chunks) 10.4 and 9.7,
// 500 14.3 and 14.2; 4 bits of bf16 [16, 8, 500, 80] (640 000) 13.5 and 12.4, 1200 tokens 19.2 and 19.4, [20, 4, 980, 128] 14.5 and
// 15.0; runs of 4 bits, blocks of 16, [1024, 1024] 7.4 and 5.0, [4096, 1024] 9.5 and 8.0; of 8 bits, blocks of 24, [2048, 1536] 8.3
// and 8.1, [4096, 1536] (786 432) 11.3 and 11.6.  Blocks that are no power of two of lanes lose earlier: of 48 f32 565 248 chunks 7.7 and
// 8.3, f16 479 232 11.4 and 12.1, of 24 f16 639 744 8.6 and 9.5, bf16 314 880 7.3 and 6.5.
// `any_group`: lanes per block that are no power of two, else 0
inline uint64_t small_lane_chunks(uint32_t any_group) { return any_group != 0 ? 7u << 16 : 3u << 18; }
// The same for the scales alone, lane by lane, which have nothing to write: of f32 behind permuted dimensions, blocks of 32, 409 600 chunks 3.7
// and 2.7, 598 016 3.6 and 3.9, 778 240 3.7 and 4.5 us.
constexpr uint64_t kSmallLaneScaleChunks = 1u << 19;

}  // namespace cq
