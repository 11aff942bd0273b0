// Rules that choose a launch's shape from a call's sizes.  Host logic only; no HIP calls.  (A constexpr function is
// device code's as well.)
#pragma once

#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace qmm {

// ---- MXFP4, 17 fp32 rows and more: tiles whose steps of K workgroups share --------------------------------------
// Tiles of `rows` x `columns`, `tiles` of them; the (tile, step) units go to `groups` workgroups.  groups 0: not shared.
struct SharedTiles {
  uint32_t rows = 0, tiles = 0, groups = 0, columns = 256;
};
// First of the units of workgroup g.
constexpr uint64_t unit_bound(uint32_t g, uint32_t groups, uint32_t tiles, uint32_t steps) {
  return static_cast<uint64_t>(g) * (static_cast<uint64_t>(tiles) * steps) / groups;
}
// The workgroup that holds unit v: the last whose bound is not above it.
constexpr uint32_t unit_owner(uint64_t v, const SharedTiles& plan, uint32_t steps) {
  uint32_t g = static_cast<uint32_t>(v * plan.groups / (static_cast<uint64_t>(plan.tiles) * steps));
  while (g + 1u < plan.groups && unit_bound(g + 1u, plan.groups, plan.tiles, steps) <= v) ++g;
  return g;
}
// The piece of tile t that workgroup g holds is block g + t: along the units one of the two grows from piece to piece.
constexpr size_t shared_tiles_bytes(const SharedTiles& plan) {
  return plan.groups == 0u ? 0 : (static_cast<size_t>(plan.groups) + plan.tiles - 1u) * plan.rows * plan.columns * 4u;
}
// Rows a tile: the padding it takes decides.  Workgroups: as many as the chip holds, at least four units each.
// Tiles are shared where whole ones, small (128 x 64) or 256 x 256, leave much of the chip idle for long.  Sides measured
// (us, whole / shared): 17 rows of 6144 x 5120 57 / 42, 100 rows 69 / 54, 453 rows of 17408 x 5120 238 / 190, 1024 of 5120 x
// 17408 591 / 349, 640 of 4096 x 2048 55 / 48; but 2048 of 6144 x 5120 (192 tiles) 254 / 262, 1500 of 4000 x 1792 (14 steps)
// 73 / 83, 20 of 520 x 1024 19 / 21: the pieces cost a launch and twice their bytes, 64 MB of 256-row tiles where the chip
// is full of them.  With few steps that is more than small tiles lose which fill a round of a workgroup a CU, or of two:
// 256 rows of 2048 x 2048 34 / 45, 128 of 8192 x 2048 (128 small tiles) 33 / 38, but of 1024 x 2048 (16) 33 / 32, 512 of 8192
// x 2048 (512) 58 / 60, 512 of 4096 x 4096 (32 steps, 256 small tiles) 61 / 66, but 256 (128) 59 / 53.
constexpr SharedTiles shared_tiles(uint64_t m, uint64_t n, uint64_t steps, uint64_t cus) {
  if (m > 256 * cus || n > 256 * cus || steps < 16) return {};
  const uint64_t rows = m <= 64 ? 64 : (m + 127) / 128 * 128 < (m + 255) / 256 * 256 ? 128 : 256;
  const uint64_t tiles = (m + rows - 1) / rows * ((n + 255) / 256), small = (m + 127) / 128 * ((n + 63) / 64);
  if (tiles * 8 > cus * 5) return {};
  if (steps < 32 && rows == 128 && small <= cus && small * 8 > cus) return {};
  if (steps < 32 && rows == 256 && small <= 2 * cus) return {};
  if (steps < 40 && small * 8 >= cus * 7 && small <= cus) return {};
  const uint64_t room = cus * (rows == 64 ? 2 : 1), most = tiles * steps / 4;
  return {static_cast<uint32_t>(rows), static_cast<uint32_t>(tiles), static_cast<uint32_t>(room < most ? room : most)};
}

// ---- Q4_K, Q5_K and Q6_K on the tensor tile: tiles whose super-blocks workgroups share -----------------------------------
// Tiles of 128 x 128 whose (tile, super-block) units go to one workgroup a CU, at least two units each.  Whole tiles of
// 128 x 64 leave most CUs idle while a few walk all of K: 512 rows of 1024 x 5120 are 64 of them.  The pieces cost a launch
// and twice their bytes, so that with few super-blocks, or tiles that fill the chip, whole ones lead; `small` counts those, and
// the limits are sixteenths of the CUs.
// Q4_K, sides measured (us, whole / shared; rows x n x k, in brackets the small tiles).  `even`: every workgroup has as many
// units; otherwise some take two tiles' pieces, which counts where a tile has few; with several row tiles sharing leads
// all the same (500 x 1728 x 3072 (108) 30.6 / 28.9, 1000 x 1728 x 4096 (216) 40.8 / 39.1).  100 x 4096 x 2048 (64) 20.9 / 19.5, x 2304 22.6 /
// 23.6, x 2816 25.7 / 25.3; 100 x 5696 x 3072 (89) 27.4 / 27.6, x 6912 (108) 27.5 / 29.2, x 8192 (128, even) 27.4 / 26.3; 128 x 13888 x
// 4352 (217) 37 / 40, 256 x 8192 x 4096 (256, even) 38 / 36; 512 x 1024 x 5120 (64) 44 / 26, 512 x 6144 x 5120 (384) 64 / 59, 2048 x
// 6144 x 5120 (1536) 183 / 220; 256 x 5120 x 17408 (160) 126 / 84, 1024 (640) 316 / 267, 2048 (1280) 452 / 492.  Four row tiles and
// more whose small tiles fill two a CU: 500 x 7168 x 6144 (448) 76 / 82, but 256 x 14336 (448) 76 / 72, 500 x 8704 (544) 115 / 87.
// Up to 64 rows whole tiles are of 32 columns and 32 or 64 rows, with no padding, and start to take longer with more than a round of
// them: 17 rows of 2048 x 2048 (32) 14.6 / 15.1, 5120 x 3072 (80) 18.9 / 17.9, 6144 x 3072 (96) 18.9 / 20.7, 8192 x 5120 (128) 27.8 / 23.7,
// 10240 x 5120 (160) 29 / 30, 17408 x 5120 (272) 29.5 / 40, 12288 x 8192 (192) 43 / 41, 5120 x 17408 (80) 82 / 40; 64 rows of 4096 x
// 2048 (64) 18.7 / 16.8, 6144 x 3072 (96) 24.7 / 23.3, 7168 x 3072 (112) 24.8 / 25.5, 12288 x 4096 (192) 32 / 30.5, 14336 x 4096 (224) 32.4 /
// 32.7, 16384 x 5120 (256) 38 / 36, 20480 x 5120 (320) 39 / 46.
constexpr uint64_t shared_q4k_limit(uint64_t m, uint64_t steps, bool even) {
  if (m <= 32) return steps < 10 ? 0 : steps < 12 ? 2 : steps < 16 ? 4 : steps < 18 ? 6 : steps < 24 ? 8 : steps < 32 ? 10 : steps < 48 ? 12 : 14;
  if (steps < 12) return steps == 9 ? 3 : 4;
  if (m <= 64) return steps < 16 ? 6 : steps < 20 ? 12 : 16;
  if (steps < 16) return steps == 12 && m <= 256 && !even ? 5 : 8;
  return steps < 18 && m <= 384 && !even ? 12 : steps < 20 ? 16 : 40;
}
// Q5_K and Q6_K, whose whole tiles need no decode and go up to 256 x 256: 100 x 512 x 2048 (8) 22 / 19, 24 x 6144 x 2048 (96) 28 /
// 33; 200 x 2048 x 3072 (64) 33 / 28, 24 x 4096 x 3072 (64) 32 / 33, 384 x 4096 x 3072 (192) 36 / 38; 512 x 1024 x 5120 (64) 46 / 28,
// 512 x 6144 x 5120 (384) 80 / 79, 200 x 6144 x 5120 (192) 57 / 59; 512 x 3072 x 8192 (192) 66 / 75.
constexpr uint64_t shared_kquant_limit(uint64_t m, uint64_t steps) {
  return (steps < 12 ? 2 : steps < 16 ? 4 : steps < 20 ? 6 : 8) / (m <= 32 && steps < 20 ? 2 : 1);
}
constexpr SharedTiles shared_f16_tiles(uint64_t m, uint64_t n, uint64_t steps, uint64_t cus, bool q4k) {
  if (m > 256 * cus || n > 256 * cus || steps < 8) return {};
  const uint64_t tiles = (m + 127) / 128 * ((n + 127) / 128), small = (m + 127) / 128 * ((n + 63) / 64);
  if (small * 16 > cus * (q4k ? shared_q4k_limit(m, steps, tiles * steps % cus == 0) : shared_kquant_limit(m, steps))) return {};
  if (q4k && m > 384 && steps < 48 && small * 2 > cus * 3 && small <= 2 * cus) return {};
  const uint64_t units = tiles * steps / 2;
  return {128, static_cast<uint32_t>(tiles), static_cast<uint32_t>(cus < units ? cus : units), 128};
}

// ---- "ffn_gate_up_silu_q4k", more than 64 rows ----------------------------------------------------------------------
// Tiles of 256 rows and 128 columns of either matrix, from column 0 on; what they leave goes to tiles of 128 rows and 64.
// As in the single product, whole rounds of a tile a CU, and none where they fill less than half the chip.  Nor with 128
// rows or fewer, half of each tile being padding (us, small tiles / 256-row tiles, in brackets as two products: 17408 x 5120
// 103 / 138 (117)), nor with 257 to 384, half of the second ones, unless they fill three quarters of a round or all of it: 300
// rows of 17408 x 5120 (136 tiles) 209 / 233 (287), of 8192 x 4096 (64) 88 / 113 (107), of 12288 x 2048 (192) 74 / 70.
constexpr uint32_t gate_up_large_tiles(uint32_t m, uint32_t n, uint32_t cus) {
  const uint32_t tiles_m = (m + 255u) / 256u, tiles_n = (n + 127u) / 128u, tiles = tiles_m * tiles_n;
  if (m <= 128u || (m > 256u && m <= 384u && (tiles * 4u < cus * 3u || tiles > cus))) return 0;
  if (tiles > cus && tiles % cus != 0 && tiles % cus <= cus / 2) return tiles / cus * cus / tiles_m;
  return tiles < cus / 2 ? 0 : tiles_n;
}

// ---- Q5_K and Q6_K from 17 rows: both operands to fp16 -------------------------------------------------------------------
// RowsFirst: one launch, the rows' workgroups first.  RowsLast: the weights' first, so that the product finds the rows' copy where
// it was left last.  RowsTwice: rows first and read twice, since a row of more than 6144 held in registers leaves five wavefronts a
// SIMD also to the weights, where Q5_K's decode wants eight.  Apart: the weights, then the rows in a launch of their own.
// Sides measured in a whole feed forward of Q4_K gate and up with silu and this product (us, rows x hidden x inter).  Q6_K, first /
// last: 256 x 5120 x 17408 373 / 382 (the product alone, called again and again, 168 / 219), 512 534 / 536, 1024 812 / 783,
// 2048 x 4096 x 11008 708 / 672; but 2048 x 5120 x 6400 528 / 542, 1024 x 4096 x 8192 282 / 284, and the product of 2048 x 5120 x 5120
// 135 / 138.  Q5_K, first / twice / apart: 100 x 5120 x 17408 244 / 232 / 235, 256 375 / 380 (the product 168 / 213), 384 464 / 453 (186 /
// 230), 1024 838 / 834 / 799, 2048 x 4096 x 11008 716 / 725 / 685, 2048 x 5120 x 6400 537 / 542 / 548; the product of 33 x 24576 x 17408
// 693 / 638 / 638, of 512 x 24576 x 8192 409 / 381 / 378, of 33 x 512 x 12288 31.0 / 31.7 / 34.1: twice where the weights are most of it.
enum class KquantOperands { RowsFirst, RowsLast, RowsTwice, Apart };
constexpr KquantOperands kquant_operands(uint32_t m, uint32_t n, uint32_t k, uint32_t bits) {
  if (k <= 6144u || (bits == 6u && (m <= 512u || k <= 8192u))) return KquantOperands::RowsFirst;
  if (bits == 6u) return KquantOperands::RowsLast;
  if (m > 512u && k >= 8192u) return KquantOperands::Apart;
  return n >= uint64_t{24} * m ? KquantOperands::RowsTwice : KquantOperands::RowsFirst;
}

// ---- Q5_K and Q6_K from 17 rows: fp16 weights, decoded by the launch before ----------------------------------------------
// `large` tiles of 256 rows and `columns` columns, from column 0 on, for each 256 rows; the columns they leave go to tiles of
// 128 x 64.  Whole rounds of 256 columns, a tile a CU, and none where they fill less than half the chip.  Where the columns
// fit one round of narrower ones, the narrowest with which they still do: 2048 x 5120 as 216 tiles of 192 columns instead of
// 160 of 256 (515 -> 455 us at K = 17408).  But not with 64 rows or fewer, nor with 128 and a short K, which leave three
// quarters or half of those tiles empty (us, small tiles / 256 x 128): 64 rows of 24576 x 1024 30 / 39, of 32000 x 2048 58 / 68,
// 128 rows 34 / 40, 64 / 69; of 17408 x 5120 and 20000 x 5120 64 rows 97 / 95, 132 / 131, 128 rows 114 / 104, 143 / 135.
struct F16wTiles {
  uint32_t large, columns;
};
constexpr F16wTiles f16w_tiles(uint32_t m, uint32_t n, uint32_t k, uint32_t cus) {
  const uint32_t tiles_m = (m + 255u) / 256u;
  if (m > 128u || (m > 64u && k >= 4096u)) {
    for (uint32_t columns : {128u, 192u}) {
      const uint32_t tiles_n = (n + columns - 1u) / columns;
      if (tiles_m * tiles_n <= cus && tiles_m * tiles_n > cus / 2) return {tiles_n, columns};
    }
  }
  const uint32_t tiles_n = (n + 255u) / 256u, tiles = tiles_m * tiles_n;
  if (tiles > cus && tiles % cus != 0 && tiles % cus <= cus / 2) return {tiles / cus * cus / tiles_m, 256u};
  return {tiles < cus / 2 ? 0u : tiles_n, 256u};
}
// The order of the tiles.  Workgroups go round the XCDs, in the launch that decodes as here, so that along the columns an XCD
// finds part of the weights that it has written itself in its L2 (also with the rows' workgroups before the weights', whose count
// is the shift: 100, 101 and 103 rows of 16384 x 1024 25 us each, shares 32); an XCD's share of neighbouring tiles (xcd_tile) instead
// reads them once for several row tiles.  The first leads with one row tile, with up to three where the weights are small, and
// where small tiles are few (us, along / shares): 100 rows of 16384 x 1024 27 / 33, 256 rows 33 / 39, 300 of 6144 x 5120 70 /
// 84, 512 of 5120 x 17408 (320 small tiles) 286 / 324, 700 of 3072 x 1024 (288) 24 / 29; 256 rows of 17408 x 5120 161 / 151, of
// 12288 x 4096 (384) 78 / 76, 512 of 6144 x 5120 (384) 84 / 80.
constexpr bool f16w_tiles_as_decoded(uint32_t m, uint32_t n, uint32_t k, uint32_t cus, bool small) {
  return m <= 128u || (m <= 384u && static_cast<uint64_t>(n) * k <= (uint64_t{32} << 20)) ||
         (small && static_cast<uint64_t>((m + 127u) / 128u) * ((n + 63u) / 64u) * 4u <= cus * 5u);
}

// ---- "rope", "mrope" -------------------------------------------------------------------------------------------------
// Heads that share a thread's angle: eight from a wavefront a SIMD on (512 rows of 24 heads of 256 23 -> 7.5 us), of one head
// none, which would be read eight times (8193 rows of 64 5.7 / 6.2 us).
constexpr uint32_t rope_heads_a_thread(uint64_t rows, uint64_t heads, uint64_t pairs) {
  return heads > 1 && rows * heads * pairs >= 65536 ? 8 : 1;
}

// ---- "quantize_fp8_pack" ---------------------------------------------------------------------------------------------
// Workgroups of a row while the rows alone cannot fill the chip, at most sixteen, each finding the row's maximum for itself:
// of 256 threads one for 1024 columns, of 1024 one for 4096 where the row is long and there are many (us, 256 / 1024
// threads: 4 rows of 5120 3.3 / 3.5, of 8192 3.1 / 3.7, of 17408 3.6 / 4.0; 64 rows of 8192 3.6 / 4.0, 100 rows 4.5 / 4.1; 32
// of 17408 4.9 / 4.3, 200 rows 12 / 10).
struct PackShape {
  uint32_t per_row, threads;
};
constexpr PackShape pack_shape(uint64_t rows, uint64_t cols) {
  if (rows >= 256) return {1, 256};
  const uint32_t threads = cols <= 6144 || rows * cols <= (uint64_t{1} << 19) ? 256 : 1024;
  const uint64_t share = (cols + threads * 4 - 1) / (threads * 4);
  return {static_cast<uint32_t>(share < 16 ? share : 16), threads};
}

// ---- "attention" with many query rows -------------------------------------------------------------------------------
// How a call over an fp16 or a quantized cache runs: 0, the rows' kernel, a workgroup for up to eight heads of a row and
// key head; else the kernel that shares 64 keys at a time among 64 (row, head) pairs, in so many parts of the keys.  `keys`:
// how many a row sees at most; `padded`: the head size, 64, 128 or 256.
//
// The shorter of the estimated times, in us: a fixed part, then for the rows' kernel what a round of a workgroup a CU takes
// by its keys (four wavefronts up to 160 keys, eight beyond; where five take 129 to 160 keys they are up to a tenth faster than
// the estimate, and of 306 such calls none takes the longer way by more than 3 %), for the other what 64 keys take, and for its parts the
// second launch and the sums' way through memory.  Fitted to 1716 calls (17 to 512 rows, 17 to 2512 keys, 2 to 32 heads over
// 1 to 8 key heads of 64, 96, 128 and 256, fp16 and int8), which they meet within 4 % on average: one call of them
// takes the longer way by more than 5 %.  Rows' kernel / one part / parts: 64 rows of 24 heads over 4 of 256 on 564 keys 21 / 34 /
// 29, on 2064 48 / 95 / 42; 512 rows of 16 over 4 of 64 on 512 27 / 14 / 39; 64 of 8 over 8 of 128 on 64 7 / 10; 300 of 24
// over 4 of 256 on 2300 285 / 105.
struct AttentionCall {
  uint64_t rows, keys, heads, kv_heads, head_dim, padded;
  bool quantized;
};
constexpr uint64_t attention_pairs64(const AttentionCall& a) { return (a.rows * (a.heads / a.kv_heads) + 63) / 64 * a.kv_heads; }
// Bytes of `parts` parts: a sum of head_dim, the largest score and the sum of weights for each.
constexpr size_t attention_parts_size(uint64_t rows, uint64_t heads, uint64_t head_dim, uint64_t parts) {
  return parts < 2 ? 0 : static_cast<size_t>(rows * heads * parts * (head_dim + 2) * 4);
}
constexpr uint64_t attention_rule(const AttentionCall& a, uint64_t cus, uint64_t most_parts, size_t most_bytes) {
  const uint64_t units = attention_pairs64(a), tiles = (a.keys + 63) / 64;
  const uint64_t row_units = a.rows * a.kv_heads * ((a.heads / a.kv_heads + 7) / 8);
  uint64_t parts = cus / units < a.keys / 256 ? cus / units : a.keys / 256;
  if (parts > most_parts) parts = most_parts;
  while (parts > 1 && attention_parts_size(a.rows, a.heads, a.head_dim, parts) > most_bytes) --parts;

  const int size = a.padded == 64 ? 0 : a.padded == 128 ? 1 : 2;
  constexpr double kRowFixed[2][3] = {{5.2, 5.5, 5.3}, {5.3, 4.1, 5.3}}, kRowRound[2][3] = {{0.3, 0.65, 3.4}, {0.5, 3.1, 3.4}};
  constexpr double kRowKey[2][3] = {{0.0047, 0.0102, 0.0194}, {0.005, 0.0083, 0.0194}};
  constexpr double kTileFixed[3] = {6.1, 8.1, 12.8}, kTile[3] = {1.0, 1.32, 2.31}, kPartsMegabyte[3] = {1.07, 0.85, 0.79};
  constexpr double kPartsFixed = 2.5;
  const int wide = a.keys > 160 ? 1 : 0;
  const uint64_t row_rounds = (row_units + cus - 1) / cus, rounds = (units + cus - 1) / cus;
  const double key_us = kRowKey[wide][size] * (a.quantized ? 1.12 : 1.0);
  const double row_us = kRowFixed[wide][size] + (a.quantized ? 0.6 : 0.0) +
                        static_cast<double>(row_rounds) * (kRowRound[wide][size] + key_us * static_cast<double>(a.keys));
  const double tile = kTile[size] * (a.quantized ? 1.25 : 1.0);
  const double one_us = kTileFixed[size] + tile * static_cast<double>(rounds * tiles);
  if (parts > 1) {
    const uint64_t part_tiles = ((a.keys + parts - 1) / parts + 63) / 64;
    const double parts_us = kTileFixed[size] + kPartsFixed + tile * static_cast<double>(part_tiles) +
                            kPartsMegabyte[size] * static_cast<double>(a.rows * a.heads * parts * a.head_dim * 4) * 1e-6;
    if (parts_us <= one_us && parts_us < 0.98 * row_us) return parts;
  }
  return one_us < 0.98 * row_us ? 1 : 0;
}

// ---- "attention_combine" ---------------------------------------------------------------------------------------------
// Wavefronts of a (row, head): sixteen where there are few and many parts, four where the rows fill the chip by themselves or
// sixteen parts are all that there are, one where its four are and that does not make a lane's run long with few rows (us, 1 /
// 4 / 16 wavefronts: 24 rows of 256 over 4 parts 3.3 / 2.9 / 3.2, over 64 15 / 6.9 / 6.0; 12288 rows of 64 over 2 parts 5.4 / 10 / 39,
// of 256 over 8 26 / 25 / 55).
constexpr uint32_t combine_waves(uint64_t rows, uint64_t head_dim, uint64_t parts) {
  if (parts <= 4 && (rows >= 1024 || head_dim <= 64 || parts == 1)) return 1;
  return parts <= 16 || rows > 256 ? 4 : 16;
}

}  // namespace qmm
