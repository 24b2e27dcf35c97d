// gemm_small_tile.h -- tile geometry and request index arithmetic of the small-tile GEMM kernel (gemm_b8_small.hip) as
// plain constexprs, shared with the host program that prints its meta.json.  Needs X17_A_COLS, X17_A_KIND, X17_B_KIND,
// X17_EPILOGUE, X17_SMALL_TILE and X17_SMALL_STAGES from common.h:
//   X17_SMALL_TILE 64   64 x 64 raw columns per workgroup, four wavefronts
//   X17_SMALL_TILE 128  128 x 128, eight wavefronts (e4m3 x int8: four)
//   X17_SMALL_STAGES    depth of the LDS ring of K steps: 2 (of 128 x 128, two workgroups share a compute unit) or 4
// The writers that normalise heads of up to 128 columns need a wavefront that owns 128 of them: with those the
// wavefront is 32 tokens x 128 columns instead of 64 x 64, the workgroup 32 x 128 or 128 x 128.
#pragma once

namespace x17 { namespace gemm_small_tile {

constexpr bool NATURAL = X17_EPILOGUE == 3 || X17_EPILOGUE == 5 || X17_EPILOGUE == 6;   // weight rows in their natural order
constexpr bool MID = X17_SMALL_TILE == 128;
static_assert(X17_SMALL_TILE == 64 || X17_SMALL_TILE == 128, "tiles of 64 or of 128");

// int32 sums are exact in any order: there several wavefronts share an output block, each a part of every K step, and
// add up their sums.  A float32 sum depends on its order, which is that of the 256 x 256 kernel -- one wavefront through
// the whole of K -- so that a row's result does not depend on how many rows are launched with it.
constexpr bool SPLIT_K = X17_A_KIND == 0 && X17_B_KIND == 0;
// Of the 128 x 128 forms e4m3 x e4m3 takes eight wavefronts of 64 x 32 (1024 rows x 4096 columns, two stages, K = 1024:
// 8.0 us, four of 64 x 64 10.3, eight of 32 x 64 9.0); e4m3 x int8, which widens every fragment it reads to f16, four of
// 64 x 64 (4096 rows, K = 2048: 62 us, 66 and 77).
constexpr bool WIDENS = X17_A_KIND != X17_B_KIND;
constexpr unsigned WAVE_M = NATURAL || (!SPLIT_K && !MID) ? 32 : 64;                  // tokens per wavefront
constexpr unsigned WAVE_N = NATURAL ? 128 : SPLIT_K || (MID && WIDENS) ? 64 : 32;     // raw output columns per wavefront
constexpr unsigned WAVES_M = MID ? 128 / WAVE_M : SPLIT_K ? 1 : 64 / WAVE_M;
constexpr unsigned WAVES_N = MID ? 128 / WAVE_N : SPLIT_K ? 1 : 64 / WAVE_N;
constexpr unsigned WAVES_K = !SPLIT_K ? 1 : MID ? 2 : 4;                              // wavefronts that share an output block
constexpr unsigned WAVES = WAVES_M * WAVES_N * WAVES_K;
// The 64 x 64 form of e4m3 x int8: four more wavefronts bring the weights into LDS and widen them to f16 on the way, once for
// the workgroup.  (An int8 fragment is twenty instructions, an e4m3 one eight: widening the tokens there as well adds more
// LDS traffic than it takes instructions out.)
constexpr bool WIDEN_ONCE = X17_A_KIND == 1 && X17_B_KIND == 0 && !MID && !NATURAL;
constexpr unsigned WIDENERS = WIDEN_ONCE ? 4 : 0;
constexpr unsigned THREADS_PER_BLOCK = 64 * (WAVES + WIDENERS);
constexpr unsigned M_PER_BLOCK = WAVE_M * WAVES_M;
constexpr unsigned N_PER_BLOCK = WAVE_N * WAVES_N;

// bytes of K per pipeline step: four e4m3 slices of 64 need 256
constexpr unsigned K_STEP = MID || WIDEN_ONCE ? 128 : 256;
constexpr unsigned STAGES = WIDEN_ONCE ? 6 : X17_SMALL_STAGES;      // LDS ring depth
constexpr unsigned STAGE_BYTES = (M_PER_BLOCK + (WIDEN_ONCE ? 0 : N_PER_BLOCK)) * K_STEP;
// two widened weight tiles behind the token tiles: one is read while the next one is written
constexpr unsigned WIDE_TILES = 2;
constexpr unsigned WIDE_OFFSET = STAGES * STAGE_BYTES;
constexpr unsigned WIDE_BYTES = N_PER_BLOCK * 2 * K_STEP;
constexpr unsigned SMEM_BYTES = WIDE_OFFSET + (WIDEN_ONCE ? WIDE_TILES * WIDE_BYTES : 0);
constexpr unsigned WAVES_PER_SIMD = 160 * 1024 / SMEM_BYTES * (WAVES + WIDENERS) / 4;      // as many workgroups as the LDS holds
static_assert(X17_A_COLS % K_STEP == 0, "K must be whole steps");
static_assert(SMEM_BYTES <= 160 * 1024, "LDS ring does not fit");

// ---- requests (global -> LDS, 16 bytes per lane).  An LDS row is K_STEP bytes = CHUNKS chunks of 16; a 64-lane request
// fills UNIT_ROWS rows; chunk c of row r is stored at position c ^ swizzle(r), so that the sixteen consecutive rows a
// ds_read_b128 serves at a time land in sixteen different 16-byte columns of the 256-byte bank line.
constexpr unsigned CHUNKS = K_STEP / 16;
constexpr unsigned UNIT_ROWS = 64 / CHUNKS;
constexpr unsigned X_UNITS = M_PER_BLOCK / UNIT_ROWS / WAVES;       // requests per wavefront and step
constexpr unsigned W_UNITS = N_PER_BLOCK / UNIT_ROWS / WAVES;
static_assert(X_UNITS * UNIT_ROWS * WAVES == M_PER_BLOCK && W_UNITS * UNIT_ROWS * WAVES == N_PER_BLOCK, "whole requests");
constexpr unsigned swizzle(unsigned row) { return (K_STEP == 256 ? row : row >> 1) & (CHUNKS - 1); }
constexpr unsigned unit_row(unsigned unit, unsigned lane) { return unit * UNIT_ROWS + lane / CHUNKS; }            // LDS row
constexpr unsigned unit_chunk(unsigned unit, unsigned lane) { return (lane % CHUNKS) ^ swizzle(unit_row(unit, lane)); }
// The weight row LDS weight row r holds (gemm_tile.h: a lane then collects consecutive output columns)
constexpr unsigned w_source_row(unsigned r) {
	unsigned const i = r % 32, bn = (r % WAVE_N) / 32;
	return NATURAL ? r : WAVE_N * (r / WAVE_N) + (WAVE_N / 2) * ((i / 4) % 2) + 16 * bn + 4 * (i / 8) + i % 4;
}
// ---- the widening form: a widener's 16-byte loads of a step's weights (consecutive lanes read consecutive bytes of a row), and
// where the eight f16 of raw bytes 8 c .. 8 c + 7 of row r are stored in a widened tile.  What eight lanes write, and the
// sixteen rows a read serves at a time, lie in different 16-byte columns of the 256-byte bank line.
constexpr unsigned WIDENER_UNITS = WIDEN_ONCE ? N_PER_BLOCK / UNIT_ROWS / WIDENERS : 1;
constexpr unsigned widener_row(unsigned wave, unsigned u, unsigned lane) { return unit_row(wave * WIDENER_UNITS + u, lane); }
constexpr unsigned widener_chunk(unsigned lane) { return lane % CHUNKS; }
constexpr unsigned wide_offset(unsigned row, unsigned c) { return row * 2 * K_STEP + ((c ^ (row & 15)) << 4); }
constexpr unsigned WIDENER_DEPTH = 6;                        // K steps of weights on their way, in registers
static_assert(WIDENER_DEPTH % WIDE_TILES == 0, "one loop over both rings");
// First token row and raw column of workgroup `lin`: each XCD (workgroups are dealt round-robin to 8 of them) gets a
// contiguous run of tiles, column tiles slowest inside bands of BAND token tiles, so that an XCD reads its weight
// columns once.  A last token tile that would overhang is moved back to end at the matrix edge.
struct TileOrigin { unsigned m, n; };
constexpr unsigned BAND = 2048 / M_PER_BLOCK;
constexpr TileOrigin tile_origin(unsigned lin, unsigned a_rows, unsigned n_raw) {
	unsigned const tiles_m = (a_rows + M_PER_BLOCK - 1) / M_PER_BLOCK, tiles_n = n_raw / N_PER_BLOCK, total = tiles_m * tiles_n;
	if (total % 8 == 0) lin = (lin % 8) * (total / 8) + lin / 8;
	unsigned const band_tiles = BAND * tiles_n, b = lin / band_tiles, in_band = lin % band_tiles;
	unsigned const rows_in_band = tiles_m - b * BAND < BAND ? tiles_m - b * BAND : BAND;
	unsigned const m = (b * BAND + in_band % rows_in_band) * M_PER_BLOCK;
	return TileOrigin{m + M_PER_BLOCK > a_rows ? a_rows - M_PER_BLOCK : m, (in_band / rows_in_band) * N_PER_BLOCK};
}

}} // namespace x17::gemm_small_tile
