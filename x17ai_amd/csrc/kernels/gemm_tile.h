// gemm_tile.h -- tile geometry of the 8-bit GEMM kernel as plain constexprs.
//
// Included by the device code (gemm_b8.hip) and by the small host program that prints
// meta.json, so that the C++ constants stay the single source of truth for the launch
// geometry, as in the reference (templates/basic_gemm/meta.cu:10-17,
// src/device/cuda/gemm.rs:529-537).  Needs X17_A_KIND / X17_B_KIND from common.h.
//
// A build may override the geometry with -DX17_GEMM_M_PER_BLOCK (128 or 256 tokens per workgroup),
// -DX17_GEMM_WAVES_M / -DX17_GEMM_WAVES_N (wavefronts along the tokens / along the raw output columns),
// -DX17_GEMM_K_STEP (64 or 128 bytes of K per pipeline step), -DX17_GEMM_STAGES (LDS ring depth) and
// -DX17_GEMM_X_STAGES (ring depth of the token operand alone: STAGES or STAGES + 1).  Needs X17_A_COLS too.
#pragma once

namespace x17 { namespace gemm_tile {

constexpr unsigned WAVE = 64;

#ifndef X17_GEMM_M_PER_BLOCK
#define X17_GEMM_M_PER_BLOCK 256
#endif
#ifndef X17_GEMM_WAVES_M
#define X17_GEMM_WAVES_M 4
#endif
#ifndef X17_GEMM_WAVES_N
#define X17_GEMM_WAVES_N 2
#endif
#ifndef X17_GEMM_K_STEP
#define X17_GEMM_K_STEP 128
#endif
#ifndef X17_GEMM_STAGES
#define X17_GEMM_STAGES 2
#endif

constexpr unsigned M_PER_BLOCK = X17_GEMM_M_PER_BLOCK;   // tokens per workgroup
constexpr unsigned N_PER_BLOCK = 256;                    // raw output columns per workgroup
constexpr unsigned WAVES_M = X17_GEMM_WAVES_M;           // waves along the token (M) dimension
constexpr unsigned WAVES_N = X17_GEMM_WAVES_N;           // waves along the output-column (N) dimension
constexpr unsigned THREADS_PER_BLOCK = WAVE * WAVES_M * WAVES_N;

constexpr unsigned WAVE_M = M_PER_BLOCK / WAVES_M;       // tokens per wave (64 or 128)
constexpr unsigned WAVE_N = N_PER_BLOCK / WAVES_N;       // raw output columns per wave (128 or 64)
constexpr unsigned K_STEP = X17_GEMM_K_STEP;             // bytes of K staged per pipeline step
constexpr unsigned STAGES = X17_GEMM_STAGES;

// The token tiles may have a ring one deeper than the weight tiles: 3 x 32 KB + 2 x 32 KB fill the 160 KB of
// LDS of a compute unit exactly, and the token loads then have two steps to arrive, the weight loads one
// (with two stages of both, a step's 64 KB of loads have a single step -- about their own latency -- to land).
#ifndef X17_GEMM_X_STAGES
#define X17_GEMM_X_STAGES \
	((X17_GEMM_STAGES == 2 && X17_GEMM_K_STEP == 128 && X17_GEMM_M_PER_BLOCK == 256 && (X17_A_COLS) / 128 >= 3) ? 3 : X17_GEMM_STAGES)
#endif
constexpr unsigned X_STAGES = X17_GEMM_X_STAGES;
static_assert(X_STAGES == STAGES || X_STAGES == STAGES + 1, "the token ring is as deep as the weight ring or one deeper");

constexpr unsigned SMEM_BYTES = (X_STAGES * M_PER_BLOCK + STAGES * N_PER_BLOCK) * K_STEP;

// The kernel is persistent (a workgroup walks tiles g, g + G, ...): the launcher starts at most this
// many workgroups, one per compute unit of an MI355X.
constexpr unsigned MAX_BLOCKS = 256;

// Wavefronts per SIMD the register budget is sized for: waves of eight 32 x 32 blocks (64 x 128 or 128 x 64)
// keep their 128 accumulators and everything else within 256 registers so that two of them share a SIMD
// (two workgroups per compute unit when a workgroup has four waves); 128 x 128 waves need all 512.
constexpr unsigned WAVES_PER_SIMD = (WAVE_M / 32) * (WAVE_N / 32) <= 8 ? 2 : 1;

// Rows of an operand per matrix instruction.  NATURAL: the writers that normalise whole heads, with an order of the weight rows of their own.
// e4m3 takes blocks of 16 from K = 2048 on: below, the accumulators' way to the writer costs more than the K loop gains (GeGLU writer,
// 4096 columns, 16384 rows, us, blocks of 32 / of 16: K = 384 37.4 / 39.9, 512 41.6 / 44.4, 1024 66.0 / 66.7, 2048 104.1 / 102.7).
// The kv writer with heads of 32 columns keeps blocks of 32: with blocks of 16 one or two of its registers spill.
// int8 gains at every K (scale writer: K = 384 41.0 / 34.9, 1024 77 / 63; GeGLU, K = 512 42.2 / 41.9, 1024 69.9 / 63.7;
// q + kv, K = 2048, 6144 columns, 3264 rows 46.4 / 44.8, 32768 rows 323 / 301; kv alone, 4096 columns, K = 2048 110 / 103, and K = 512 41.5 both).
constexpr bool NATURAL = X17_EPILOGUE == 3 || X17_EPILOGUE == 5 || X17_EPILOGUE == 6;
#if X17_EPILOGUE == 3
constexpr bool SPILLS16 = X17_HEAD_DIM == 32;
#else
constexpr bool SPILLS16 = false;
#endif
// (their tile requests are buffer loads, whose resource has 32 bits for a tile's bytes: from K = 2^24 on, blocks of 32)
constexpr unsigned long long RESOURCE_BYTES = 256ull * (X17_A_COLS);
constexpr bool BLOCKS16 = X17_A_KIND == X17_B_KIND && !SPILLS16 && STAGES == 2 && X_STAGES == 3 && (X17_A_COLS) / K_STEP >= X_STAGES
	&& WAVE_N == 128 && (WAVE_M == 64 || WAVE_M == 128) && (X17_A_KIND == 0 || (WAVES_PER_SIMD == 1 && (X17_A_COLS) >= 2048)) && RESOURCE_BYTES < 1ull << 32;
constexpr unsigned BLOCK = BLOCKS16 ? 16 : 32;

// ---- index arithmetic of the tile requests (global -> LDS, 16 bytes per lane).  The kernel calls these; so does the
// host-side audit (gemm_requests_audit.cpp), which enumerates every request of a launch on the CPU and checks that it
// stays inside its operand.
// LDS rows hold K_STEP bytes = CHUNKS chunks of 16; one 64-lane load fills UNIT_ROWS rows ("a load unit").
constexpr unsigned CHUNKS = K_STEP / 16;
constexpr unsigned SWZ_SHIFT = K_STEP == 128 ? 1 : 2;
constexpr unsigned UNIT_ROWS = 64 / CHUNKS;
// Chunk c of an LDS row is stored at position c ^ swizzle(row).  The LDS serves a ds_read_b128 sixteen lanes at a time, lanes 0 .. 3,
// 12 .. 15, 20 .. 23 and 24 .. 27 together (and so on); with blocks of 16 rows the last eight ask for another chunk than
// the first.  With 128-byte rows the map of a row pair's number keeps their sixteen 16-byte positions apart whichever chunk that is:
// pairs 0, 1, 6, 7 take keys 0 .. 3, pairs 2 .. 5 keys 4 .. 7.
constexpr unsigned swizzle(unsigned row) {
	unsigned const t = (row >> SWZ_SHIFT) & (CHUNKS - 1);
	return CHUNKS == 8 ? (t & 1) | (t >> 2) << 1 | ((t >> 1 ^ t >> 2) & 1) << 2 : t;
}
// With eight waves, two per SIMD, only the first of each pair (waves 0 .. 3) requests tiles.
constexpr unsigned LOADER_WAVES = WAVES_M * WAVES_N == 8 ? 4 : WAVES_M * WAVES_N;
constexpr unsigned X_UNITS = M_PER_BLOCK / UNIT_ROWS / LOADER_WAVES;   // load units per loading wave, step and tile
constexpr unsigned W_UNITS = N_PER_BLOCK / UNIT_ROWS / LOADER_WAVES;
// The weight row that LDS weight row r0 (a multiple of UNIT_ROWS) starts from.  With WN = WAVE_N columns per wave, a lane collects
// WN / GROUPS consecutive output columns: LDS weight row R = WN*wn + BLOCK*bn + i holds weight row
//   blocks of 32 (GROUPS = 2: lanes 32 apart)    WN*wn + (WN/2)*((i/4)%2) + 16*bn + 4*(i/8) + i%4
//   blocks of 16 (GROUPS = 4: lanes 16 apart)    WN*wn + (WN/4)*(i/4) + 4*bn + i%4
// The head-normalising writers keep the natural order in blocks of 32, and in blocks of 16 take
//   16*bn + 8*((i%4)/2) + 2*(i/4) + i%2     of a wave's columns: lane group i/4 holds those with (column % 8) / 2 == i / 4.
constexpr unsigned GROUPS = 64 / BLOCK;
constexpr unsigned w_unit_row(unsigned r0, bool natural) {
	if (natural && BLOCKS16) return r0 / 16 * 16 + 2 * (r0 % 16 / 4);
	return natural ? r0 : WAVE_N * (r0 / WAVE_N) + (BLOCK * BLOCK / 64) * ((r0 % WAVE_N) / BLOCK)
	                      + (BLOCKS16 ? (WAVE_N / 4) * ((r0 % 16) / 4) : 4 * ((r0 % 32) / 8));
}
// Row inside its load unit, as an operand row offset, and 16-byte chunk of the K step that lane `lane` fetches
// (`odd`: parity of the unit, which shifts the swizzle phase).
constexpr unsigned x_lane_row(unsigned lane) { return lane / CHUNKS; }
constexpr unsigned w_lane_row(unsigned lane, bool natural) {
	unsigned const j = lane / CHUNKS;
	if (natural && BLOCKS16) return 8 * ((j & 3) / 2) + 2 * (j >> 2) + (j & 1);
	return natural ? j : BLOCKS16 ? (WAVE_N / 4) * (j >> 2) + (j & 3) : (WAVE_N / 2) * ((j >> 2) & 1) + 4 * (j >> 3) + (j & 3);
}
constexpr unsigned lane_chunk(unsigned lane, unsigned odd) {
	unsigned const j = lane / CHUNKS, p = lane % CHUNKS;
	return p ^ swizzle(odd * UNIT_ROWS + j);
}
// The largest row that a lane's 32-bit operand offset holds: of its load unit, and with one wavefront per SIMD, which keeps an offset per unit,
// of its wave's share.
constexpr unsigned max_offset_row(bool natural) {
	unsigned most = 0;
	for (unsigned wave = 0; wave < LOADER_WAVES; ++wave) {
		for (unsigned u = 0; u < (WAVES_PER_SIMD == 1 ? W_UNITS : 1); ++u) {
			for (unsigned lane = 0; lane < 64; ++lane) {
				unsigned const first = wave * W_UNITS * UNIT_ROWS;
				unsigned const row = w_unit_row(first + u * UNIT_ROWS, natural) - w_unit_row(first, natural) + w_lane_row(lane, natural);
				most = row > most ? row : most;
			}
		}
	}
	unsigned const x = (WAVES_PER_SIMD == 1 ? X_UNITS : 1) * UNIT_ROWS - 1;
	return x > most ? x : most;
}
// First token row and first raw column of tile `lin` of the persistent walk: each XCD (the hardware deals workgroups
// round-robin to 8 of them) gets a contiguous run of tiles, walked in bands of `band` token tiles; a last tile that
// would overhang the matrix is moved back to end at its edge.
struct TileOrigin { unsigned m, n; };
constexpr TileOrigin tile_origin(unsigned lin, unsigned a_rows, unsigned n_raw, unsigned band) {
	unsigned const tiles_m = (a_rows + M_PER_BLOCK - 1) / M_PER_BLOCK;
	unsigned const tiles_n = (n_raw + N_PER_BLOCK - 1) / N_PER_BLOCK;
	unsigned const total = tiles_m * tiles_n;
	if (total % 8 == 0) {
		lin = (lin % 8) * (total / 8) + lin / 8;
	}
	unsigned const band_tiles = band * tiles_n;
	unsigned const b = lin / band_tiles;
	unsigned const in_band = lin % band_tiles;
	unsigned const rows_in_band = (tiles_m - b * band) < band ? (tiles_m - b * band) : band;
	unsigned m = (b * band + in_band % rows_in_band) * M_PER_BLOCK;
	unsigned n = (in_band / rows_in_band) * N_PER_BLOCK;
	m = m + M_PER_BLOCK > a_rows ? a_rows - M_PER_BLOCK : m;
	n = n + N_PER_BLOCK > n_raw ? n_raw - N_PER_BLOCK : n;
	return TileOrigin{m, n};
}
#ifdef X17_GEMM_BAND
constexpr unsigned BAND = X17_GEMM_BAND;
#else
constexpr unsigned BAND = 2048 / M_PER_BLOCK;
#endif

static_assert(M_PER_BLOCK == 128 || M_PER_BLOCK == 256, "tokens per workgroup: 128 or 256");
static_assert(WAVE_M == 64 || WAVE_M == 128, "a wave owns 64 or 128 tokens");
static_assert(WAVE_N == 128 || WAVE_N == 64, "a wave owns 128 or 64 raw output columns");
static_assert(K_STEP == 64 || K_STEP == 128, "K step: 64 or 128 bytes");
static_assert(STAGES >= 2 && STAGES <= 4, "2 to 4 stages");
static_assert(SMEM_BYTES <= 160 * 1024, "LDS ring does not fit");

}} // namespace x17::gemm_tile
