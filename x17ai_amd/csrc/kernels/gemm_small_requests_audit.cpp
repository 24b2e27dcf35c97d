// Host-side audit of the small-tile GEMM kernel's requests (gemm_b8_small.hip), as gemm_requests_audit.cpp is of the
// 256 x 256 kernel's: compiled with a form's own common.h and gemm_small_tile.h, whose functions the kernel calls, it
// enumerates every 16-byte direct-to-LDS request of a launch with `a_rows` token rows -- every tile, K step, wavefront,
// unit and lane, the repeats past the last step included.  Each stays inside its operand, a step's chunks are requested
// exactly once and stored where the fragment reads look for them, every output tile is walked once, and the weight rows
// are permuted as the writers expect.  Prints the extents as JSON.
//
//     gemm_small_requests_audit <a_rows> [rows the token operand really has, default a_rows]
#include "common.h"
#include "gemm_small_tile.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

namespace gt = x17::gemm_small_tile;

static int fail(char const *what, unsigned long long a, unsigned long long b) {
	std::printf("{\"ok\": false, \"error\": \"%s\", \"value\": %llu, \"limit\": %llu}\n", what, a, b);
	return 1;
}

int main(int argc, char **argv) {
	if (argc != 2 && argc != 3) {
		std::fprintf(stderr, "usage: %s <a_rows> [allocated rows]\n", argv[0]);
		return 2;
	}
	unsigned long long const a_rows_arg = std::strtoull(argv[1], nullptr, 10);
	unsigned long long const a_rows_allocated = argc == 3 ? std::strtoull(argv[2], nullptr, 10) : a_rows_arg;
	constexpr unsigned long long K = X17_A_COLS;
	constexpr unsigned N_RAW = X17_B_ROWS, K_STEPS = X17_A_COLS / gt::K_STEP;
#if X17_EPILOGUE == 6
	constexpr unsigned Q_COLS = X17_Q_COLS;
#else
	constexpr unsigned Q_COLS = N_RAW;       // one weight matrix
#endif
	if (a_rows_arg < 256 || a_rows_arg % 64 != 0 || a_rows_arg > 0xFFFFFFFFull) {
		return fail("token rows must be a multiple of 64, at least 256 and fit 32 bits (the launcher rejects them)", a_rows_arg, 256);
	}
	unsigned const a_rows = (unsigned)a_rows_arg;

	// one tile and step: the requests of an operand's part of `rows` LDS rows, `units` per wavefront
	unsigned long long per_step = 0;
	unsigned max_chunk = 0;
	auto pattern = [&](unsigned rows, unsigned units, bool weights) -> char const * {
		std::vector<unsigned> source(rows * gt::CHUNKS, 0), stored(rows * gt::CHUNKS, 0);
		for (unsigned wave = 0; wave < gt::WAVES; ++wave) {
			for (unsigned u = 0; u < units; ++u) {
				for (unsigned lane = 0; lane < 64; ++lane) {
					unsigned const unit = wave * units + u, row = gt::unit_row(unit, lane), chunk = gt::unit_chunk(unit, lane);
					if (row >= rows) return "row of a request outside its tile";
					if (chunk >= gt::CHUNKS) return "chunk of a request outside the K step";
					// lane l of unit u lands at u * 1024 + 16 * l of the operand's part of the slot
					unsigned const position = (unit * 1024 + 16 * lane) % gt::K_STEP / 16;
					if ((unit * 1024 + 16 * lane) / gt::K_STEP != row) return "request stored in another row";
					// fragment reads: logical chunk c of row r at position c ^ swizzle(r % 32)
					if (position != (chunk ^ gt::swizzle(row % 32))) return "chunk stored where no fragment read looks for it";
					unsigned const from = weights ? gt::w_source_row(row) : row;
					if (from >= rows) return "source row of a request outside its tile";
					++source[from * gt::CHUNKS + chunk];
					++stored[row * gt::CHUNKS + position];
					max_chunk = chunk > max_chunk ? chunk : max_chunk;
					++per_step;
				}
			}
		}
		for (unsigned v : source) if (v != 1) return weights ? "a weight-tile chunk is not requested exactly once" : "a token-tile chunk is not requested exactly once";
		for (unsigned v : stored) if (v != 1) return "a position of the slot is not filled exactly once";
		return nullptr;
	};
	if (char const *what = pattern(gt::M_PER_BLOCK, gt::X_UNITS, false)) return fail(what, gt::M_PER_BLOCK, 0);
	// the widening form: every chunk of the weights is loaded by one widener lane, and every 16 bytes of a widened tile are
	// written once and read as one fragment
	auto widened = [&]() -> char const * {
		std::vector<unsigned> source(gt::N_PER_BLOCK * gt::CHUNKS, 0), stored(gt::WIDE_BYTES / 16, 0), read(gt::WIDE_BYTES / 16, 0);
		auto touch = [&](std::vector<unsigned> &v, unsigned at) { return at % 16 == 0 && at / 16 < v.size() ? (++v[at / 16], true) : false; };
		for (unsigned wave = 0; wave < gt::WIDENERS; ++wave) for (unsigned u = 0; u < gt::WIDENER_UNITS; ++u) for (unsigned lane = 0; lane < 64; ++lane) {
			unsigned const row = gt::widener_row(wave, u, lane), chunk = gt::widener_chunk(lane);
			if (row >= gt::N_PER_BLOCK || gt::w_source_row(row) >= gt::N_PER_BLOCK) return "row of a widener's load outside its tile";
			if (chunk >= gt::CHUNKS) return "chunk of a widener's load outside the K step";
			++source[gt::w_source_row(row) * gt::CHUNKS + chunk];
			max_chunk = chunk > max_chunk ? chunk : max_chunk;
			for (unsigned h = 0; h < 2; ++h) if (!touch(stored, gt::wide_offset(row, 2 * chunk + h))) return "a widened chunk is stored outside its tile";
			++per_step;
		}
		// fragment reads: 32-byte slice s, K half of the lane, matrix instruction h
		for (unsigned row = 0; row < gt::N_PER_BLOCK; ++row) for (unsigned s = 0; s < gt::K_STEP / 32; ++s) for (unsigned half = 0; half < 2; ++half) {
			for (unsigned h = 0; h < 2; ++h) if (!touch(read, gt::wide_offset(row, 4 * s + 2 * half + h))) return "a widened chunk is read outside its tile";
		}
		for (unsigned v : source) if (v != 1) return "a weight-tile chunk is not loaded exactly once";
		for (unsigned v : stored) if (v != 1) return "a position of the widened tile is not filled exactly once";
		for (unsigned v : read) if (v != 1) return "a position of the widened tile is not one fragment's";
		return nullptr;
	};
	if (char const *what = gt::WIDEN_ONCE ? widened() : pattern(gt::N_PER_BLOCK, gt::W_UNITS, true)) return fail(what, gt::N_PER_BLOCK, 0);
	// matrix block bn of a wavefront, register r of a lane half: the writer takes it as column (WAVE_N / 2) * half + 16 * bn + r
	if (!gt::NATURAL) {
		for (unsigned wn = 0; wn < gt::WAVES_N; ++wn) for (unsigned bn = 0; bn < gt::WAVE_N / 32; ++bn) for (unsigned half = 0; half < 2; ++half) for (unsigned r = 0; r < 16; ++r) {
			unsigned const lds_row = gt::WAVE_N * wn + 32 * bn + 8 * (r / 4) + 4 * half + r % 4;
			unsigned const column = gt::WAVE_N * wn + gt::WAVE_N / 2 * half + 16 * bn + r;
			if (gt::w_source_row(lds_row) != column) return fail("a weight row is not the column its results are written to", gt::w_source_row(lds_row), column);
		}
	}

	unsigned const tiles_m = (a_rows + gt::M_PER_BLOCK - 1) / gt::M_PER_BLOCK, tiles_n = N_RAW / gt::N_PER_BLOCK, total = tiles_m * tiles_n;
	unsigned long long a_extent = 0, bq_extent = 0, bkv_extent = 0;
	std::vector<unsigned char> tile_seen((size_t)tiles_m * tiles_n, 0);
	for (unsigned lin = 0; lin < total; ++lin) {
		gt::TileOrigin const o = gt::tile_origin(lin, a_rows, N_RAW);
		if (o.m % 32 != 0 || o.m + gt::M_PER_BLOCK > a_rows) return fail("tile leaves the token rows", o.m + gt::M_PER_BLOCK, a_rows);
		if (o.n % gt::N_PER_BLOCK != 0 || o.n + gt::N_PER_BLOCK > N_RAW) return fail("tile leaves the raw columns", o.n + gt::N_PER_BLOCK, N_RAW);
		// (a moved-back tile keeps its place in the grid of tiles: the last tile row)
		unsigned const gm = (o.m + gt::M_PER_BLOCK - 1) / gt::M_PER_BLOCK, gn = o.n / gt::N_PER_BLOCK;
		if (tile_seen[(size_t)gm * tiles_n + gn]++) return fail("a tile is walked twice", lin, total);
		bool const kv_side = o.n >= Q_COLS;
		if (!kv_side && o.n + gt::N_PER_BLOCK > Q_COLS) return fail("a tile straddles the q and kv weights", o.n + gt::N_PER_BLOCK, Q_COLS);
		unsigned long long const w_first = kv_side ? o.n - Q_COLS : o.n, w_rows = kv_side ? N_RAW - Q_COLS : Q_COLS;
		// (requests run STAGES - 1 steps ahead, a widener's loads WIDENER_DEPTH + 2)
		for (unsigned step = 0; step < K_STEPS + (gt::WIDEN_ONCE ? gt::WIDENER_DEPTH + 2 : gt::STAGES - 1); ++step) {
			unsigned long long const k0 = (step < K_STEPS ? step : K_STEPS - 1) * (unsigned long long)gt::K_STEP;
			unsigned long long const col_end = k0 + 16ull * max_chunk + 16;
			if (col_end > K) return fail("request leaves its operand row", col_end, K);
			unsigned long long const a_end = (o.m + gt::M_PER_BLOCK - 1) * K + col_end, w_end = (w_first + gt::N_PER_BLOCK - 1) * K + col_end;
			if (a_end > a_rows_allocated * K) return fail("token request past the end of a", a_end, a_rows_allocated * K);
			if (w_end > w_rows * K) return fail("weight request past the end of b", w_end, w_rows * K);
			a_extent = a_end > a_extent ? a_end : a_extent;
			(kv_side ? bkv_extent : bq_extent) = w_end > (kv_side ? bkv_extent : bq_extent) ? w_end : (kv_side ? bkv_extent : bq_extent);
		}
	}
	// a lane offset inside a tile fits its 32 bits
	if ((gt::M_PER_BLOCK - 1) * K + K > 0xFFFFFFFFull || (gt::N_PER_BLOCK - 1) * K + K > 0xFFFFFFFFull) return fail("lane offsets exceed 32 bits", K, 0);
	std::printf("{\"ok\": true, \"tiles\": %u, \"requests\": %llu, \"a_extent\": %llu, \"a_bytes\": %llu, \"b_extent\": %llu, \"b_bytes\": %llu, "
	            "\"b_kv_extent\": %llu, \"b_kv_bytes\": %llu}\n",
	            total, per_step * (K_STEPS + gt::STAGES - 1) * total, a_extent, a_rows_allocated * K, bq_extent, (unsigned long long)Q_COLS * K,
	            bkv_extent, (unsigned long long)(N_RAW - Q_COLS) * K);
	return 0;
}
