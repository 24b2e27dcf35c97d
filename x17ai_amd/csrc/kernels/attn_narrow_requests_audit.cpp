// Host-side audit of the attention kernel with sixteen queries per wavefront (attn_fwd_i8_narrow.hip): compiled with the kernel's
// own common.h and attn_narrow_tile.h, whose functions the kernel calls, it checks on the CPU that operand reads name what
// the requests and the widening wrote, inside their tiles and without bank conflicts, and, for every workgroup of a launch,
// that its walk stays inside its own sequence and covers the keys its queries see.
//
//     attn_narrow_requests_audit <seq_len> <batch> <window_size> [rows q / kv really have, default seq_len * batch]
#include "common.h"
#include "attn_narrow_tile.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

namespace at = x17::attn_tile;
namespace nt = x17::attn_narrow_tile;

static int fail(char const *what, unsigned long long a, unsigned long long b) {
	std::printf("{\"ok\": false, \"error\": \"%s\", \"value\": %llu, \"limit\": %llu}\n", what, a, b);
	return 1;
}

int main(int argc, char **argv) {
	if (argc != 4 && argc != 5) {
		std::fprintf(stderr, "usage: %s <seq_len> <batch> <window_size> [allocated rows]\n", argv[0]);
		return 2;
	}
	unsigned const seq_len = (unsigned)std::strtoull(argv[1], nullptr, 10), batch = (unsigned)std::strtoull(argv[2], nullptr, 10);
	unsigned const window_size = (unsigned)std::strtoull(argv[3], nullptr, 10);
	constexpr unsigned HD = X17_HEAD_DIM, H = X17_N_HEADS, KV_STRIDE = X17_KV_STRIDE, CPR = at::CHUNKS_PER_ROW, KEYS = at::KV_PER_STEP;
	if (seq_len % 64 != 0 || seq_len < at::Q_PER_BLOCK || batch == 0 || (window_size != 0 && window_size % 16 != 0)) {
		return fail("the launcher rejects this shape (seq_len % 64, at least 128 rows, window % 16)", seq_len, at::Q_PER_BLOCK);
	}
	unsigned long long const rows = argc == 5 ? std::strtoull(argv[4], nullptr, 10) : (unsigned long long)seq_len * batch;
	unsigned const wr = at::rounded_window(window_size);

	// ---- K: thread t's request lands in stored chunk t; a read of (key, chunk) must name the thread that asked for it
	for (unsigned key = 0; key < KEYS; ++key) for (unsigned c = 0; c < CPR; ++c) {
		unsigned const off = at::k_chunk_offset(key, c);
		if (off + 16 > at::K_TILE_BYTES || !at::is_stager(off / 16)) return fail("a K read leaves the tile", off + 16, at::K_TILE_BYTES);
		if (at::stage_k_offset(off / 16, KV_STRIDE) != key * KV_STRIDE + 16 * c) return fail("a K read names a chunk that holds another key", key, c);
	}
	// the lanes' reads: key 16 tile + lane % 16, chunk 4 s + lane / 16 (head_dim 32: none above the row, chunk 0)
	for (unsigned lane = 0; lane < 64; ++lane) for (unsigned s = 0; s < (HD + 63) / 64; ++s) {
		if (16 * (lane / 16) < HD && 4 * s + lane / 16 >= CPR) return fail("a K read's chunk is outside the row", 4 * s + lane / 16, CPR);
	}
	// ---- V: thread t widens chunk t (in order) into granule (key t / CPR, t % CPR)
	std::vector<unsigned> written(at::V_TILE_BYTES / 32, 0);
	for (unsigned tid = 0; tid < at::THREADS_PER_BLOCK; ++tid) {
		if (!at::is_stager(tid)) continue;
		if (at::stage_v_offset(tid, KV_STRIDE) != (tid / CPR) * KV_STRIDE + HD + 16 * (tid % CPR)) return fail("a V chunk is not in order", tid, 0);
		unsigned const dst = nt::widened_offset(tid);
		if (dst % 32 != 0 || dst + 32 > at::V_TILE_BYTES) return fail("a widened granule leaves the tile", dst + 32, at::V_TILE_BYTES);
		++written[dst / 32];
	}
	for (unsigned v : written) if (v != 1) return fail("a granule of the f16 tile is not written exactly once", v, 1);
	// scores, probabilities and values meet in matrix row r of a 16-key tile: K read there, V stored there, keys 0-3, 8-11, 4-7, 12-15
	unsigned const quad_of_group[4] = {0, 2, 1, 3};
	for (unsigned r = 0; r < 16; ++r) {
		unsigned const key = nt::key_of_row(r);
		if (key != 4 * quad_of_group[r / 4] + r % 4) return fail("a matrix row holds another key", r, key);
		for (unsigned t = 0; t < 2; ++t) for (unsigned c = 0; c < CPR; ++c) {
			if (nt::widened_offset((16 * t + key) * CPR + c) != nt::v_granule_offset(16 * t + r, c)) return fail("a key's values are not in its scores' row", r, key);
		}
	}
	for (unsigned dt = 0; dt < HD / 16; ++dt) for (unsigned row0 = 0; row0 < 16; row0 += 8) {
		unsigned mask = 0;
		for (unsigned r = 0; r < 8; ++r) {
			unsigned const off = nt::v_granule_offset(row0 + r, dt);
			mask |= 1u << ((off >> 5) & 7);
			if (off + nt::SIXTEEN_KEYS != nt::v_granule_offset(16 + row0 + r, dt)) return fail("sixteen keys further is not a constant stride", off, nt::v_granule_offset(16 + row0 + r, dt));
		}
		if (mask != 0xFF) return fail("transposed reads of eight consecutive keys share a bank column", mask, 0xFF);
	}
	if (nt::SMEM_BYTES > 160 * 1024 || nt::SCALE_RING_OFFSET + (at::ROW_SCALES ? nt::RING * at::SCALE_TILE_BYTES : 0) > nt::SMEM_BYTES) return fail("LDS map", nt::SMEM_BYTES, 160 * 1024);

	// ---- the walk of every workgroup
	unsigned long long extent = 0, walked = 0;
	if (seq_len % nt::Q_PER_BLOCK != 0) return fail("query blocks do not divide the sequence", seq_len, nt::Q_PER_BLOCK);
	for (unsigned long long seq = 0; seq < batch; ++seq) for (unsigned q0 = 0; q0 < seq_len; q0 += nt::Q_PER_BLOCK) {
		unsigned const begin = at::first_key_block(q0, wr), end = nt::end_key_block(q0);
		if (end <= begin || end * KEYS > seq_len) return fail("the walk is empty or reaches behind its sequence", end * KEYS, seq_len);
		for (unsigned w = 0; w < at::Q_WAVES; ++w) {
			// the walk is that of the 32 queries the wavefront shares with its twin
			unsigned const qw = (q0 + w * nt::Q_PER_WAVE) & ~(nt::PAIR - 1), first = at::first_key_block(qw, wr), last = qw / KEYS;
			if (first < begin || last >= end) return fail("a wavefront's keys are outside its workgroup's walk", last, end);
			if (((q0 + w * nt::Q_PER_WAVE) ^ nt::Q_PER_WAVE) / nt::Q_PER_BLOCK != q0 / nt::Q_PER_BLOCK) return fail("a twin is in another workgroup", q0, w);
			// every key a query of the 32 sees: max(0, i - W') .. i - 1
			unsigned const lowest = qw > wr ? qw - wr : 0, highest = qw + nt::PAIR - 2;
			if (lowest / KEYS < first || highest / KEYS > last) return fail("a visible key is outside the wavefront's blocks", highest / KEYS, last);
			unsigned const inside = nt::first_inside_block(qw, wr);
			for (unsigned kb = first; kb < last; ++kb) {
				bool const whole = kb * KEYS + KEYS - 1 < qw && (unsigned long long)qw + nt::PAIR - 1 - kb * KEYS <= wr;
				if (whole != (kb >= inside)) return fail("a block is taken as fully visible and is not, or the other way round", kb, inside);
			}
		}
		unsigned const n = end - begin;
		for (unsigned t = 0; t < n + at::PREFETCH + 2; ++t) {
			unsigned const tile = t < n ? t : n - 1;       // (requests past the end repeat the last tile)
			unsigned long long const row_end = seq * seq_len + (unsigned long long)(begin + tile + 1) * KEYS;
			if (row_end > (seq + 1) * seq_len) return fail("tile reaches behind its sequence", row_end, (seq + 1) * seq_len);
			unsigned long long const byte_end = (row_end - 1) * KV_STRIDE + (unsigned long long)H * 2 * HD;
			if (byte_end > rows * KV_STRIDE) return fail("K/V request past the end of kv", byte_end, rows * KV_STRIDE);
			extent = byte_end > extent ? byte_end : extent;
		}
		walked += n;
	}
	std::printf("{\"ok\": true, \"steps\": %llu, \"kv_extent\": %llu, \"kv_bytes\": %llu}\n", walked * H, extent, rows * (unsigned long long)KV_STRIDE);
	return 0;
}
