// Host-side audit of the backward-with-respect-to-q kernel's K/V tile requests and LDS layouts.  Compiled with the kernel's own
// common.h and attn_bwd_tile.h -- the index arithmetic below IS the kernel's (attn_d_q_i8.hip calls the same functions) -- it
// checks on the CPU that every 16-byte position of the widened tiles is written once and every operand read stays inside its
// tile and finds the key and dims it is for; and it walks every workgroup of a launch (sequence, head, query block) through the
// request schedule: K and V tile min(s + 3, last) into ring slot (s + 3) % 4 behind the barrier of step s, where all requests but
// the last step's have landed.  Every tile a step multiplies or widens must have landed in the slot it is read from, no
// request may overwrite a slot that is still read, and every request and load must stay inside its operand and its sequence.
//
//     attn_bwd_requests_audit <seq_len> <batch> <window_size> [rows the operands really have, default seq_len * batch]
//
// No GPU is involved; a kernel whose requests would leave an operand is found here, not on the device.
#include "common.h"
#include "attn_bwd_tile.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

namespace at = x17::attn_tile;
namespace bt = x17::attn_bwd_tile;

static int fail(char const *what, unsigned long long a, unsigned long long b) {
	std::printf("{\"ok\": false, \"error\": \"%s\", \"value\": %llu, \"limit\": %llu}\n", what, a, b);
	return 1;
}

int main(int argc, char **argv) {
	if (argc != 4 && argc != 5) {
		std::fprintf(stderr, "usage: %s <seq_len> <batch> <window_size> [allocated rows]\n", argv[0]);
		return 2;
	}
	unsigned long long const seq_len_arg = std::strtoull(argv[1], nullptr, 10), batch = std::strtoull(argv[2], nullptr, 10);
	unsigned const window_size = (unsigned)std::strtoull(argv[3], nullptr, 10);
	constexpr unsigned HD = X17_HEAD_DIM, H = X17_N_HEADS, Q_STRIDE = X17_Q_STRIDE, KV_STRIDE = X17_KV_STRIDE, O_STRIDE = X17_O_STRIDE;
	constexpr unsigned CPR = bt::CPR, KEYS = at::KV_PER_STEP, RING = bt::RING;
	if (seq_len_arg % 64 != 0 || seq_len_arg < at::Q_PER_BLOCK || batch == 0 || seq_len_arg * batch > 0xFFFFFFFFull
	    || (window_size != 0 && window_size % 16 != 0)) {
		return fail("the launcher rejects this shape (seq_len % 64, at least one query block, window % 16)", seq_len_arg, at::Q_PER_BLOCK);
	}
	unsigned const seq_len = (unsigned)seq_len_arg, wr = at::rounded_window(window_size);
	unsigned long long const rows = argc == 5 ? std::strtoull(argv[4], nullptr, 10) : seq_len_arg * batch;

	// ---- tiles: what lands where.  A 16-byte position is named key * HD + first dim + 1 (0: nothing).
	std::vector<unsigned> raw_k(KEYS * CPR, 0), raw_v(KEYS * CPR, 0), k_f16(2 * KEYS * CPR, 0), v_f16(2 * KEYS * CPR, 0);
	unsigned stagers = 0;
	for (unsigned tid = 0; tid < bt::THREADS_PER_BLOCK; ++tid) {
		if (!at::is_stager(tid)) continue;
		++stagers;
		unsigned const ko = at::stage_k_offset(tid, KV_STRIDE), vo = at::stage_v_offset(tid, KV_STRIDE);
		unsigned const kr = ko / KV_STRIDE, kc = ko % KV_STRIDE, vr = vo / KV_STRIDE, vc = vo % KV_STRIDE;
		if (kr >= KEYS || vr >= KEYS) return fail("a staging thread's key row is outside the tile", kr > vr ? kr : vr, KEYS);
		if (kc % 16 != 0 || kc + 16 > HD) return fail("a K chunk leaves the head's K columns", kc + 16, HD);
		if (vc % 16 != 0 || vc < HD || vc + 16 > 2 * HD) return fail("a V chunk leaves the head's V columns", vc + 16, 2 * HD);
		if (raw_k[tid] != 0 || raw_v[tid] != 0) return fail("a raw position is requested twice", tid, 1);
		raw_k[tid] = kr * HD + kc + 1;
		raw_v[tid] = vr * HD + (vc - HD) + 1;
		for (unsigned half = 0; half < 2; ++half) {
			unsigned const kd = bt::k_widened_offset(tid) + 16 * half, vd = bt::v_widened_offset(tid, half);
			if (kd % 16 != 0 || kd + 16 > bt::F16_TILE_BYTES || vd % 16 != 0 || vd + 16 > bt::F16_TILE_BYTES) return fail("a widened chunk leaves its tile", kd > vd ? kd : vd, bt::F16_TILE_BYTES);
			if (k_f16[kd / 16] != 0 || v_f16[vd / 16] != 0) return fail("a widened position is written twice", kd, vd);
			k_f16[kd / 16] = kr * HD + kc + 8 * half + 1;
			v_f16[vd / 16] = vr * HD + (vc - HD) + 8 * half + 1;
		}
	}
	if (stagers != KEYS * CPR) return fail("number of staging threads", stagers, KEYS * CPR);
	// ---- the operand reads (every lane of a wavefront)
	for (unsigned lane = 0; lane < 64; ++lane) {
		unsigned const half = lane / 32, qlane = lane % 32, t = lane % 16, dh = (lane / 16) % 2;
		for (unsigned s = 0; s < HD / 32; ++s) {
			unsigned const off = at::k_chunk_offset(qlane, 2 * s + half);
			if (off % 16 != 0 || off + 16 > bt::RAW_TILE_BYTES || raw_k[off / 16] != qlane * HD + 32 * s + 16 * half + 1) return fail("a raw K read finds another chunk", off, lane);
		}
		for (unsigned sl = 0; sl < HD / 16; ++sl) {
			unsigned const off = bt::vrow_offset(qlane, 2 * sl + half);
			if (off % 16 != 0 || off + 16 > bt::F16_TILE_BYTES || v_f16[off / 16] != qlane * HD + 16 * sl + 8 * half + 1) return fail("a V row read finds another chunk", off, lane);
		}
		for (unsigned tile = 0; tile < 2; ++tile) {
			for (unsigned db = 0; db < HD / 32; ++db) {
				for (unsigned upper = 0; upper < 2; ++upper) {          // keys 4 half + t / 4 and eight further, four dims each
					unsigned const base = upper == 0 || CPR >= 4 ? bt::granule_offset(4 * half + (t >> 2), 2 * db + dh) + 8 * (t & 3) + (upper ? 8 * CPR * 32 : 0)
					                                             : bt::granule_offset(8 + 4 * half + (t >> 2), 2 * db + dh) + 8 * (t & 3);
					unsigned const off = base + tile * (16 * CPR * 32);
					unsigned const key = 16 * tile + 8 * upper + 4 * half + (t >> 2), dim = 32 * db + 16 * dh + 4 * (t & 3);
					if (off % 8 != 0 || off + 8 > bt::F16_TILE_BYTES || k_f16[off / 16] != key * HD + dim / 8 * 8 + 1 || off % 16 != (dim % 8) * 2) return fail("a transposed K read finds another key or dim", off, lane);
				}
			}
		}
	}

	// ---- the walks
	unsigned long long requests = 0, kv_extent = 0, q_extent = 0, o_extent = 0, row_extent = 0;
	unsigned const q_blocks = (seq_len + at::Q_PER_BLOCK - 1) / at::Q_PER_BLOCK;
	for (unsigned long long seq = 0; seq < batch; ++seq) {
		unsigned long long const row_base = seq * seq_len;
		for (unsigned qb = 0; qb < q_blocks; ++qb) {
			unsigned const q0 = at::block_first_query(qb, seq_len);
			if (q0 % 64 != 0 || q0 + at::Q_PER_BLOCK > seq_len) return fail("query block leaves its sequence", q0 + at::Q_PER_BLOCK, seq_len);
			unsigned const kb_begin = at::first_key_block(q0, wr), kb_end = at::end_key_block(q0);
			if (kb_end <= kb_begin || kb_end - kb_begin < RING) return fail("a workgroup walks fewer tiles than its ring holds", kb_end - kb_begin, RING);
			unsigned const n_steps = kb_end - kb_begin, last = n_steps - 1;
			std::vector<unsigned> slot_of_request, tile_of_request;
			auto request = [&](unsigned slot, unsigned t) -> int {
				if (t > last) return fail("request for a tile behind the walk's last", t, last);
				unsigned long long const first_key = (unsigned long long)(kb_begin + t) * KEYS;
				if (first_key + KEYS > seq_len) return fail("tile reaches behind its sequence", first_key + KEYS, seq_len);
				for (unsigned head = 0; head < H; head += H - 1 ? H - 1 : 1) {       // first and last head bound the columns
					unsigned long long const end = (row_base + first_key + KEYS - 1) * KV_STRIDE + (unsigned long long)head * 2 * HD + 2 * HD;
					if (end > rows * KV_STRIDE) return fail("K/V request past the end of kv", end, rows * KV_STRIDE);
					kv_extent = end > kv_extent ? end : kv_extent;
				}
				slot_of_request.push_back(slot);
				tile_of_request.push_back(t);
				requests += 2ull * stagers;
				return 0;
			};
			// the tile that has landed last in a slot when all requests but the newest `in_flight` have (-1: none), or -2 while a
			// request into that slot is under way
			auto landed = [&](unsigned slot, unsigned in_flight) -> long long {
				long long tile = -1;
				for (unsigned r = 0; r < slot_of_request.size(); ++r) {
					if (slot_of_request[r] != slot) continue;
					tile = r + in_flight < slot_of_request.size() ? (long long)tile_of_request[r] : -2;
				}
				return tile;
			};
			for (unsigned j = 0; j < bt::PREFETCH; ++j) if (int rc = request(j, j)) return rc;
			unsigned src_tile = bt::PREFETCH;
			if (landed(0, 2) != 0) return fail("tile 0 has not landed when it is widened", 0, 0);          // vmcnt(4)
			std::vector<int> widened = {0, -1};
			for (unsigned s = 0; s < n_steps; ++s) {
				// vmcnt(2), barrier: the newest request may be in flight
				if (s <= last && landed(s % RING, 1) != (long long)s) return fail("a step reads a raw tile that is not there", s, n_steps);
				if (widened[s & 1] != (int)s) return fail("a step reads widened tiles that are not there", s, n_steps);
				if (s + 1 <= last && landed((s + 1) % RING, 1) != (long long)s + 1) return fail("a step widens a tile that has not landed", s + 1, n_steps);
				// its own request goes into a slot nobody reads in this step or widens from
				unsigned const slot = (s + bt::PREFETCH) % RING;
				if (slot == s % RING || slot == (s + 1) % RING) return fail("a request overwrites a slot that is read", slot, s);
				if (int rc = request(slot, src_tile)) return rc;
				if (at::further_tile_exists(s, n_steps)) ++src_tile;
				widened[(s + 1) & 1] = s + 1 <= last ? (int)s + 1 : -1;
			}
			if (src_tile != last) return fail("the source pointer does not end on the last tile", src_tile, last);
			// the runs of each wavefront: idle, masked, fully visible, the diagonal, idle; the unrolled trips have a further tile each
			for (unsigned wave = 0; wave < at::Q_WAVES; ++wave) {
				unsigned const w0 = q0 + wave * at::Q_PER_WAVE, first = at::first_key_block(w0, wr), diagonal = w0 / KEYS;
				unsigned const inside = w0 + 31 > wr ? (w0 + 62 - wr) / 32 : 0;
				unsigned const full = inside < first ? first : (inside > diagonal ? diagonal : inside);
				if (first < kb_begin || diagonal >= kb_end) return fail("a wavefront's blocks leave the workgroup's walk", first, diagonal);
				for (unsigned kb = kb_begin; kb < kb_end; ++kb) {
					bool any = false, all = true;
					for (unsigned q = w0; q < w0 + at::Q_PER_WAVE; ++q) {
						for (unsigned key = kb * KEYS; key < kb * KEYS + KEYS; ++key) {
							bool const visible = key < q && q - 1 - key <= wr - 1;
							any |= visible;
							all &= visible;
						}
					}
					if (any && (kb < first || kb > diagonal)) return fail("a visible key in an idle step", kb, w0);
					if (!all && kb >= full && kb < diagonal) return fail("a hidden key in a step without a mask", kb, w0);
				}
				unsigned i = full - kb_begin;
				unsigned const d = diagonal - kb_begin;
				for (; i < d && i % RING != 0; ++i) {}
				for (; i + RING <= d && i + 2 * RING <= n_steps; i += RING) {
					for (unsigned j = 0; j < RING; ++j) if (!at::further_tile_exists(i + j, n_steps)) return fail("an unrolled step without a further tile", i + j, n_steps);
				}
			}
			unsigned long long const row_end = row_base + q0 + at::Q_PER_BLOCK;
			unsigned long long const q_end = (row_end - 1) * Q_STRIDE + (unsigned long long)H * HD, o_end = (row_end - 1) * O_STRIDE + (unsigned long long)H * HD;
			if (q_end > rows * Q_STRIDE || o_end > rows * O_STRIDE || row_end > rows) return fail("query rows past the end of q, out, d_out, L or D", row_end, rows);
			q_extent = q_end > q_extent ? q_end : q_extent;
			o_extent = o_end > o_extent ? o_end : o_extent;
			row_extent = row_end > row_extent ? row_end : row_extent;
		}
	}
	std::printf("{\"ok\": true, \"workgroups\": %llu, \"requests\": %llu, \"kv_extent\": %llu, \"kv_bytes\": %llu, \"q_extent\": %llu, \"q_bytes\": %llu, "
	            "\"o_extent\": %llu, \"o_bytes\": %llu, \"row_extent\": %llu, \"rows\": %llu}\n",
	            batch * q_blocks * H, requests * H, kv_extent, rows * KV_STRIDE, q_extent, rows * Q_STRIDE, o_extent, rows * O_STRIDE, row_extent, rows);
	return 0;
}
