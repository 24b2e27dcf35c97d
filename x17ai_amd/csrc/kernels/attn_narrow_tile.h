// attn_narrow_tile.h -- tile geometry and LDS layouts of the attention kernel with sixteen queries per wavefront
// (attn_fwd_i8_narrow.hip) as plain constexprs, shared with the host program that prints its meta.json and with the
// request audit (attn_narrow_requests_audit.cpp).  Key tiles, their requests and their rings are attn_tile.h's.
#pragma once

#include "attn_tile.h"

namespace x17 { namespace attn_narrow_tile {

namespace at = x17::attn_tile;

constexpr unsigned Q_PER_WAVE = 16;
constexpr unsigned Q_PER_BLOCK = at::Q_WAVES * Q_PER_WAVE;      // 64 queries of one head per workgroup
constexpr unsigned THREADS_PER_BLOCK = at::THREADS_PER_BLOCK;
constexpr unsigned RING = at::RING;

// LDS map: that of attn_tile.h
constexpr unsigned K_RING_OFFSET = at::K_RING_OFFSET;
constexpr unsigned RAW_V_RING_OFFSET = at::RAW_V_RING_OFFSET;
constexpr unsigned V_TILES_OFFSET = at::V_TILES_OFFSET;
constexpr unsigned SCALE_RING_OFFSET = at::SCALE_RING_OFFSET;
constexpr unsigned SMEM_BYTES = at::SMEM_BYTES;

// (sequence lengths are multiples of 64: query blocks divide them.)  One past the last key block a workgroup walks
constexpr unsigned end_key_block(unsigned q_block0) { return q_block0 / at::KV_PER_STEP + Q_PER_BLOCK / at::KV_PER_STEP; }
// A wavefront walks the key blocks of the 32 queries it shares with its twin (q_pair0 .. + 31).  First one inside the window of all
// of them: q_pair0 + 31 - 32 kb <= wr
constexpr unsigned PAIR = 2 * Q_PER_WAVE;
constexpr unsigned first_inside_block(unsigned q_pair0, unsigned wr) {
	return q_pair0 + PAIR - 1 > wr ? (q_pair0 + PAIR - 1 - wr + at::KV_PER_STEP - 1) / at::KV_PER_STEP : 0;
}

// Row r of a 16-key tile in the matrix instructions is key 4 j + r % 4 of it with j = 0, 2, 1, 3: bits 2 and 3 change places.  (Its own
// inverse; the keys of a lane group of four stay neighbours.)
constexpr unsigned key_of_row(unsigned r) { return (r & 3) | ((r & 4) << 1) | ((r & 8) >> 1); }

// f16 V tile, by matrix rows (row r of key block 16 * t: r = 16 t + row of the tile), read transposed: 32-byte granule n = r * CPR + c
// (16 dims) in 256-byte line n / 8 at position (n % 8) ^ (line % CPR): the 32 lanes a ds_read_b64_tr_b16 serves at a time ask for
// one granule of eight consecutive rows, which then lie in eight different 32-byte columns
constexpr unsigned v_granule_offset(unsigned row, unsigned c) {
	unsigned const n = row * at::CHUNKS_PER_ROW + c, line = n >> 3;
	return (line << 8) | (((n & 7) ^ (line & (at::CHUNKS_PER_ROW - 1))) << 5);
}
// where staging thread `tid` puts the chunk it widens: key tid / CPR, chunk tid % CPR
constexpr unsigned widened_offset(unsigned tid) {
	unsigned const key = tid / at::CHUNKS_PER_ROW;
	return v_granule_offset((key & 16) | key_of_row(key & 15), tid % at::CHUNKS_PER_ROW);
}
constexpr unsigned SIXTEEN_KEYS = 16 * at::HEAD_DIM * 2;       // bytes from a row's granule to that of the row sixteen further

}} // namespace x17::attn_narrow_tile
