// attn_bwd_tile.h -- tile geometry and LDS layouts of the attention backward-with-respect-to-q kernel (attn_d_q_i8.hip) as
// plain constexprs, shared with the host program that prints its meta.json and with the request audit
// (attn_bwd_requests_audit.cpp).  Needs X17_HEAD_DIM from common.h.
// The query blocking is the forward kernel's (attn_tile.h): 128 queries of one head per workgroup, a wavefront owns
// 32 queries, 32 keys per step.
#pragma once

#include "attn_tile.h"

namespace x17 { namespace attn_bwd_tile {

namespace at = x17::attn_tile;

constexpr unsigned THREADS_PER_BLOCK = at::THREADS_PER_BLOCK;
constexpr unsigned Q_PER_BLOCK = at::Q_PER_BLOCK;
// raw int8 K / V tiles are fetched PREFETCH steps ahead into rings of PREFETCH + 1 slots; one step before its use a
// tile is widened to f16 by the threads that fetched it, into one of two f16 tiles
constexpr unsigned PREFETCH = 3;
constexpr unsigned RING = PREFETCH + 1;
// 64 accumulators of dQ^T, the f16 dO fragments of all of head_dim and the forward's Q fragments stay in registers:
// two wavefronts per SIMD
constexpr unsigned WAVES_PER_SIMD = 2;

constexpr unsigned RAW_TILE_BYTES = at::KV_PER_STEP * at::HEAD_DIM;          // int8, as it arrives
constexpr unsigned F16_TILE_BYTES = at::KV_PER_STEP * at::HEAD_DIM * 2;
// LDS map: raw K ring | raw V ring | two f16 K tiles (granule layout, read transposed) | two f16 V tiles (row layout)
constexpr unsigned RAW_K_RING_OFFSET = 0;
constexpr unsigned RAW_V_RING_OFFSET = RING * RAW_TILE_BYTES;
constexpr unsigned K_F16_OFFSET = RAW_V_RING_OFFSET + RING * RAW_TILE_BYTES;
constexpr unsigned V_F16_OFFSET = K_F16_OFFSET + 2 * F16_TILE_BYTES;
constexpr unsigned SMEM_BYTES = V_F16_OFFSET + 2 * F16_TILE_BYTES;

constexpr unsigned CPR = at::CHUNKS_PER_ROW;                 // 16-byte chunks of an int8 row of the head

// f16 K tile, the forward's f16 V layout: 32-byte granule n = key * CPR + c (16 dims) lives in 256-byte line n / 8 at
// position (n % 8) ^ ((line & 3) << 1); the transposed 8-byte reads of 32 lanes then cover all banks once.
constexpr unsigned granule_offset(unsigned key, unsigned c) {
	unsigned const n = key * CPR + c, line = n >> 3;
	return (line << 8) | (((n & 7) ^ ((line & 3) << 1)) << 5);
}
// f16 V tile, read by rows: a key row is 2 * CPR chunks of 16 bytes (8 dims); 16 / (2 * CPR) keys share a 256-byte
// line, and chunk c16 of a key is stored at position c16 ^ line inside its key's part of the line: the sixteen keys
// a ds_read_b128 serves at a time (same c16) land in sixteen different slots for head_dim 32, 64 and 128.
constexpr unsigned vrow_offset(unsigned key, unsigned c16) {
	unsigned const R = 2 * CPR, KPL = 16 / R, line = key / KPL;
	return line * 256 + ((key % KPL) * R + (c16 ^ (line & (R - 1)))) * 16;
}
// Where staging thread `tid` puts the sixteen f16 of each raw chunk it requested.  Stored chunk `tid` of the raw K tile holds
// logical chunk n: key n / CPR, dims 16 * (n % CPR) .. + 15; the V tile is in order.
constexpr unsigned k_widened_offset(unsigned tid) {
	unsigned const line = tid >> 3, n = (line << 3) | ((tid & 7) ^ ((line >> 1) & 7));
	return granule_offset(n / CPR, n % CPR);
}
constexpr unsigned v_widened_offset(unsigned tid, unsigned half) { return vrow_offset(tid / CPR, 2 * (tid % CPR) + half); }

}} // namespace x17::attn_bwd_tile
