// attn_bwd_kv_tile.h -- tile geometry and index arithmetic of the attention backward-with-respect-to-k-and-v kernel
// (attn_d_kv_i8.hip) as plain constexprs, shared by the device code, the host program that prints its meta.json and the
// host-side audit of its tile requests (attn_bwd_kv_requests_audit.cpp).  Needs X17_HEAD_DIM from common.h.
// Structure of the reference's attn_d_kv.cuh:26-37: a workgroup owns a block of keys and walks the queries that see it.
#pragma once

#include "attn_tile.h"

namespace x17 { namespace attn_bwd_kv_tile {

namespace at = x17::attn_tile;

constexpr unsigned HEAD_DIM = at::HEAD_DIM;
constexpr unsigned KEY_WAVES = 4;
constexpr unsigned KEYS_PER_WAVE = 16;
constexpr unsigned KEYS_PER_BLOCK = KEY_WAVES * KEYS_PER_WAVE;        // 64 keys of one head per workgroup at a time
constexpr unsigned Q_PER_STEP = 32;                                    // queries staged per pipeline step
constexpr unsigned THREADS_PER_BLOCK = at::WAVE * KEY_WAVES;
// The launcher's smallest sequence is the forward's query block.  gridDim.x says into how many runs the sequence's key blocks
// are cut (a block each by this library's launchers, two where a grid is made of the forward's blocks).
constexpr unsigned LAUNCH_BLOCK = at::Q_PER_BLOCK;
constexpr unsigned blocks_per_run(unsigned seq_len, unsigned runs) { return (seq_len / KEYS_PER_BLOCK + runs - 1) / runs; }
// 16 keys per wavefront on the 16 x 16 matrix instructions: 64 accumulators (dK^T and dV^T of 16 keys x head_dim 128)
// and the keys' own K and V fragments leave room for three wavefronts per SIMD, i.e. three workgroups per compute unit.
// A wavefront issues one instruction in about ten clocks whatever its neighbours do, so a step takes its number of
// instructions times that, and what counts is how many wavefronts a SIMD has (four, at 128 registers, spill inside the
// loop; with smaller heads they do not).
constexpr unsigned WAVES_PER_SIMD = HEAD_DIM == 128 ? 3 : 4;

constexpr unsigned CPR = at::CHUNKS_PER_ROW;                // 16-byte chunks of an int8 row of the head
constexpr unsigned WIDE_CPR = 2 * CPR;                      // ... of a bf16 row
constexpr unsigned Q_STAGERS = Q_PER_STEP * CPR;            // threads that request the raw Q tile: 16-byte chunk t each; they widen it
constexpr unsigned WIDE_CHUNKS = Q_PER_STEP * WIDE_CPR;
// dO requests: thread t < WIDE_STAGERS asks for chunk t and, where the tile has more chunks than the workgroup threads, for
// chunk t + WIDE_STAGERS, sixteen rows further
constexpr unsigned WIDE_STAGERS = WIDE_CHUNKS < THREADS_PER_BLOCK ? WIDE_CHUNKS : THREADS_PER_BLOCK;
constexpr unsigned WIDE_PASSES = WIDE_CHUNKS / WIDE_STAGERS;
static_assert(WIDE_STAGERS % at::WAVE == 0 && Q_STAGERS % at::WAVE == 0 && Q_STAGERS <= THREADS_PER_BLOCK, "whole wavefronts request, one chunk per lane");
static_assert(WIDE_PASSES == 1 || (WIDE_PASSES == 2 && WIDE_STAGERS == 16 * WIDE_CPR), "the second pass starts sixteen rows further");
constexpr unsigned LD_WAVE = KEY_WAVES - 1;                 // the wavefront that requests the tile's L and D and makes its constants
constexpr unsigned Q_RAW_BYTES = Q_PER_STEP * HEAD_DIM;     // int8 queries as they arrive
constexpr unsigned WIDE_BYTES = Q_PER_STEP * HEAD_DIM * 2;  // a bf16 tile (dO as it arrives, Q widened)
constexpr unsigned LD_BYTES = 2 * Q_PER_STEP * 4;           // the tile's L and D values (f32)
constexpr unsigned CONST_BYTES = 3 * Q_PER_STEP * 4;        // the per-query constants temperature | L - lg2(255) | D
// LDS: raw Q ring (tiles requested three steps ahead, widened to bf16 one step before their use) | L and D ring | two dO tiles
// (requested one step ahead: a third one is the LDS of the third workgroup) | two widened Q tiles | two blocks of constants
constexpr unsigned RING = 4;
constexpr unsigned Q_RAW_OFFSET = 0;
constexpr unsigned LD_OFFSET = Q_RAW_OFFSET + RING * Q_RAW_BYTES;
constexpr unsigned DO_OFFSET = LD_OFFSET + RING * LD_BYTES;
constexpr unsigned Q_WIDE_OFFSET = DO_OFFSET + 2 * WIDE_BYTES;
constexpr unsigned CONST_OFFSET = Q_WIDE_OFFSET + 2 * WIDE_BYTES;
constexpr unsigned SMEM_BYTES = CONST_OFFSET + 2 * CONST_BYTES;
// at the end every wavefront turns its keys' rows (dK then dV, bf16) around in a region of its own over all of this
constexpr unsigned OUT_CPR = HEAD_DIM / 4;                  // 16-byte chunks of such a row
constexpr unsigned OUT_BYTES_PER_WAVE = KEYS_PER_WAVE * OUT_CPR * 16;
static_assert(KEY_WAVES * OUT_BYTES_PER_WAVE <= SMEM_BYTES, "the rows fit the workgroup's LDS");
constexpr unsigned out_offset(unsigned row, unsigned c) { return (row * OUT_CPR + (c ^ (row & (OUT_CPR - 1)))) * 16; }

// ---- the walk (sequence lengths are multiples of 64: key blocks divide them)
constexpr unsigned block_first_key(unsigned key_block_index) { return key_block_index * KEYS_PER_BLOCK; }
// last query that sees a key of [.., last_key]: query i sees key j iff j < i <= j + W' (wr: the rounded window, 2^32 - 1 = none)
constexpr unsigned last_seeing_query(unsigned last_key, unsigned wr, unsigned seq_len) {
	return wr >= seq_len || wr >= seq_len - 1 - last_key ? seq_len - 1 : last_key + wr;
}
// query tiles (Q_PER_STEP queries) walked for the keys [first_key, last_key]: [first, end)
constexpr unsigned first_query_tile(unsigned first_key) { return first_key / Q_PER_STEP; }
constexpr unsigned end_query_tile(unsigned last_key, unsigned wr, unsigned seq_len) { return last_seeing_query(last_key, wr, seq_len) / Q_PER_STEP + 1; }

// ---- LDS layouts (byte offsets inside a tile) and the requests that fill them.  A request moves 16 bytes per lane to
// consecutive LDS addresses, so a layout is made by choosing which chunk of the source a lane asks for: position p
// (in 16-byte units) of a tile receives the source chunk the *_source function names.
constexpr bool is_q_stager(unsigned tid) { return tid < Q_STAGERS; }
constexpr bool is_wide_stager(unsigned tid) { return tid < WIDE_STAGERS; }
// raw int8 Q tile: the forward's K tile layout (linear chunk n = row * CPR + c in 128-byte line n / 8 at position
// (n % 8) ^ ((line >> 1) & 7)): one request per staging thread
constexpr unsigned q_raw_offset(unsigned row, unsigned c) {
	unsigned const n = row * CPR + c, line = n >> 3;
	return (line << 7) | (((n & 7) ^ ((line >> 1) & 7)) << 4);
}
constexpr unsigned q_raw_logical_chunk(unsigned p) {
	unsigned const line = p >> 3;
	return (line << 3) | ((p & 7) ^ ((line >> 1) & 7));
}
constexpr unsigned q_raw_source(unsigned p, unsigned row_stride_bytes) {
	unsigned const n = q_raw_logical_chunk(p);
	return (n / CPR) * row_stride_bytes + (n % CPR) * 16;
}
// bf16 tile: a row is WIDE_CPR chunks of 16 bytes; 16 / WIDE_CPR rows share a 256-byte line and chunk c of a row sits at
// position c ^ key(line) inside its row's part of the line.  It is read in two ways, both without bank conflicts: by rows
// (eight dims of one query per lane; the same chunk of sixteen rows lands in sixteen different positions, key being a
// bijection), and transposed (eight queries of one dim per lane: the 32 lanes a ds_read_b64_tr_b16 serves at a time ask for the
// same two chunks of eight consecutive rows, which lie in eight different 32-byte columns, key / 2 being different for
// the lines of eight consecutive rows)
constexpr unsigned line_key(unsigned line) { return ((line << 1) | ((line & (WIDE_CPR - 1)) / (WIDE_CPR / 2))) & (WIDE_CPR - 1); }
constexpr unsigned rows_offset(unsigned row, unsigned c) {
	constexpr unsigned RPL = 16 / WIDE_CPR;
	unsigned const line = row / RPL;
	return line * 256 + ((row % RPL) * WIDE_CPR + (c ^ line_key(line))) * 16;
}
constexpr unsigned rows_source(unsigned p, unsigned row_stride_bytes) {
	constexpr unsigned RPL = 16 / WIDE_CPR;
	unsigned const line = p / 16, slot = p % 16;
	return (line * RPL + slot / WIDE_CPR) * row_stride_bytes + ((slot % WIDE_CPR) ^ line_key(line)) * 16;
}
// the eight bytes at dims 4 piece .. 4 piece + 3 of a row, as a transposed read asks for them
constexpr unsigned piece_offset(unsigned row, unsigned piece) { return rows_offset(row, piece / 2) + 8 * (piece % 2); }
// the same row's chunk (piece) `dims` dims further, dims a multiple of 16 above the lane's own: those address bits are flipped
constexpr unsigned dims_flip(unsigned dims) { return dims * 2; }
// Q tile int8 -> bf16: a staging thread widens the chunk it requested (16 codes), into two chunks that differ in address bit 4
constexpr unsigned widened_offset(unsigned tid) {
	unsigned const n = q_raw_logical_chunk(tid);
	return rows_offset(n / CPR, 2 * (n % CPR));
}

}} // namespace x17::attn_bwd_kv_tile
