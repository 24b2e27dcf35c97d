// gemm_b8_small.hip -- the GEMM of gemm_b8.hip (same operands, writers and module ABI) over small tiles, for launches
// whose output has too few 256 x 256 tiles to fill the chip.
//
// With 256 token rows a 4096-column product is sixteen 256 x 256 tiles: sixteen of 256 compute units work, each through
// the whole of K.  Here a workgroup owns 64 x 64 outputs (or 128 x 128: X17_SMALL_TILE).  With int8 operands its
// wavefronts split K: every wavefront computes the whole 64 x 64 block over its part of each K step, so that the operand
// fragments it reads from LDS are used as often as in a large tile (16 bytes of fragment per lane and matrix
// instruction), and the partial sums are exchanged through LDS once at the end, each wavefront finishing and writing a
// part of the block.  Sums of e4m3 operands are float32 and depend on their order: there a wavefront walks all of K for
// a block of its own (32 x 32 of the 64 x 64; of the 128 x 128 64 x 32, and 64 x 64 of e4m3 x int8), in the 256 x 256
// kernel's order, and every form gives that kernel's bytes.
// What bounds int8 and e4m3 is the stream of tiles from L2 / HBM into LDS: X17_SMALL_STAGES - 1 K steps of requests are
// kept in flight per workgroup, one barrier per step.
// e4m3 x int8 in 64 x 64 tiles is bound by the instructions around the f16 matrix instructions, which one wavefront per SIMD
// issues at one in about ten clocks.  Of 34 per 32 bytes of K twenty widened a weight fragment, the same one in two
// wavefronts; four further wavefronts now do that once, from memory through registers, and leave f16 in LDS (gemm_small_tile.h:
// WIDEN_ONCE).  256 rows, 4096 columns, K = 8192: 34.8 -> 30.7 us (39.1 -> 34 with weights from memory; vector ALU 28 %, matrix
// cores 21 %, LDS 37 % busy: the step's chain barrier - reads - widening - multiplications bounds it); 320 rows, two
// workgroups per compute unit: 61 -> 44 us.  Tried: token tiles through the same registers 34.6 / 49.7 us, half a step's
// fragments read across the barrier from a third widened tile 32.2 / 45.5 us.

#include "common.h"
#include "x17_device.h"
#include "gemm_small_tile.h"

using namespace x17;
namespace gt = x17::gemm_small_tile;
namespace {
// after the exchange a wavefront writes 32-column blocks one at a time; the head-normalising writers need all 128 columns
constexpr int LANE_COLS = gt::NATURAL ? 64 : 16;
}
#include "gemm_parts.h"

// Two workgroups of eight wavefronts share a compute unit in the two-stage 128 x 128 form: 128 registers each.  The compiler
// unrolls loops of 9 .. 28 steps altogether, and with e4m3 fragments (two steps' worth are 96 registers) it then spills;
// unrolled by two it does not, unless a step is left over (K = 2048, 8192 columns, 2048 rows: 41.1 -> 38.5 us).
#if X17_A_KIND == 1 && X17_B_KIND == 1 && X17_SMALL_TILE == 128 && X17_SMALL_STAGES == 2 && X17_A_COLS > 1024
#if X17_A_COLS / 128 % 2
#define X17_SMALL_LOOP_PRAGMA _Pragma("clang loop unroll(disable)")
#else
#define X17_SMALL_LOOP_PRAGMA _Pragma("clang loop unroll_count(2)")
#endif
#else
#define X17_SMALL_LOOP_PRAGMA
#endif

namespace {

constexpr u32 K_STEPS = K_TOTAL / gt::K_STEP;
constexpr u32 X_TILE_BYTES = gt::M_PER_BLOCK * ROW_BYTES;
constexpr u32 LOADS_PER_STAGE = gt::X_UNITS + gt::W_UNITS;
constexpr u32 SLICES_PER_WAVE = SLICES / gt::WAVES_K;
static_assert(SLICES_PER_WAVE * gt::WAVES_K == SLICES, "K steps divide evenly over the wavefronts that share a block");
static_assert(N_RAW % gt::N_PER_BLOCK == 0, "raw output columns are whole tiles");
// One workgroup of one or two wavefronts per SIMD fills a compute unit in the four-stage forms, and nothing runs beside a
// step's start: there the fragment reads go out in front of the requests' instructions, and all before anything waits for
// one.  What it gives depends on where the weights come from.  us, requests first / reads first, from L2 or the memory-side
// cache | from memory (128 x 128, 4096 columns unless said):
//   int8, K = 8192, 512 rows              28.7 / 26.1 | 37.5 / 36.9      int8, K = 2048, 256 rows   8.9 / 8.5 | 8.9 / 8.5
//   int8 GeGLU, 16384 columns, K = 2048, 256 rows (256 workgroups)       12.0 / 11.7 | 14.9 / 14.6
//   e4m3, K = 16384, 8192 columns, 320 rows            61 / 56 | 72.6 / 71.6: a pair whose weights no cache holds gains 1 %
// No launch of 58 lost.  (The first slice's reads alone: half of it.)  In the two-stage form the other workgroup runs beside a
// step's start, and a request that goes out later is waited for (int8, 512 rows x 16384 columns: 18.7 and 20.1 us).
constexpr bool READS_FIRST = gt::STAGES >= 4;

// the exchange: blocks of 32 x 32 outputs, 16 registers per lane; block j belongs to wavefront owner(j) of the WAVES_K
constexpr int BLOCKS = BN * BM;
constexpr u32 BLOCK_BYTES = 64 * 64;
constexpr u32 owner(int j) { return gt::NATURAL ? 0 : (u32)j * gt::WAVES_K / BLOCKS; }
// where wavefront `from` leaves its sums of block j, which it does not own
constexpr u32 GROUP_BYTES = BLOCKS * (gt::WAVES_K - 1) * BLOCK_BYTES;
X17_DEV u32 exchange_offset(int j, u32 from) { return (j * (gt::WAVES_K - 1) + (from < owner(j) ? from : from - 1)) * BLOCK_BYTES; }
static_assert(gt::WAVES / gt::WAVES_K * GROUP_BYTES <= gt::SMEM_BYTES, "the exchange fits the ring");

// The widening form's second half of a workgroup: weights from memory into registers, WIDENER_DEPTH K steps ahead, and from
// there as f16 into the tile behind the one the matrix wavefronts are at, widened one step before that.  Past the
// end the last step is loaded again, into tiles nobody reads any more.
[[maybe_unused]] X17_DEV void widen_and_store(u8 *smem, u8 const *b_tile, u32 widener, u32 lane) {
	constexpr u32 UNITS = gt::WIDENER_UNITS;
	u32 src[UNITS];
	u8 *dst[UNITS][2];
	X17_UNROLL for (u32 u = 0; u < UNITS; ++u) {
		u32 const row = gt::widener_row(widener, u, lane), chunk = gt::widener_chunk(lane);
		src[u] = gt::w_source_row(row) * K_TOTAL + 16 * chunk;
		X17_UNROLL for (u32 h = 0; h < 2; ++h) dst[u][h] = smem + gt::WIDE_OFFSET + gt::wide_offset(row, 2 * chunk + h);
	}
	// (buffer loads: lane offset and step's offset need no vector arithmetic; bounded by the tile's rows)
	auto const rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<u8 *>(b_tile), 0, gt::N_PER_BLOCK * K_TOTAL, 0x00020000);
	v4i raw[gt::WIDENER_DEPTH][UNITS];
	v8h wide[UNITS][2];
	auto load = [&](u32 step, u32 slot) __attribute__((always_inline)) {
		u32 const k0 = (step < K_STEPS ? step : K_STEPS - 1) * gt::K_STEP;
		X17_UNROLL for (u32 u = 0; u < UNITS; ++u) raw[slot][u] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rows, src[u], k0, 0));
	};
	auto widen = [&](u32 slot) __attribute__((always_inline)) {
		X17_UNROLL for (u32 u = 0; u < UNITS; ++u) {
			X17_UNROLL for (u32 h = 0; h < 2; ++h) wide[u][h] = widen8(raw[slot][u][2 * h], raw[slot][u][2 * h + 1], B_KIND);
		}
	};
	auto store = [&](u32 tile) __attribute__((always_inline)) {
		X17_UNROLL for (u32 u = 0; u < UNITS; ++u) {
			X17_UNROLL for (u32 h = 0; h < 2; ++h) *reinterpret_cast<v8h *>(dst[u][h] + tile * gt::WIDE_BYTES) = wide[u][h];
		}
	};
	X17_UNROLL for (u32 d = 0; d < gt::WIDENER_DEPTH; ++d) load(d, d);
	X17_UNROLL for (u32 d = 0; d < gt::WIDE_TILES; ++d) {
		widen(d);
		load(d + gt::WIDENER_DEPTH, d);
		if (d + 1 < gt::WIDE_TILES) store(d);
	}
	for (u32 base = 0; base < K_STEPS; base += gt::WIDENER_DEPTH) {
		X17_UNROLL for (u32 j = 0; j < gt::WIDENER_DEPTH; ++j) {
			if (base + j < K_STEPS) {
				step_barrier();
				__builtin_amdgcn_sched_barrier(0);
				store((j + 1) % gt::WIDE_TILES);
				widen((j + 2) % gt::WIDENER_DEPTH);
				load(base + j + 2 + gt::WIDENER_DEPTH, (j + 2) % gt::WIDENER_DEPTH);
			}
		}
	}
}

} // namespace

extern "C" __global__ __launch_bounds__(gt::THREADS_PER_BLOCK)
__attribute__((amdgpu_waves_per_eu(gt::WAVES_PER_SIMD)))
void kernel(
	u8 const *a, u32 a_rows,
	u8 const *b, u32 b_rows,
	u8 *c
#if X17_EPILOGUE == 3
	, f32 *rrms
#elif X17_EPILOGUE == 2
	, i8 const *residual
#elif X17_EPILOGUE == 4
	, f32 const *row_scale, f32 const *col_scale
#elif X17_EPILOGUE == 5
	, u16 const *q_norm_scales
#elif X17_EPILOGUE == 6
	, f32 *rrms, u8 const *b_kv, u8 *c_kv
#endif
) {
	extern __shared__ __attribute__((aligned(1024))) u8 smem[];
	(void)b_rows;

	u32 const tiles = ((a_rows + gt::M_PER_BLOCK - 1) / gt::M_PER_BLOCK) * (N_RAW / gt::N_PER_BLOCK);
	u32 const group = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
	if (group >= tiles) return;
	gt::TileOrigin const tile = gt::tile_origin(group, a_rows, N_RAW);

	u32 const tid = threadIdx.x;
	u32 const lane = tid % 64;
	u32 const wave = __builtin_amdgcn_readfirstlane(tid / 64);
	u32 const half = lane / 32;
	u32 const wk = wave % gt::WAVES_K;
	u32 const wn = (wave / gt::WAVES_K) % gt::WAVES_N;
	u32 const wm = wave / (gt::WAVES_K * gt::WAVES_N);

	u8 const *a_tile = a + (size_t)tile.m * K_TOTAL;
#if X17_EPILOGUE == 6
	static_assert(X17_Q_COLS % gt::N_PER_BLOCK == 0, "the q part is whole tiles");
	u8 const *b_tile = tile.n < X17_Q_COLS ? b + (size_t)tile.n * K_TOTAL : b_kv + (size_t)(tile.n - X17_Q_COLS) * K_TOTAL;
#else
	u8 const *b_tile = b + (size_t)tile.n * K_TOTAL;
#endif

	if constexpr (gt::WIDEN_ONCE) {
		if (wave >= gt::WAVES) {
			widen_and_store(smem, b_tile, wave - gt::WAVES, lane);
			return;
		}
	}

	// ---- requests: this wavefront's units of the token tile and of the weight tile
	u32 x_src[gt::X_UNITS], w_src[gt::W_UNITS];
	X17_UNROLL for (u32 u = 0; u < gt::X_UNITS; ++u) {
		u32 const unit = wave * gt::X_UNITS + u;
		x_src[u] = gt::unit_row(unit, lane) * K_TOTAL + 16 * gt::unit_chunk(unit, lane);
	}
	X17_UNROLL for (u32 u = 0; u < gt::W_UNITS; ++u) {
		u32 const unit = wave * gt::W_UNITS + u;
		w_src[u] = gt::w_source_row(gt::unit_row(unit, lane)) * K_TOTAL + 16 * gt::unit_chunk(unit, lane);
	}
	u8 *const x_dst = smem + wave * gt::X_UNITS * 1024;
	u8 *const w_dst = smem + X_TILE_BYTES + wave * gt::W_UNITS * 1024;
	// past the end the last step is requested again, into a slot nobody reads any more: the waits stay constant
	auto request = [&](u32 step, u32 slot) __attribute__((always_inline)) {
		u32 const k0 = (step < K_STEPS ? step : K_STEPS - 1) * gt::K_STEP;
		X17_UNROLL for (u32 u = 0; u < gt::X_UNITS; ++u) load_to_lds_16(x_dst + slot * gt::STAGE_BYTES + u * 1024, a_tile + k0, x_src[u]);
		X17_UNROLL for (u32 u = 0; u < gt::W_UNITS; ++u) load_to_lds_16(w_dst + slot * gt::STAGE_BYTES + u * 1024, b_tile + k0, w_src[u]);
	};
	if constexpr (!gt::WIDEN_ONCE) {
		X17_UNROLL for (u32 s = 0; s + 1 < gt::STAGES; ++s) request(s, s);
	}

	Acc acc[BN][BM];
	X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
		X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
			X17_UNROLL for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0;
		}
	}
	u32 const swz = gt::swizzle(lane % 32);
	u32 const x_off = (wm * gt::WAVE_M + lane % 32) * ROW_BYTES;
	u32 const w_off = X_TILE_BYTES + (wn * gt::WAVE_N + lane % 32) * ROW_BYTES;

	if constexpr (gt::WIDEN_ONCE) {
		// a lane's fragments in a token and in a widened tile; the rings' positions are immediates beside them
		u8 const *x_at[SLICES], *w_at[SLICES][2];
		X17_UNROLL for (u32 s = 0; s < SLICES; ++s) {
			x_at[s] = smem + x_off + (((2 * s + half) ^ swz) << 4);
			X17_UNROLL for (u32 h = 0; h < 2; ++h) {
				w_at[s][h] = smem + gt::WIDE_OFFSET + gt::wide_offset(wn * gt::WAVE_N + lane % 32, 4 * s + 2 * half + h);
			}
		}
		auto request_x = [&](u32 step, u32 to) __attribute__((always_inline)) {
			u8 const *const from = a_tile + (step < K_STEPS ? step : K_STEPS - 1) * gt::K_STEP;
			X17_UNROLL for (u32 u = 0; u < gt::X_UNITS; ++u) load_to_lds_16(x_dst + to * gt::STAGE_BYTES + u * 1024, from, x_src[u]);
		};
		X17_UNROLL for (u32 s = 0; s + 1 < gt::STAGES; ++s) request_x(s, s);
		static_assert(!gt::WIDEN_ONCE || gt::STAGES % gt::WIDE_TILES == 0, "one loop over both rings");
		for (u32 base = 0; base < K_STEPS; base += gt::STAGES) {
			X17_UNROLL for (u32 j = 0; j < gt::STAGES; ++j) {
				if (base + j < K_STEPS) {
					// this wavefront's requests of the step have landed and its reads of the step before are done; behind the barrier
					// so are everybody's, the step's weights are widened, and the slot of the token tile before is free
					wait_vmcnt<(gt::STAGES - 2) * gt::X_UNITS>();
					step_barrier();
					__builtin_amdgcn_sched_barrier(0);
					v4i raw[SLICES];
					v8h wide[SLICES][2];
					X17_UNROLL for (u32 s = 0; s < SLICES; ++s) {
						raw[s] = *reinterpret_cast<v4i const *>(x_at[s] + j * gt::STAGE_BYTES);
						X17_UNROLL for (u32 h = 0; h < 2; ++h) wide[s][h] = *reinterpret_cast<v8h const *>(w_at[s][h] + j % gt::WIDE_TILES * gt::WIDE_BYTES);
					}
					__builtin_amdgcn_sched_barrier(0);      // (all reads are on their way before anything waits for one)
					request_x(base + j + gt::STAGES - 1, (j + gt::STAGES - 1) % gt::STAGES);
					X17_UNROLL for (u32 s = 0; s < SLICES; ++s) {
						X17_UNROLL for (u32 h = 0; h < 2; ++h) {        // mma_slice's order
							v8h const xf = widen8(raw[s][2 * h], raw[s][2 * h + 1], A_KIND);
							v16f const r = __builtin_amdgcn_mfma_f32_32x32x16_f16(wide[s][h], xf, __builtin_bit_cast(v16f, acc[0][0]), 0, 0, 0);
							acc[0][0] = __builtin_bit_cast(Acc, r);
						}
					}
				}
			}
		}
	}
	u32 slot = 0;
	X17_SMALL_LOOP_PRAGMA
	for (u32 ks = 0; ks < (gt::WIDEN_ONCE ? 0 : K_STEPS); ++ks) {
		// this wavefront's requests of step ks have landed and its reads of step ks - 1 are done; behind the barrier so
		// are everybody's, and the slot of step ks - 1 takes the requests of step ks + STAGES - 1
		wait_vmcnt<(gt::STAGES - 2) * LOADS_PER_STAGE>();
		step_barrier();
		u8 const *stage = smem + slot * gt::STAGE_BYTES;
		Frags frags[SLICES_PER_WAVE];
		auto read = [&](u32 s) __attribute__((always_inline)) {
			load_frags(frags[s], stage + w_off, stage + x_off, wk * SLICES_PER_WAVE + s, half, swz);
		};
		u32 const free_slot = slot == 0 ? gt::STAGES - 1 : slot - 1;
		if constexpr (READS_FIRST) {
			X17_UNROLL for (u32 s = 0; s < SLICES_PER_WAVE; ++s) read(s);
			__builtin_amdgcn_sched_barrier(0);
			request(ks + gt::STAGES - 1, free_slot);
		} else {
			request(ks + gt::STAGES - 1, free_slot);
			X17_UNROLL for (u32 s = 0; s < SLICES_PER_WAVE; ++s) read(s);
		}
		X17_UNROLL for (u32 s = 0; s < SLICES_PER_WAVE; ++s) mma_slice(frags[s], acc);
		slot = slot + 1 == gt::STAGES ? 0 : slot + 1;
	}

	// ---- the wavefronts that share a block add up their partial sums: each writes the blocks it does not own, the
	// owner reads them back.  (The last requests write the ring too: they must have landed, everywhere.)
	wait_vmcnt<0>();
	u8 *const exchange = smem + (wave / gt::WAVES_K) * GROUP_BYTES + lane * 16;
	if constexpr (gt::WAVES_K > 1) {
		__builtin_amdgcn_s_waitcnt(0xC07F);
		__builtin_amdgcn_s_barrier();
		X17_UNROLL for (int j = 0; j < BLOCKS; ++j) {
			if (owner(j) != wk) {
				X17_UNROLL for (int q = 0; q < 4; ++q) {
					Acc const v = acc[j / BM][j % BM];
					*reinterpret_cast<v4i *>(exchange + exchange_offset(j, wk) + q * 1024) = v4i{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
				}
			}
		}
		__syncthreads();
	}

	u32 const row0 = tile.m + wm * gt::WAVE_M + lane % 32;
	u32 const col0 = tile.n + wn * gt::WAVE_N;                 // the wavefront's first raw column
	auto total_of = [&](int j, f32 (&x)[16]) __attribute__((always_inline)) {
		if constexpr (ACC_F32) {
			v16f const sum = __builtin_bit_cast(v16f, acc[j / BM][j % BM]);
			X17_UNROLL for (int r = 0; r < 16; ++r) x[r] = sum[r];
		} else {
			Acc sum = acc[j / BM][j % BM];
			X17_UNROLL for (u32 other = 0; other < gt::WAVES_K; ++other) {
				if (other != owner(j)) {
					X17_UNROLL for (int q = 0; q < 4; ++q) {
						v4i const part = *reinterpret_cast<v4i const *>(exchange + exchange_offset(j, other) + q * 1024);
						X17_UNROLL for (int i = 0; i < 4; ++i) sum[4 * q + i] = sum[4 * q + i] + part[i];
					}
				}
			}
			X17_UNROLL for (int r = 0; r < 16; ++r) x[r] = f32(sum[r]);
		}
	};
	if constexpr (gt::NATURAL) {
		static_assert(!gt::NATURAL || BM == 1, "a wavefront of the head-normalising writers has 32 tokens");
		if (wk == 0) {
			f32 x[64];
			X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
				f32 part[16];
				total_of(bn, part);
				X17_UNROLL for (int r = 0; r < 16; ++r) x[16 * bn + r] = part[r];
			}
#if X17_EPILOGUE == 3
			NaturalWriters::l2norm_row(x, c, rrms, row0, col0, N_RAW, half);
#elif X17_EPILOGUE == 5
			NaturalWriters::qnorm_row(x, c, q_norm_scales, row0, col0, half);
#elif X17_EPILOGUE == 6
			constexpr u32 Q_COLS = X17_Q_COLS;
			if (col0 < Q_COLS) {
				NaturalWriters::scale_row(x, c, row0, col0, Q_COLS, half);
			} else {
				NaturalWriters::l2norm_row(x, c_kv, rrms, row0, col0 - Q_COLS, N_RAW - Q_COLS, half);
			}
#endif
		}
	} else {
		X17_UNROLL for (int j = 0; j < BLOCKS; ++j) {
			if (owner(j) == wk) {
				f32 x[16];
				total_of(j, x);
				u32 const row = row0 + 32 * (j % BM);
				// a lane of a 64-column wavefront holds 32 consecutive columns, 16 per block
				u32 const n = col0 + (gt::WAVE_N / 2) * half + 16 * (j / BM);
#if X17_EPILOGUE == 0
				ScaleEpilogue::run(x, c, row, n, nullptr);
#elif X17_EPILOGUE == 1
				GeGluEpilogue::run(x, c, row, n, nullptr);
#elif X17_EPILOGUE == 2
				ResidualEpilogue::run(x, c, row, n, residual);
#elif X17_EPILOGUE == 4
				DequantEpilogue::run(x, c, row, n, row_scale, col_scale);
#endif
			}
		}
	}
}
