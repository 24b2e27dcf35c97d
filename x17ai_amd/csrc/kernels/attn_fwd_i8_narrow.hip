// attn_fwd_i8_narrow.hip -- the speed build of attn_fwd_i8.hip (same operands, recurrence and module ABI) with sixteen queries
// per wavefront, for launches that leave most of the chip idle.
//
// A launch of few workgroups takes as long as one wavefront's walk over its window, and a wavefront alone on its SIMD issues
// one instruction in about ten clocks: the walk is bound by its number of instructions.  Sixteen queries on the 16 x 16
// matrix instructions instead of thirty-two halve what a 32-key step spends on probabilities and output, and blocks of 64
// queries instead of 128 make twice the workgroups and walk two steps less.  1024 tokens, 8 heads of 64, window 256, row scales: 64
// workgroups and 12 steps, 128 and 10; the launch 15.5 -> 11.4 us.  Once the chip is full the 32-query kernel is ahead: it
// widens and reads a tile for twice the queries.
//
// What differs from attn_fwd_i8.hip, whose comments explain the recurrence and the arithmetic of the speed build:
//   * One workgroup = 4 wavefronts = 64 queries of one head (grid: query blocks of 64, heads, sequences).
//   * S^T = K . Q^T on v_mfma_i32_16x16x64_i8 (a lane owns query lane % 16 and four keys of each 16-key tile); O^T += V^T . P^T on
//     v_mfma_f32_16x16x16_f16, whose "B" operand those four probabilities are.
//   * The row maximum crosses four lanes instead of two when it moves.
//   * The f16 V tile's layout: eight keys of one 32-byte granule (what 32 lanes of a transposed read ask for) in eight columns.
// The bytes are the 32-query kernel's, so that a token's result does not depend on what is launched with it:
//   * Lane group g owns keys 4 j .. 4 j + 3 with j = 0, 2, 1, 3 (nt::key_of_row): the order in which the 32 x 32 x 16 instruction of
//     the other kernel takes its sixteen products.  With it the 16 x 16 x 16 instruction rounds as that one does (4 million results
//     over four distributions of operands: all the same; with keys in their own order 13 to 37 % differ).
//   * There a whole wavefront brings O and its sums down when one of its 32 queries asks for it.  So a wavefront follows its
//     twin, the sixteen queries that share such a 32 with it: their scores (the key fragments are there), their running maximum in
//     lanes, and whether that asks.  It walks the blocks of the 32.  (0.4 of the 11.4 us.)
//   * Everything else is the same operations per query; the partial sums are added in the reference's order.
//
// common.h: as for attn_fwd_i8.hip, X17_STRICT_MATH 0.

#include "common.h"
#include "x17_device.h"
#include "attn_narrow_tile.h"
#include "attn_parts.h"

using namespace x17;
namespace at = x17::attn_tile;
namespace nt = x17::attn_narrow_tile;
using namespace x17::attn_parts;

namespace {

constexpr u32 HD = X17_HEAD_DIM;
constexpr u32 Q_STRIDE = X17_Q_STRIDE;
constexpr u32 KV_STRIDE = X17_KV_STRIDE;
constexpr u32 O_STRIDE = X17_O_STRIDE;
constexpr u32 K_SLICES = (HD + 63) / 64;   // 64 bytes of head_dim per QK MFMA (head_dim 32: the upper half of Q is zero)
constexpr u32 D_TILES = HD / 16;           // 16 output dims per PV MFMA
constexpr u32 CPR = HD / 16;               // 16-byte chunks per key row
constexpr bool ROW_SCALES = at::ROW_SCALES;
constexpr bool OUT_BF16 = X17_ATTN_OUT_BF16 != 0;
static_assert(X17_STRICT_MATH == 0, "the strict build has one order of operations: attn_fwd_i8.hip");
static_assert(ROW_SCALES || !OUT_BF16, "the bf16 output needs the row-scaled build (it supplies out_scale)");
static_assert(HD == 32 || HD == 64 || HD == 128, "head_dim must be 32, 64 or 128");

constexpr f32 BASE_TEMPERATURE = ROW_SCALES ? f32(constexpr_inv_sqrt(f64(HD)))
                                            : f32(constexpr_inv_sqrt(f64(HD)) / 64.0);   // :47, :447-449

typedef short v4s __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// every lane's value and those of the three lanes that own the same query, combined (op commutative and associative)
template <class Op>
X17_DEV u32 over_groups(u32 x, Op op) {
	auto const a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
	u32 const pair = op((u32)a[0], (u32)a[1]);
	auto const b = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
	return op((u32)b[0], (u32)b[1]);
}

} // namespace

extern "C" __global__ __launch_bounds__(at::THREADS_PER_BLOCK)
__attribute__((amdgpu_waves_per_eu(2)))      // (or the accumulators live in the second half of the register file, a move away)
void kernel(
	u32 seq_len,
	i8 const *q,
	i8 const *kv,
	i8 const *sink_k,
	i8 const *sink_v,
	f32 const *attn_temperature,
	i8 *out,
	f32 *l_out,
	u32 window_size
#if X17_ATTN_ROW_SCALES
	,
	f32 const *q_scale,          // [n_heads, rows]
	f32 const *k_scale,          // [n_heads, rows]
	f32 const *v_weight,         // [n_heads, rows]
	f32 const *sink_v_weight,    // [n_heads]
	f32 const *out_scale         // [n_heads]
#endif
) {
	extern __shared__ __attribute__((aligned(1024))) u8 smem[];

	u32 const tid = threadIdx.x;
	u32 const lane = tid % 64;
	u32 const wave = __builtin_amdgcn_readfirstlane(tid / 64);
	u32 const group = lane / 16;
	u32 const qlane = lane % 16;

	// query blocks slowest, from the last one (the longest walk) to the first, as in the 32-query kernel
	u32 const head = blockIdx.y;
	size_t const row_base = (size_t)blockIdx.z * seq_len;
	size_t const all_rows = (size_t)gridDim.z * seq_len;
	u32 const q_block0 = (gridDim.x - 1 - blockIdx.x) * nt::Q_PER_BLOCK;
	u32 const q_wave0 = q_block0 + wave * nt::Q_PER_WAVE;
	u32 const qi = q_wave0 + qlane, twin_qi = qi ^ nt::Q_PER_WAVE;
	u32 const q_pair0 = q_wave0 & ~(2 * nt::Q_PER_WAVE - 1);
	u32 const own_keys = nt::key_of_row(4 * group);          // this lane's keys of a 16-key tile: own_keys .. + 3

	u32 const wr = at::rounded_window(window_size);
	u32 const vis_bound = wr - 1 < 0x7FFFFFFFu ? wr - 1 : 0x7FFFFFFFu;
	u32 const kb_begin = at::first_key_block(q_block0, wr);
	u32 const n_steps = nt::end_key_block(q_block0) - kb_begin;
	u32 const wave_kb_first = at::first_key_block(q_pair0, wr);
	u32 const wave_kb_last = q_pair0 / at::KV_PER_STEP;

	i8 const *q_head = q + row_base * Q_STRIDE + (size_t)head * HD;
	i8 const *kv_head = kv + row_base * KV_STRIDE + (size_t)head * 2 * HD;

	// ---- tile requests, by hand, as in the 32-query kernel: step s asks for K tile s + 3 (and its scales) and raw V tile s + 4,
	// past the end for the last one again, into slots nobody reads any more.  Order: V0, (K0, V1), (K1, V2), (K2, V3), ...
	bool const stager = at::is_stager(tid);
	u32 const stage_k_src = stager ? at::stage_k_offset(tid, KV_STRIDE) : 0;
	u32 const stage_v_src = stager ? at::stage_v_offset(tid, KV_STRIDE) : 0;
	u32 const lds_wave = (u32)(size_t)X17_LDS_PTR(smem) + wave * 1024;
	i8 const *const tiles = kv_head + (size_t)(kb_begin * at::KV_PER_STEP) * KV_STRIDE;
	constexpr u32 TILE_STEP_BYTES = at::KV_PER_STEP * KV_STRIDE;
	auto request_16 = [&](u32 lds_offset, u32 tile, u32 lane_offset) __attribute__((always_inline)) {
		i8 const *src = tiles + (size_t)(tile < n_steps ? tile : n_steps - 1) * TILE_STEP_BYTES;
		// (a scalar write of M0 needs one wait state before a direct-to-LDS load reads it)
		asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
		             :: "s"(lds_wave), "s"(__builtin_amdgcn_readfirstlane(lds_offset)), "v"(lane_offset), "s"(src) : "memory", "m0", "scc");
	};
	// row-scaled build, first wavefront: lanes 0..31 the scales of the tile's keys, lanes 32..63 the weights of its value rows
	[[maybe_unused]] f32 const *sc_base = nullptr;
#if X17_ATTN_ROW_SCALES
	sc_base = (lane < 32 ? k_scale : v_weight) + (size_t)head * all_rows + row_base + (size_t)kb_begin * at::KV_PER_STEP + lane % 32;
#endif
	auto request_k = [&](u32 tile, u32 slot) __attribute__((always_inline)) {
		if (ROW_SCALES && wave == 0) {
			asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, off"
			             :: "s"(lds_wave), "s"(__builtin_amdgcn_readfirstlane(nt::SCALE_RING_OFFSET + slot * at::SCALE_TILE_BYTES)),
			                "v"(sc_base + (size_t)(tile < n_steps ? tile : n_steps - 1) * at::KV_PER_STEP) : "memory", "m0", "scc");
		}
		if (CPR == 8 || stager) request_16(nt::K_RING_OFFSET + slot * at::K_TILE_BYTES, tile, stage_k_src);
	};
	auto request_v = [&](u32 tile, u32 slot) __attribute__((always_inline)) {
		if (CPR == 8 || stager) request_16(nt::RAW_V_RING_OFFSET + slot * at::RAW_V_TILE_BYTES, tile, stage_v_src);
	};
	static_assert(nt::RING == 4, "the waits below are written for rings of four");
	request_v(0, 0);
	X17_UNROLL for (u32 j = 0; j < 3; ++j) {
		request_k(j, j);
		request_v(j + 1, j + 1);
	}

	// ---- per-query setup (cuda/attn_fwd_i8.cuh:444-517), behind the requests
	bool const group_in_row = 16 * group < HD;            // (head_dim 32: the row has half the bytes of a slice)
	v4i qf[K_SLICES], twin_qf[K_SLICES];
	i32 sink_dot = 0, twin_sink_dot = 0;
	X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
		qf[s] = twin_qf[s] = v4i{0, 0, 0, 0};
		if (group_in_row) {
			qf[s] = *reinterpret_cast<v4i const *>(q_head + (size_t)qi * Q_STRIDE + 64 * s + 16 * group);
			twin_qf[s] = *reinterpret_cast<v4i const *>(q_head + (size_t)twin_qi * Q_STRIDE + 64 * s + 16 * group);
			v4i const sk = *reinterpret_cast<v4i const *>(sink_k + (size_t)head * HD + 64 * s + 16 * group);
			X17_UNROLL for (int w = 0; w < 4; ++w) {
				sink_dot = __builtin_amdgcn_sdot4(qf[s][w], sk[w], sink_dot, false);
				twin_sink_dot = __builtin_amdgcn_sdot4(twin_qf[s][w], sk[w], twin_sink_dot, false);
			}
		}
	}
	auto const add = [](u32 a, u32 b) { return a + b; };
	sink_dot = (i32)over_groups((u32)sink_dot, add);
	twin_sink_dot = (i32)over_groups((u32)twin_sink_dot, add);
	// (the lower 32 lanes compute the wavefront's temperatures, the upper ones the twin's)
	u32 const some_qi = group < 2 ? qi : twin_qi;
	u32 const visible = some_qi < wr ? some_qi : wr;
	f32 some_temperature = BASE_TEMPERATURE * strict::lg2(f32(visible + 4u));
	some_temperature = some_temperature * attn_temperature[head];
#if X17_ATTN_ROW_SCALES
	some_temperature = some_temperature * q_scale[(size_t)head * all_rows + row_base + some_qi];
#endif
	auto const both_temperatures = __builtin_amdgcn_permlane32_swap(f2u(some_temperature), f2u(some_temperature), false, false);
	f32 const temperature = u2f((u32)both_temperatures[0]);
	bool const positive_temperature = __builtin_amdgcn_readfirstlane(f2u(attn_temperature[head])) - 1u < 0x7F7FFFFFu;

	v4i s_bias;
	X17_UNROLL for (int r = 0; r < 4; ++r) s_bias[r] = ROW_SCALES ? 0 : 0x4B400000;
	f32 const abs_t = __builtin_fabsf(temperature), twin_abs_t = __builtin_fabsf(u2f((u32)both_temperatures[1]));
	f32 const sgn = positive_temperature ? 1.0f : -1.0f;
	auto const sink_extreme = [&](i32 dot) { return ROW_SCALES ? (f32(dot) * 0.125f) * sgn : (f32(dot) + DOT_BIAS) * sgn; };
	f32 ext = sink_extreme(sink_dot);
	f32 twin_ext = sink_extreme(twin_sink_dot), twin_ext_ref = twin_ext;      // (twin_ext: of this lane's keys and the sink)
	f32 mb, fine;
	set_subtrahend<ROW_SCALES>(ext, abs_t, mb, fine);
	f32 ext_ref = ext;                       // O and the sum refer to the maximum HEADROOM above this extreme's score
	f32 lift = LIFT0, sum_lift = LIFT0 * fine;
	v2h lift2 = {(_Float16)LIFT0, (_Float16)LIFT0}, neg_bias2 = {(_Float16)(-1024.0f * LIFT0), (_Float16)(-1024.0f * LIFT0)};
	f32 sum = 0.25f * PROB_SCALE * LIFT0;    // the reference's partial sum own_keys / 4
	v4f o_acc[D_TILES];                      // O^T: lane = query, register r = dim 16 dt + 4 group + r
	{
#if X17_ATTN_ROW_SCALES
		f32 const sink_weight = sink_v_weight[head];
#endif
		X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
			u32 const word = *reinterpret_cast<u32 const *>(sink_v + (size_t)head * HD + 16 * dt + 4 * group);
			X17_UNROLL for (int b = 0; b < 4; ++b) {
				f32 o = f32((i32)(i8)((word >> (8 * b)) & 0xFFu)) * PROB_SCALE;
#if X17_ATTN_ROW_SCALES
				o = o * sink_weight;
#endif
				o_acc[dt][b] = o * LIFT0;
			}
		}
	}

	// ---- lane offsets of the operand reads and of the widening
	u32 k_lane_off[2][K_SLICES], v_lane_off[D_TILES];
	X17_UNROLL for (u32 tile = 0; tile < 2; ++tile) {
		X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) k_lane_off[tile][s] = at::k_chunk_offset(16 * tile + nt::key_of_row(qlane), group_in_row ? 4 * s + group : 0);
	}
	X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) v_lane_off[dt] = nt::v_granule_offset(4 * group + (qlane >> 2), dt) + 8 * (qlane & 3);
	u32 const widen_dst = stager ? nt::widened_offset(tid) : 0;
	auto widen_v = [&](u32 slot, u32 buf) __attribute__((always_inline)) {
		if (CPR == 8 || stager) {
			v4u const raw = *reinterpret_cast<v4u const *>(smem + nt::RAW_V_RING_OFFSET + slot * at::RAW_V_TILE_BYTES + tid * 16);
			u32 w[8];
			widen16(raw, w);
			u8 *dst = smem + nt::V_TILES_OFFSET + buf * at::V_TILE_BYTES + widen_dst;
			*reinterpret_cast<v4u *>(dst) = v4u{w[0], w[1], w[2], w[3]};
			*reinterpret_cast<v4u *>(dst + 16) = v4u{w[4], w[5], w[6], w[7]};
		}
	};

	// ---- one pipeline step.  SLOT: its position in the rings as a compile-time number, or -1 for "compute it".
	auto stage = [&]<int SLOT>(u32 i) __attribute__((always_inline)) {
		u32 const slot = SLOT >= 0 ? (u32)SLOT : i % nt::RING;
		if (ROW_SCALES && wave == 0) {
			__builtin_amdgcn_s_waitcnt(0x0F76);      // vmcnt(6): three loads per step in the first wavefront
		} else {
			__builtin_amdgcn_s_waitcnt(0x0F74);      // vmcnt(4): K tile i and raw V tile i + 1 have landed
		}
		__builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0): own LDS traffic of step i - 1 is complete
		__builtin_amdgcn_s_barrier();                // ... and so is everybody else's: tiles i are visible
		request_k(i + 3, (slot + 3) % nt::RING);
		request_v(i + 4, slot);
	};
	auto widen_next = [&]<int SLOT>(u32 i) __attribute__((always_inline)) {
		u32 const slot = SLOT >= 0 ? (u32)SLOT : i % nt::RING;
		widen_v((slot + 1) % nt::RING, (slot + 1) & 1);
	};
	static_assert(MAX_LIFT == 32.0f);
	auto const larger = [](u32 a, u32 b) { return f2u(__builtin_fmaxf(u2f(a), u2f(b))); };
	auto compute = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
		u32 const slot = SLOT >= 0 ? (u32)SLOT : i % nt::RING;
		u8 const *k_tile = smem + nt::K_RING_OFFSET + slot * at::K_TILE_BYTES;
		u8 const *v_tile = smem + nt::V_TILES_OFFSET + (slot & 1) * at::V_TILE_BYTES;
		v4i s_acc[2], twin_s_acc[2];
		X17_UNROLL for (u32 tile = 0; tile < 2; ++tile) {
			s_acc[tile] = twin_s_acc[tile] = s_bias;
			X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
				v4i const kf = *reinterpret_cast<v4i const *>(k_tile + k_lane_off[tile][s]);
				s_acc[tile] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, qf[s], s_acc[tile], 0, 0, 0);
				twin_s_acc[tile] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf, twin_qf[s], twin_s_acc[tile], 0, 0, 0);
			}
		}
		widen_next.template operator()<SLOT>(i);
		X17_UNROLL for (u32 tile = 0; tile < 2; ++tile) {
			f32 y[4], twin_y[4];
			[[maybe_unused]] bool vis[4];
			[[maybe_unused]] f32 const *sc = nullptr;
			if constexpr (ROW_SCALES) {
				sc = reinterpret_cast<f32 const *>(smem + nt::SCALE_RING_OFFSET + slot * at::SCALE_TILE_BYTES) + 16 * tile + own_keys;
				v4f const ks = *reinterpret_cast<v4f const *>(sc);
				X17_UNROLL for (u32 r = 0; r < 4; ++r) {
					y[r] = f32(s_acc[tile][r]) * ks[r];
					twin_y[r] = f32(twin_s_acc[tile][r]) * ks[r];
				}
			} else {
				X17_UNROLL for (u32 r = 0; r < 4; ++r) {
					y[r] = u2f((u32)s_acc[tile][r]);
					twin_y[r] = u2f((u32)twin_s_acc[tile][r]);
				}
			}
			auto const largest = [](f32 const (&x)[4]) { return __builtin_fmaxf(__builtin_fmaxf(x[0], x[1]), __builtin_fmaxf(x[2], x[3])); };
			f32 tmax, twin_tmax;
			if constexpr (!MASKED) {
				// (positive temperature: sgn = 1)
				tmax = largest(y);
				twin_tmax = largest(twin_y);
			} else {
				u32 const first_key = (kb_begin + i) * at::KV_PER_STEP + 16 * tile + own_keys;
				f32 ym[4], twin_ym[4];
				X17_UNROLL for (u32 r = 0; r < 4; ++r) {
					vis[r] = qi - 1 - first_key - r <= vis_bound;
					y[r] = y[r] * sgn;
					ym[r] = vis[r] ? y[r] : -__builtin_inff();
					twin_ym[r] = twin_qi - 1 - first_key - r <= vis_bound ? twin_y[r] * sgn : -__builtin_inff();
				}
				tmax = largest(ym);
				twin_tmax = largest(twin_ym);
			}
			// The twin asks for a smaller scale when its lift, 2^(this), is above MAX_LIFT = 2^5
			twin_ext = __builtin_fmaxf(twin_ext, twin_tmax);
			bool const twin_asks = __any(fmaf32(twin_ext - twin_ext_ref, twin_abs_t, -HEADROOM) > 5.0f);
			if (__any(tmax > ext) || twin_asks) {
				tmax = u2f(over_groups(f2u(tmax), larger));
				ext = tmax > ext ? tmax : ext;
				set_subtrahend<ROW_SCALES>(ext, abs_t, mb, fine);
				lift = hw::ex2(fmaf32(ext - ext_ref, abs_t, -HEADROOM));      // (the difference is exact)
				if (__any(lift > MAX_LIFT) || twin_asks) {
					// O and the partial sum come down to the scale of the new maximum
					f32 const down = hw::rcp(lift) * LIFT0;
					X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
						X17_UNROLL for (int r = 0; r < 4; ++r) o_acc[dt][r] = o_acc[dt][r] * down;
					}
					sum = sum * down;
					ext_ref = ext;
					lift = LIFT0;
					twin_ext = twin_ext_ref = u2f(over_groups(f2u(twin_ext), larger));
				}
				lift2 = v2h{(_Float16)lift, (_Float16)lift};
				neg_bias2 = lift2 * v2h{(_Float16)-1024.0f, (_Float16)-1024.0f};     // exact
				sum_lift = lift * fine;
			}
			f32 p[4];
			X17_UNROLL for (u32 r = 0; r < 4; ++r) {
				f32 const arg = fmaf32(y[r], abs_t, -mb);       // lg2 of 255 * 2^(score - maximum)
				p[r] = hw::ex2(MASKED && !vis[r] ? -__builtin_inff() : arg);
			}
			sum = fmaf32((p[0] + p[1]) + (p[2] + p[3]), sum_lift, sum);
			f32 f[4];
			if constexpr (ROW_SCALES) {
				v4f const vw = *reinterpret_cast<v4f const *>(sc + 32);
				X17_UNROLL for (u32 r = 0; r < 4; ++r) f[r] = vw[r];
			} else {
				X17_UNROLL for (u32 r = 0; r < 4; ++r) f[r] = fine;
			}
			v2u pp;
			X17_UNROLL for (int w = 0; w < 2; ++w) {
				u32 const lo16 = f2u(fmaf32(p[2 * w], f[2 * w], PACK_MAGIC)), hi16 = f2u(fmaf32(p[2 * w + 1], f[2 * w + 1], PACK_MAGIC));
				u32 const pair = __builtin_amdgcn_perm(hi16, lo16, 0x05040100u);           // f16 (1024 + P) twice
				pp[w] = __builtin_bit_cast(u32, __builtin_elementwise_fma(__builtin_bit_cast(v2h, pair), lift2, neg_bias2));
			}
			v4h const pfrag = __builtin_bit_cast(v4h, pp);
			X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
				v4s const vf = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)(v_tile + v_lane_off[dt] + tile * nt::SIXTEEN_KEYS));
				o_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h, vf), pfrag, o_acc[dt], 0, 0, 0);
			}
		}
	};
	auto step = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
		stage.template operator()<SLOT>(i);
		compute.template operator()<MASKED, SLOT>(i);
	};
	auto idle_step = [&](u32 i) __attribute__((always_inline)) {
		stage.template operator()<-1>(i);
		widen_next.template operator()<-1>(i);
	};

	if (ROW_SCALES && wave == 0) {
		__builtin_amdgcn_s_waitcnt(0x0F79);   // vmcnt(9): raw V tile 0 has landed (three loads per later tile)
	} else {
		__builtin_amdgcn_s_waitcnt(0x0F76);   // vmcnt(6): raw V tile 0 has landed
	}
	widen_v(0, 0);
	u32 const first_active = wave_kb_first - kb_begin;
	u32 const diagonal = wave_kb_last - kb_begin;
	u32 const inside_kb = nt::first_inside_block(q_pair0, wr);
	u32 const inside_clamped = inside_kb < wave_kb_first ? wave_kb_first : (inside_kb > wave_kb_last ? wave_kb_last : inside_kb);
	u32 const first_full = (positive_temperature ? inside_clamped : wave_kb_last) - kb_begin;
	u32 i = 0;
	for (; i < first_active; ++i) idle_step(i);
	for (; i < first_full; ++i) step.template operator()<true, -1>(i);
	for (; i < diagonal && i % nt::RING != 0; ++i) step.template operator()<false, -1>(i);
	for (; i + nt::RING <= diagonal; i += nt::RING) {
		step.template operator()<false, 0>(i);
		step.template operator()<false, 1>(i + 1);
		step.template operator()<false, 2>(i + 2);
		step.template operator()<false, 3>(i + 3);
	}
	for (; i < diagonal; ++i) step.template operator()<false, -1>(i);
	step.template operator()<true, -1>(i);
	for (++i; i < n_steps; ++i) idle_step(i);
	__builtin_amdgcn_s_waitcnt(0x0F70);   // the last requests write LDS: they land before the workgroup gives it back

	// ---- finish (cuda/attn_fwd_i8.cuh:293-351): the sums are at the scale of the maximum HEADROOM above ext_ref's score
	f32 const m = ROW_SCALES ? fmaf32(ext_ref * sgn, temperature, HEADROOM) : fmaf32(fmaf32(ext_ref, sgn, -DOT_BIAS), temperature, HEADROOM);
	// (s0 + s1) + (s2 + s3): lane groups 0 and 2 hold s0 and s1
	auto const across = __builtin_amdgcn_permlane32_swap(f2u(sum), f2u(sum), false, false);
	f32 const half_total = u2f((u32)across[0]) + u2f((u32)across[1]);
	auto const beside = __builtin_amdgcn_permlane16_swap(f2u(half_total), f2u(half_total), false, false);
	f32 const total = u2f((u32)beside[0]) + u2f((u32)beside[1]);
	if (l_out != nullptr && group == 0) {
		l_out[(size_t)head * all_rows + row_base + qi] = sfu::lg2(total) + m;
	}
	f32 inv = sfu::rcp(total);
#if X17_ATTN_ROW_SCALES
	f32 const head_out_scale = out_scale[head];
	if constexpr (OUT_BF16) {
		u16 *o_row = reinterpret_cast<u16 *>(out) + (row_base + qi) * O_STRIDE + (size_t)head * HD;
		X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
			f32 b[4];
			X17_UNROLL for (int e = 0; e < 4; ++e) b[e] = (o_acc[dt][e] * inv) * head_out_scale;
			*reinterpret_cast<v2u *>(o_row + 16 * dt + 4 * group) = v2u{pack2_bf16_rne(b[0], b[1]), pack2_bf16_rne(b[2], b[3])};
		}
		return;
	}
	X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
		X17_UNROLL for (int r = 0; r < 4; ++r) o_acc[dt][r] = (o_acc[dt][r] * inv) * head_out_scale;
	}
	inv = 1.0f;
#endif
	i8 *o_row = out + (row_base + qi) * O_STRIDE + (size_t)head * HD;
	X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
		*reinterpret_cast<u32 *>(o_row + 16 * dt + 4 * group) = scaled_codes(o_acc[dt][0], o_acc[dt][1], o_acc[dt][2], o_acc[dt][3], inv);
	}
}
