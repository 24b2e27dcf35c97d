// attn_d_q_i8.hip -- backward of the int8 sliding-window attention with respect to q, for gfx950.
//
// The reference's backward kernels (attn_d_q.cuh:1-410) belong to its bf16 generation; its int8 / e4m3 generation has
// no backward yet.  This kernel keeps the structure of attn_d_q.cuh -- probabilities recomputed from the forward's
// log-sum-exp L, D = rowsum(dO * O) written out for a later dK/dV kernel, dS = P * (dP - D), dQ = dS . K -- on the
// forward semantics of attn_fwd_i8.hip (cuda/attn_fwd_i8.cuh:368-619): FixedI8 q / k / v codes (real = code / 8), a
// sink key AND value per head, scores in base 2 with the scalable-softmax temperature, causal sliding window.
// Per head and query i (position inside its sequence), with t_i = hd^-1/2 * lg2(min(W', i) + 4) * head_temp[h]:
//   P_ij  = 2^(t_i (q_i . k_j) - (L_i - lg2 255))     for the keys j in [max(0, i - W'), i - 1] and the sink
//   D_i   = dO_i . o_i,  o_i = out_code_i / 8         (the forward output as stored)
//   dS_ij = ln 2 * P_ij * (dO_i . v_j - D_i)
//   dq_i  = t_i * sum_j dS_ij k_j                      (gradient with respect to the REAL q; bf16)
// The forward's 8-bit rounding of P and the quantisation of q are treated as the identity.
//
// Design, MI355X-first (the forward kernel's blocking, so that its index arithmetic and tile layouts carry over):
//   * One workgroup = 4 wavefronts = 128 queries of one head; a wavefront owns 32 queries; 32 keys per step.
//   * S^T = K . Q^T on v_mfma_i32_32x32x32_i8 exactly as in the forward (keys are the "A" operand: a lane owns one
//     query and 8 keys of each 16-key tile).
//   * dP^T = V . dO^T and dQ^T += K^T . dS^T run on v_mfma_f32_32x32x16_f16.  K and V arrive as int8 (global -> LDS
//     directly, three steps ahead) and are widened to f16 once per workgroup, LDS -> LDS, one step ahead, by the
//     threads that fetched them: K into the granule layout that ds_read_b64_tr_b16 reads transposed (the "A" operand
//     K^T needs eight keys of one dim per lane), V into swizzled rows (the "A" operand V needs eight dims of one key).
//   * dO is bf16 in memory.  Everything is linear in dO_i, so each query row is scaled by a power of two that brings
//     its largest element into [1, 2) before it is rounded to f16 (more significand bits than bf16 for every element
//     that matters, and no underflow however small the gradients are); dq_i and D_i are scaled back at the end.
//     A lane keeps the f16 fragments of its whole row in registers: they are the "B" operand of dP^T directly.
//   * dS stays in registers: packed to f16 it is the "B" operand of the dQ^T product, as P is in the forward.
//
// common.h (generated per kernel) provides X17_N_HEADS, X17_HEAD_DIM, X17_Q_STRIDE, X17_KV_STRIDE, X17_O_STRIDE,
// X17_STRICT_MATH.  gridDim = (query blocks, head groups, sequences), as for the forward.

#include "common.h"
#include "x17_device.h"
#include "attn_bwd_tile.h"
#include "attn_parts.h"

using namespace x17;
namespace at = x17::attn_tile;
namespace bt = x17::attn_bwd_tile;
using namespace x17::attn_parts;

namespace {

constexpr u32 HD = X17_HEAD_DIM;
constexpr u32 N_HEADS = X17_N_HEADS;
constexpr u32 Q_STRIDE = X17_Q_STRIDE;
constexpr u32 KV_STRIDE = X17_KV_STRIDE;
constexpr u32 O_STRIDE = X17_O_STRIDE;
constexpr u32 HPK = at::HEADS_PER_KERNEL;
constexpr u32 K_SLICES = HD / 32;      // 32 bytes of head_dim per QK MFMA
constexpr u32 D_SLICES = HD / 16;      // 16 dims per dP MFMA
constexpr u32 D_BLOCKS = HD / 32;      // 32 output dims per dQ MFMA
constexpr u32 CPR = at::CHUNKS_PER_ROW;

static_assert(HD == 32 || HD == 64 || HD == 128, "head_dim must be 32, 64 or 128");
static_assert(N_HEADS % HPK == 0, "n_heads must be divisible by heads_per_kernel");

constexpr f32 BASE_TEMPERATURE = f32(constexpr_inv_sqrt(f64(HD)) / 64.0);  // for dots of codes (8 q . 8 k)
// dq = t_real * ln 2 * sum_j w_j k_j with t_real = 64 * temperature (the temperature below is for dots of codes)
// and k = code / 8: 64 * ln 2 / 8
constexpr f32 EIGHT_LN2 = 5.5451774444795625f;

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));

X17_DEV f32 i8_of(u32 word, int b) { return f32((i32)(i8)((word >> (8 * b)) & 0xFFu)); }

} // namespace

extern "C" __global__ __launch_bounds__(bt::THREADS_PER_BLOCK)
__attribute__((amdgpu_waves_per_eu(bt::WAVES_PER_SIMD, bt::WAVES_PER_SIMD)))
void kernel(
	u32 seq_len,
	i8 const *q,
	i8 const *kv,
	i8 const *sink_k,
	i8 const *sink_v,
	f32 const *attn_temperature,
	i8 const *out,               // the forward's output codes [rows, O_STRIDE]
	u16 const *d_out,            // bf16 [rows, O_STRIDE]: gradient with respect to the real output
	u16 *d_q,                    // bf16 [rows, Q_STRIDE]: gradient with respect to the real q
	f32 const *l,                // the forward's log-sum-exp [H, rows]
	f32 *d_rows,                 // D [H, rows] (may be null)
	u32 window_size
) {
	extern __shared__ __attribute__((aligned(1024))) u8 smem[];

	u32 const tid = threadIdx.x;
	u32 const lane = tid % 64;
	u32 const wave = __builtin_amdgcn_readfirstlane(tid / 64);
	u32 const half = lane / 32;
	u32 const qlane = lane % 32;

	// the forward's workgroup order: the query block is the slowest index and runs from the last block to the first
	u32 const pairs = gridDim.y * gridDim.z;
	u32 const lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
	u32 const pair = lin % pairs;
	u32 const q_block_index = gridDim.x - 1 - lin / pairs;
	// heads of this workgroup, one behind the other: the grid says how many groups they were cut into (one group per head
	// by this library's launchers, groups of 128 / head_dim heads by src/device/cuda/attn.rs:60-66)
	u32 const heads_here = HPK == 1 ? 1 : N_HEADS / gridDim.y;
	u32 const head_group = pair % gridDim.y;
	u32 const seq = pair / gridDim.y;
	size_t const row_base = (size_t)seq * seq_len;
	size_t const all_rows = (size_t)gridDim.z * seq_len;
	u32 const q_block0 = at::block_first_query(q_block_index, seq_len);
	u32 const q_wave0 = q_block0 + wave * at::Q_PER_WAVE;
	u32 const qi = q_wave0 + qlane;
	u32 const wr = at::rounded_window(window_size);
	u32 const vis_bound = wr - 1 < 0x7FFFFFFFu ? wr - 1 : 0x7FFFFFFFu;
	u32 const kb_begin = at::first_key_block(q_block0, wr);
	u32 const kb_end = at::end_key_block(q_block0);
	u32 const wave_kb_first = at::first_key_block(q_wave0, wr);
	u32 const wave_kb_last = q_wave0 / at::KV_PER_STEP;
	u32 const n_steps = kb_end - kb_begin;

	for (u32 hh = 0; hh < heads_here; ++hh) {
		u32 const head = head_group * heads_here + hh;
		i8 const *q_head = q + row_base * Q_STRIDE + (size_t)head * HD;
		i8 const *kv_head = kv + row_base * KV_STRIDE + (size_t)head * 2 * HD;

		// ---- staging: thread t fetches 16-byte chunk t of the K tile and of the V tile and later widens them
		bool const stager = at::is_stager(tid);
		u32 stage_k_src = 0, stage_v_src = 0, k_f16_dst = 0, v_f16_dst0 = 0, v_f16_dst1 = 0;
		if (stager) {
			stage_k_src = at::stage_k_offset(tid, KV_STRIDE);
			stage_v_src = at::stage_v_offset(tid, KV_STRIDE);
			k_f16_dst = bt::k_widened_offset(tid);
			v_f16_dst0 = bt::v_widened_offset(tid, 0);
			v_f16_dst1 = bt::v_widened_offset(tid, 1);
		}
		auto widen = [&](u32 slot, u32 buf) __attribute__((always_inline)) {
			if (CPR == 8 || stager) {          // (head_dim 128: every thread stages)
				u32 w[8];
				widen16<false>(*reinterpret_cast<v4u const *>(smem + bt::RAW_K_RING_OFFSET + slot * bt::RAW_TILE_BYTES + tid * 16), w);
				u8 *kd = smem + bt::K_F16_OFFSET + buf * bt::F16_TILE_BYTES + k_f16_dst;
				*reinterpret_cast<v4u *>(kd) = v4u{w[0], w[1], w[2], w[3]};
				*reinterpret_cast<v4u *>(kd + 16) = v4u{w[4], w[5], w[6], w[7]};
				widen16<true>(*reinterpret_cast<v4u const *>(smem + bt::RAW_V_RING_OFFSET + slot * bt::RAW_TILE_BYTES + tid * 16), w);
				u8 *vd = smem + bt::V_F16_OFFSET + buf * bt::F16_TILE_BYTES;
				*reinterpret_cast<v4u *>(vd + v_f16_dst0) = v4u{w[0], w[1], w[2], w[3]};
				*reinterpret_cast<v4u *>(vd + v_f16_dst1) = v4u{w[4], w[5], w[6], w[7]};
			}
		};
		constexpr u32 TILE_STEP_BYTES = at::KV_PER_STEP * KV_STRIDE;
		u32 const lds_wave = (u32)(size_t)X17_LDS_PTR(smem) + wave * 1024;
		i8 const *src = kv_head + (size_t)(kb_begin * at::KV_PER_STEP) * KV_STRIDE;      // the tile the next request takes
		auto request = [&](u32 slot) __attribute__((always_inline)) {
			if (CPR == 8 || stager) {
				// (a scalar write of M0 needs one wait state before a direct-to-LDS load reads it)
				// (the slot is the same in every lane; reading its offset from the first one tells the compiler so)
				u32 const slot_bytes = __builtin_amdgcn_readfirstlane(slot * bt::RAW_TILE_BYTES);
				asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
				             :: "s"(lds_wave), "s"(bt::RAW_K_RING_OFFSET + slot_bytes), "v"(stage_k_src), "s"(src) : "memory", "m0", "scc");
				asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
				             :: "s"(lds_wave), "s"(bt::RAW_V_RING_OFFSET + slot_bytes), "v"(stage_v_src), "s"(src) : "memory", "m0", "scc");
			}
		};
		// the first tiles are requested ahead of the per-query set-up and land behind it
		__syncthreads();                      // previous head's tiles are no longer read
		// (every workgroup walks at least four tiles: 0 .. 3 exist)
		X17_UNROLL for (u32 j = 0; j < bt::PREFETCH; ++j) {
			request(j);
			src += TILE_STEP_BYTES;
		}

		// ---- per-query set-up
		v4i qf[K_SLICES];
		X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
			qf[s] = *reinterpret_cast<v4i const *>(q_head + (size_t)qi * Q_STRIDE + 32 * s + 16 * half);
		}
		u32 const visible = qi < wr ? qi : wr;
		f32 temperature = BASE_TEMPERATURE * strict::lg2(f32(visible + 4u));
		temperature = temperature * attn_temperature[head];
		f32 const l_hat = l[(size_t)head * all_rows + row_base + qi] - LOG2_PROB_SCALE;

		// dO row: this lane's half of every 16-dim slice (dims 16 sl + 8 half .. + 7), bf16 -> f32
		u16 const *do_row = d_out + (row_base + qi) * O_STRIDE + (size_t)head * HD;
		i8 const *o_row = out + (row_base + qi) * O_STRIDE + (size_t)head * HD;
		f32 dof[D_SLICES][8];
		f32 row_max = 0.0f;
		X17_UNROLL for (u32 sl = 0; sl < D_SLICES; ++sl) {
			v4u const raw = *reinterpret_cast<v4u const *>(do_row + 16 * sl + 8 * half);
			X17_UNROLL for (int w = 0; w < 4; ++w) {
				dof[sl][2 * w] = u2f(raw[w] << 16);
				dof[sl][2 * w + 1] = u2f(raw[w] & 0xFFFF0000u);
				row_max = __builtin_fmaxf(row_max, __builtin_fmaxf(__builtin_fabsf(dof[sl][2 * w]), __builtin_fabsf(dof[sl][2 * w + 1])));
			}
		}
		row_max = __builtin_fmaxf(row_max, partner_f32(row_max, half));
		// power of two that brings the row's largest magnitude into [1, 2) (1 for an all-zero, infinite or NaN row)
		u32 const max_exp = (f2u(row_max) >> 23) & 0xFFu;
		bool const scalable = max_exp != 0 && max_exp != 0xFFu;
		f32 const scale = scalable ? u2f((254u - max_exp) << 23) : 1.0f;
		f32 const inv_scale = scalable ? u2f(max_exp << 23) : 1.0f;
		v8h dofrag[D_SLICES];                 // "B" operand of dP^T: lane = query, slots = dims 16 sl + 8 half + 0..7
		f32 d_part = 0.0f, dps_part = 0.0f;   // partial sums of D' = dO' . o and of dO' . sink_v (this lane's dims)
		X17_UNROLL for (u32 sl = 0; sl < D_SLICES; ++sl) {
			v2u const oc = *reinterpret_cast<v2u const *>(o_row + 16 * sl + 8 * half);
			v2u const sv = *reinterpret_cast<v2u const *>(sink_v + (size_t)head * HD + 16 * sl + 8 * half);
			X17_UNROLL for (int e = 0; e < 8; ++e) {
				_Float16 const hval = (_Float16)(dof[sl][e] * scale);       // round to nearest even
				dofrag[sl][e] = hval;
				f32 const back = (f32)hval;
				d_part = fmaf32(back, i8_of(oc[e / 4], e % 4), d_part);
				dps_part = fmaf32(back, i8_of(sv[e / 4], e % 4), dps_part);
			}
		}
		f32 const d_other = partner_f32(d_part, half), dps_other = partner_f32(dps_part, half);
		// (both in code units of o and v: 8 times the real dot products; the lower half's partial sum first)
		f32 const d8 = half == 0 ? d_part + d_other : d_other + d_part;
		f32 const dps8 = half == 0 ? dps_part + dps_other : dps_other + dps_part;

		// the sink: a key and a value every query sees
		i32 sink_dot = 0;
		X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
			v4i sk = *reinterpret_cast<v4i const *>(sink_k + (size_t)head * HD + 32 * s + 16 * half);
			X17_UNROLL for (int w = 0; w < 4; ++w) sink_dot = __builtin_amdgcn_sdot4(qf[s][w], sk[w], sink_dot, false);
		}
		sink_dot += partner_i32(sink_dot, half);
		f32 const p_sink = sfu::ex2(f32(sink_dot) * temperature - l_hat);
		// lane offsets of the operand fragments (the forward's transposed-read addressing for K^T)
		u32 kt_lane_off[D_BLOCKS];
		[[maybe_unused]] u32 kt_lane_off8[D_BLOCKS];
		{
			u32 const t = lane % 16, dh = (lane / 16) % 2;
			X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
				kt_lane_off[db] = bt::granule_offset(4 * half + (t >> 2), 2 * db + dh) + 8 * (t & 3);
				kt_lane_off8[db] = bt::granule_offset(8 + 4 * half + (t >> 2), 2 * db + dh) + 8 * (t & 3);
			}
		}

		// ---- the key loop, built like the forward's (attn_fwd_i8.hip): a wave's steps fall into runs -- nothing to do, the
		// window's edge, fully visible, the diagonal, nothing to do -- each its own loop; every step requests a tile by
		// hand (past the end the last one again, into a slot nobody reads any more), so the waits are constants; the long
		// run is unrolled over the four slots of the rings, so that every LDS address is a register plus an immediate.
		// A score costs a conversion, a multiplication, a subtraction, an exponential, dP - D, the product and half a conversion to
		// f16, each rounded by itself.  (One fused multiply-add on accumulators that start at a bias, and dP accumulators that
		// start at -D, are 57 instructions fewer per step and 5 % of the launch, but round otherwise: a gradient's bytes
		// then depend on the version.  They also make NaN of a row whose L is +inf, which weighs nothing.)  V is widened
		// to its real value, code / 8, so that D needs no factor.
		// Bound by the rate at which a wavefront issues (one instruction in about ten clocks, two wavefronts per SIMD): a fully
		// visible step is 237 instructions; it was 357, around requests that were drained in the step that made them.  16 heads
		// of 128, 4 x 8192 tokens, window 512: 333 -> 284 us, of which 160 are set-up, output and the first steps (window 32).
		f32 const w_sink = p_sink * ((dps8 - d8) * 0.125f);
		v16f dq_acc[D_BLOCKS];               // dQ^T: lane = query, register r = dim 32 db + 8 (r / 4) + 4 half + r % 4
		X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
			X17_UNROLL for (int r4 = 0; r4 < 4; ++r4) {
				u32 const word = *reinterpret_cast<u32 const *>(sink_k + (size_t)head * HD + 32 * db + 8 * r4 + 4 * half);
				X17_UNROLL for (int b = 0; b < 4; ++b) dq_acc[db][4 * r4 + b] = w_sink * i8_of(word, b);
			}
		}
		f32 const d1 = d8 * 0.125f;           // D in the units of dO . v (real v)
		u32 k_lane_off[K_SLICES], v_lane_off[D_SLICES];
		X17_UNROLL for (u32 sl = 0; sl < K_SLICES; ++sl) k_lane_off[sl] = at::k_chunk_offset(qlane, 2 * sl + half);
		X17_UNROLL for (u32 sl = 0; sl < D_SLICES; ++sl) v_lane_off[sl] = bt::vrow_offset(qlane, 2 * sl + half);

		// SLOT: the step's position in the rings (s % RING) as a compile-time number, or -1 for "compute it"; SLOT >= 0 also
		// says that tile s + 4 exists (the caller's loop bound)
		auto stage = [&]<int SLOT>(u32 s) __attribute__((always_inline)) {
			__builtin_amdgcn_s_waitcnt(0x0F72);          // vmcnt(2): tile s + 1 has landed (this thread's chunks), s + 2 may be in flight
			__builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0): own LDS traffic of step s - 1 is complete
			__builtin_amdgcn_s_barrier();                // ... and so is everybody else's: tiles s are visible
			// step s requests tile min(s + 3, last) into the slot of tile s - 1, which nobody reads any more
			request(SLOT >= 0 ? (SLOT + 3) % bt::RING : (s + 3) % bt::RING);
			if (SLOT >= 0 || at::further_tile_exists(s, n_steps)) {
				src += TILE_STEP_BYTES;
			}
		};
		static_assert(bt::PREFETCH == 3 && bt::RING == 4 && at::PREFETCH == 3, "the waits, the requests and the unrolled run are written for rings of four");
		auto compute = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
			u32 const slot = SLOT >= 0 ? (u32)SLOT : i % bt::RING;
			u32 const buf = SLOT >= 0 ? (u32)SLOT & 1u : i & 1u;
			u8 const *k_raw = smem + bt::RAW_K_RING_OFFSET + slot * bt::RAW_TILE_BYTES;
			u8 const *k_f16 = smem + bt::K_F16_OFFSET + buf * bt::F16_TILE_BYTES;
			u8 const *v_f16 = smem + bt::V_F16_OFFSET + buf * bt::F16_TILE_BYTES;
			// S^T block: rows = 32 keys, columns = this wave's 32 queries; dP'^T for the same keys
			v16i s_acc = {0};
			X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
				v4i const kf = *reinterpret_cast<v4i const *>(k_raw + k_lane_off[s]);
				s_acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[s], s_acc, 0, 0, 0);
			}
			v16f dp_acc = {0};
			X17_UNROLL for (u32 sl = 0; sl < D_SLICES; ++sl) {
				v8h const vf = *reinterpret_cast<v8h const *>(v_f16 + v_lane_off[sl]);
				dp_acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, dofrag[sl], dp_acc, 0, 0, 0);
			}
			widen((slot + 1) % bt::RING, buf ^ 1u);       // (behind the matrix instructions, whose results are not ready yet)
			X17_UNROLL for (u32 tile = 0; tile < 2; ++tile) {
				// this lane's keys of the tile: 4 half + {0..3} and 8 + 4 half + {0..3}
				f32 w[8];
				[[maybe_unused]] u32 const first = qi - 1 - ((kb_begin + i) * at::KV_PER_STEP + 16 * tile + 4 * half);
				X17_UNROLL for (u32 r = 0; r < 8; ++r) {
					f32 const score = f32(s_acc[8 * tile + r]) * temperature;
					f32 p = sfu::ex2(score - l_hat);
					if constexpr (MASKED) {
						// key j is visible iff the distance qi - 1 - j, as an unsigned number, is at most W' - 1
						u32 const distance = first - (8 * (r / 4) + (r % 4));
						p = distance <= vis_bound ? p : 0.0f;
					}
					w[r] = p * (dp_acc[8 * tile + r] - d1);
				}
				v8h wfrag;
				X17_UNROLL for (u32 r = 0; r < 8; ++r) wfrag[r] = (_Float16)w[r];
				X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
					u8 const *p0 = k_f16 + kt_lane_off[db] + tile * (16 * CPR * 32);
					u8 const *p1 = CPR >= 4 ? p0 + 8 * CPR * 32 : k_f16 + kt_lane_off8[db] + tile * (16 * CPR * 32);
					v4s const lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)p0);
					v4s const hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)p1);
					v8s const both = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
					dq_acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, both), wfrag, dq_acc[db], 0, 0, 0);
				}
			}
		};
		auto step = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
			stage.template operator()<SLOT>(i);
			compute.template operator()<MASKED, SLOT>(i);
		};
		auto idle_step = [&](u32 i) __attribute__((always_inline)) {
			stage.template operator()<-1>(i);
			widen((i + 1) % bt::RING, (i + 1) & 1);
		};
		u32 const first_active = wave_kb_first - kb_begin;
		u32 const diagonal = wave_kb_last - kb_begin;
		// first block that lies inside the window of all 32 queries: q_wave0 + 31 - 32 kb <= wr
		u32 const inside_kb = q_wave0 + 31 > wr ? (q_wave0 + 62 - wr) / 32 : 0;
		u32 const inside_clamped = inside_kb < wave_kb_first ? wave_kb_first : (inside_kb > wave_kb_last ? wave_kb_last : inside_kb);
		u32 const first_full = inside_clamped - kb_begin;

		__builtin_amdgcn_s_waitcnt(0x0F74);   // vmcnt(4): tile 0 has landed
		widen(0, 0);
		u32 i = 0;
		for (; i < first_active; ++i) idle_step(i);
		for (; i < first_full; ++i) step.template operator()<true, -1>(i);
		for (; i < diagonal && i % bt::RING != 0; ++i) step.template operator()<false, -1>(i);
		for (; i + bt::RING <= diagonal && i + 2 * bt::RING <= n_steps; i += bt::RING) {
			step.template operator()<false, 0>(i);
			step.template operator()<false, 1>(i + 1);
			step.template operator()<false, 2>(i + 2);
			step.template operator()<false, 3>(i + 3);
		}
		for (; i < diagonal; ++i) step.template operator()<false, -1>(i);
		step.template operator()<true, -1>(i);
		for (++i; i < n_steps; ++i) idle_step(i);
		__builtin_amdgcn_s_waitcnt(0x0F70);   // the last requests write LDS: they land before the tiles are reused

		// ---- output: dq = 8 ln 2 * temperature * dq_acc / scale, D = d8 / (8 scale)
		f32 const out_scale = (temperature * EIGHT_LN2) * inv_scale;
		u16 *dq_row = d_q + (row_base + qi) * Q_STRIDE + (size_t)head * HD;
		X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
			X17_UNROLL for (int g = 0; g < 4; ++g) {
				f32 b[4];
				X17_UNROLL for (int e = 0; e < 4; ++e) b[e] = dq_acc[db][4 * g + e] * out_scale;
				v2u const pair = {pack2_bf16_rne(b[0], b[1]), pack2_bf16_rne(b[2], b[3])};
				*reinterpret_cast<v2u *>(dq_row + 32 * db + 8 * g + 4 * half) = pair;
			}
		}
		if (d_rows != nullptr && half == 0) {
			d_rows[(size_t)head * all_rows + row_base + qi] = (d8 * 0.125f) * inv_scale;
		}
	}
}
