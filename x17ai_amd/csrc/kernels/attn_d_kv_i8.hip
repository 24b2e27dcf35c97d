// attn_d_kv_i8.hip -- backward of the int8 sliding-window attention with respect to k and v, for gfx950.
//
// The reference's backward kernels (attn_d_kv.cuh:1-431) belong to its bf16 generation; its int8 / e4m3 generation has
// no backward yet.  This kernel keeps the structure of attn_d_kv.cuh:200-400 -- a workgroup owns a block of keys and
// walks the query tiles that see it; per tile S = Q . K^T, P from the forward's log-sum-exp L, dP = dO . V^T,
// dV += P^T . dO, dS = P * (dP - D) with D from the dQ pass, dK += dS^T . Q; P and dS are rounded to bf16 for their
// products as the reference does -- on the forward semantics of attn_fwd_i8.hip (cuda/attn_fwd_i8.cuh:368-619): FixedI8
// q / k / v codes (real = code / 8), scores in base 2 with the scalable-softmax temperature, causal sliding window.
// Per head, key j and the queries i that see it (j < i <= j + W'), t_i = hd^-1/2 * lg2(min(W', i) + 4) * head_temp[h]:
//   P_ij  = 2^(t_i (q_i . k_j) - (L_i - lg2 255))
//   dv_j  = sum_i P_ij dO_i
//   dS_ij = ln 2 * P_ij * (dO_i . v_j - D_i)
//   dk_j  = sum_i t_i dS_ij q_i                        (gradients with respect to the REAL k and v; bf16)
// Like attn_d_kv.cuh, no gradient is formed for the sink or the temperatures; the sink enters through L and D only.
//
// Design, MI355X-first:
//   * One workgroup = 4 wavefronts = 64 keys of one head; a wavefront owns 16 keys and works on the 16 x 16 matrix
//     instructions: its int8 K fragments, its V fragments widened to bf16 and the 2 x 32 accumulators of dK^T and dV^T
//     (dims x keys) stay in registers, and three workgroups share a compute unit.
//   * Orientation: S and dP are (queries x keys), so a lane owns ONE key and 8 queries of the 32-query tile.  Their
//     MFMA results are then, packed to bf16, directly the "B" operand (contraction over the tile's 32 queries) of
//     dV^T += dO^T . P and dK^T += Q^T . dS; no lane exchange, no LDS round trip.
//   * S runs on v_mfma_i32_16x16x64_i8 from the raw int8 Q tile; dP, dV^T, dK^T on v_mfma_f32_16x16x32_bf16 (dO is bf16
//     in memory and is used as it is; int8 codes are exact in bf16): 28 matrix instructions per step for head_dim 128.
//   * Tiles of 32 queries arrive global -> LDS directly, by hand-written requests with constant waits: the raw Q rows and the
//     tile's L and D values three steps ahead, the dO rows one step ahead -- one copy that is read by rows ("A" of dP: eight
//     dims of one query) as well as by ds_read_b64_tr_b16 ("A" of dV^T: eight queries of one dim); the layout is chosen by which source
//     chunk a lane requests.  One step ahead the workgroup widens the Q tile to bf16 into the same layout ("A" of dK^T)
//     and one wavefront writes the tile's per-query constants (temperature, L - lg2 255, D).
//
// common.h (generated per kernel) provides X17_N_HEADS, X17_HEAD_DIM, X17_Q_STRIDE, X17_KV_STRIDE, X17_O_STRIDE,
// X17_STRICT_MATH.  gridDim = (runs of key blocks, head groups, sequences).

#include "common.h"
#include "x17_device.h"
#include "attn_bwd_kv_tile.h"

using namespace x17;
namespace at = x17::attn_tile;
namespace kt = x17::attn_bwd_kv_tile;

namespace {

constexpr u32 HD = X17_HEAD_DIM;
constexpr u32 N_HEADS = X17_N_HEADS;
constexpr u32 Q_STRIDE = X17_Q_STRIDE;
constexpr u32 KV_STRIDE = X17_KV_STRIDE;
constexpr u32 O_STRIDE = X17_O_STRIDE;
constexpr u32 HPK = at::HEADS_PER_KERNEL;
constexpr u32 K_SLICES = (HD + 63) / 64;   // 64 bytes of head_dim per QK MFMA (head_dim 32: the upper half is zero)
constexpr u32 D_SLICES = HD / 32;          // 32 dims per dP MFMA
constexpr u32 D_TILES = HD / 16;           // 16 output dims per dK^T / dV^T MFMA
constexpr u32 Q_TILES = kt::Q_PER_STEP / 16;   // S and dP: two 16-query tiles per step
constexpr u32 CPR = kt::CPR;

static_assert(HD == 32 || HD == 64 || HD == 128, "head_dim must be 32, 64 or 128");
static_assert(N_HEADS % HPK == 0, "n_heads must be divisible by heads_per_kernel");
// Registers next to the 64 accumulators: D is read when P is there, and the strict build, whose exponential needs more of them,
// multiplies dP then as well (in the speed build that costs 0.5 %)
constexpr bool DP_LATE = X17_STRICT_MATH && HD == 128;

static_assert(kt::RING == 4, "the pipeline below is written for a ring of four and pairs of tiles");

constexpr f32 LOG2_PROB_SCALE = 7.9943534368588578f;                       // lg2(255): the forward's L carries it
constexpr f32 BASE_TEMPERATURE = f32(constexpr_inv_sqrt(f64(HD)) / 64.0);  // for dots of codes (8 q . 8 k)
// dk = t_real * ln 2 * sum_i w_i q_i with t_real = 64 * temperature (the temperature below is for dots of codes)
// and q = code / 8: 64 * ln 2 / 8
constexpr f32 EIGHT_LN2 = 5.5451774444795625f;

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));

// four int8 codes, times a power of two, as four bf16, exact
X17_DEV v2u widen4(u32 word, f32 factor = 1.0f) {
	f32 f[4];
	X17_UNROLL for (int b = 0; b < 4; ++b) f[b] = f32((i32)(i8)((word >> (8 * b)) & 0xFFu)) * factor;
	return v2u{pack2_bf16_rne(f[0], f[1]), pack2_bf16_rne(f[2], f[3])};
}

X17_DEV v8bf transposed_fragment(u8 const *p0, u8 const *p1) {
	v4s const lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)p0);
	v4s const hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)p1);
	v8s const both = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
	return __builtin_bit_cast(v8bf, both);
}

} // namespace

extern "C" __global__ __launch_bounds__(kt::THREADS_PER_BLOCK)
__attribute__((amdgpu_waves_per_eu(kt::WAVES_PER_SIMD, kt::WAVES_PER_SIMD)))
void kernel(
	u32 seq_len,
	i8 const *q,
	i8 const *kv,
	f32 const *attn_temperature,
	u16 const *d_out,            // bf16 [rows, O_STRIDE]: gradient with respect to the real output
	f32 const *l,                // the forward's log-sum-exp [H, rows]
	f32 const *d_rows,           // D [H, rows] of the dQ pass
	u16 *d_kv,                   // bf16 [rows, KV_STRIDE]: per head dK then dV, the layout of kv
	u32 window_size
) {
	extern __shared__ __attribute__((aligned(1024))) u8 smem[];

	u32 const wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
	u32 const lds_wave = (u32)(size_t)X17_LDS_PTR(smem) + wave * 1024;

	u32 const pairs = gridDim.y * gridDim.z;
	u32 const lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
	u32 const pair = lin % pairs;
	u32 const run = lin / pairs;
	// key blocks and heads of this workgroup, one behind the other: the grid says how many runs and groups they were cut into (a
	// block and a head each by this library's launchers, groups of 128 / head_dim heads by src/device/cuda/attn.rs:60-66)
	u32 const blocks_here = kt::blocks_per_run(seq_len, gridDim.x);
	u32 const heads_here = HPK == 1 ? 1 : N_HEADS / gridDim.y;
	u32 const head_group = pair % gridDim.y;
	u32 const seq = pair / gridDim.y;
	size_t const row_base = (size_t)seq * seq_len;
	size_t const all_rows = (size_t)gridDim.z * seq_len;
	u32 const wr = at::rounded_window(window_size);
	u32 const vis_bound = wr - 1 < 0x7FFFFFFFu ? wr - 1 : 0x7FFFFFFFu;

	for (u32 item = 0; item < heads_here * blocks_here; ++item) {
		u32 const head = head_group * heads_here + item % heads_here;
		u32 const key_block0 = kt::block_first_key(run * blocks_here + item / heads_here);
		if (key_block0 >= seq_len) {
			break;
		}
		// (opaque: what an item derives from it is derived anew for the next one, not kept in registers from here on)
		u32 tid = threadIdx.x;
		asm volatile("" : "+v"(tid));
		u32 const lane = tid % 64;
		u32 const group = lane / 16;          // the lane's k-group in the operands, its row group in the results
		u32 const klane = lane % 16;          // its key in S, dP and the accumulators; its row or dim in the "A" operands
		u32 const key_wave0 = key_block0 + wave * kt::KEYS_PER_WAVE;
		u32 const key = key_wave0 + klane;
		u32 const tile_begin = kt::first_query_tile(key_block0);
		u32 const tile_end = kt::end_query_tile(key_block0 + kt::KEYS_PER_BLOCK - 1, wr, seq_len);
		u32 const wave_tile_first = kt::first_query_tile(key_wave0);
		u32 const wave_tile_last = kt::end_query_tile(key_wave0 + kt::KEYS_PER_WAVE - 1, wr, seq_len) - 1;
		u32 const n_steps = tile_end - tile_begin;
		// ---- lane constants of the requests and of the operand reads
		bool const q_stager = kt::is_q_stager(tid), wide_stager = kt::is_wide_stager(tid);
		u32 const q_src = kt::q_raw_source(tid, Q_STRIDE);
		u32 const do_src = kt::rows_source(tid, O_STRIDE * 2);
		u32 const q_wide_dst = kt::widened_offset(tid);
		// "A" of S: query 16 qt + klane, the 16 bytes 64 s + 16 group of its row (none for head_dim 32's upper half)
		bool const k_group_in_row = 16 * group < HD;
		u32 q_read_off[Q_TILES][K_SLICES];
		X17_UNROLL for (u32 qt = 0; qt < Q_TILES; ++qt) {
			X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
				// (head_dim 128: sixteen queries further is a constant stride)
				q_read_off[qt][s] = HD == 128 && qt != 0 ? q_read_off[0][s] + 16 * HD : kt::q_raw_offset(16 * qt + klane, k_group_in_row ? 4 * s + group : 0);
			}
		}
		// "A" of dP: query 16 qt + klane, dims 32 sl + 8 group + 0..7.  Sixteen queries further is a constant stride; another 32 dims
		// flips address bits (kt::dims_flip)
		u32 const do_read_base = kt::rows_offset(klane, group);
		// transposed reads ("A" of dV^T and dK^T: dim 16 dt + klane, the 8 queries 4 group + 0..3 and 16 + 4 group + 0..3):
		// lane t of sixteen asks for eight bytes of query 4 group + t / 4
		u32 const tr_base = kt::piece_offset(4 * group + (klane >> 2), klane & 3);
		constexpr u32 SIXTEEN_ROWS = 16 * HD * 2;
		i8 const *q_head = q + row_base * Q_STRIDE + (size_t)head * HD;
		i8 const *kv_head = kv + row_base * KV_STRIDE + (size_t)head * 2 * HD;
		u8 const *do_head = reinterpret_cast<u8 const *>(d_out) + (row_base * O_STRIDE + (size_t)head * HD) * 2;
		f32 const *l_head = l + (size_t)head * all_rows + row_base;
		f32 const *d_head = d_rows + (size_t)head * all_rows + row_base;
		f32 const head_temperature = attn_temperature[head];

		// the addresses of the next tile to request; a step past the walk's end requests the last tile again, into a slot
		// nobody reads any more, so that the waits are constants
		i8 const *q_tile = q_head + (size_t)(tile_begin * kt::Q_PER_STEP) * Q_STRIDE;
		u8 const *do_tile = do_head + (size_t)(tile_begin * kt::Q_PER_STEP) * (O_STRIDE * 2);
		f32 const *ld_tile = (lane < 32 ? l_head : d_head) + tile_begin * kt::Q_PER_STEP + lane % 32;      // lanes 0..31 L, 32..63 D
		// (slots are the same in every lane; reading their offsets from the first one tells the compiler so.  A scalar write of
		// M0 needs one wait state before a direct-to-LDS load reads it)
		auto request_q = [&](u32 slot, bool further) __attribute__((always_inline)) {
			if (kt::Q_STAGERS == kt::THREADS_PER_BLOCK || q_stager) {
				asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
				             :: "s"(lds_wave + __builtin_amdgcn_readfirstlane(slot * kt::Q_RAW_BYTES)), "i"(kt::Q_RAW_OFFSET), "v"(q_src), "s"(q_tile) : "memory", "m0", "scc");
			}
			if (wave == kt::LD_WAVE) {
				asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, off"
				             :: "s"(lds_wave + __builtin_amdgcn_readfirstlane(slot * kt::LD_BYTES)), "i"(kt::LD_OFFSET - kt::LD_WAVE * 1024), "v"(ld_tile) : "memory", "m0", "scc");
				ld_tile += further ? kt::Q_PER_STEP : 0;
			}
			q_tile += further ? (size_t)kt::Q_PER_STEP * Q_STRIDE : 0;
		};
		auto request_do = [&](u32 slot, bool further) __attribute__((always_inline)) {
			if (kt::WIDE_STAGERS == kt::THREADS_PER_BLOCK || wide_stager) {
				u32 const base = lds_wave + __builtin_amdgcn_readfirstlane(slot * kt::WIDE_BYTES);
				asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
				             :: "s"(base), "i"(kt::DO_OFFSET), "v"(do_src), "s"(do_tile) : "memory", "m0", "scc");
				if constexpr (kt::WIDE_PASSES == 2) {
					asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
					             :: "s"(base), "i"(kt::DO_OFFSET + kt::WIDE_STAGERS * 16), "v"(do_src), "s"(do_tile + (size_t)16 * O_STRIDE * 2) : "memory", "m0", "scc");
				}
			}
			do_tile += further ? (size_t)kt::Q_PER_STEP * (O_STRIDE * 2) : 0;
		};
		// Q tile int8 -> bf16, by the threads that requested it, and the tile's per-query constants
		auto prepare = [&](u32 tile, u32 slot, u32 buf) __attribute__((always_inline)) {
			if (kt::Q_STAGERS == kt::THREADS_PER_BLOCK || q_stager) {
				v4u const raw = *reinterpret_cast<v4u const *>(smem + kt::Q_RAW_OFFSET + slot * kt::Q_RAW_BYTES + tid * 16);
				u8 *dst = smem + kt::Q_WIDE_OFFSET + buf * kt::WIDE_BYTES;
				v2u const a = widen4(raw[0]), b = widen4(raw[1]), c = widen4(raw[2]), d = widen4(raw[3]);
				*reinterpret_cast<v4u *>(dst + q_wide_dst) = v4u{a[0], a[1], b[0], b[1]};
				*reinterpret_cast<v4u *>(dst + (q_wide_dst ^ 16u)) = v4u{c[0], c[1], d[0], d[1]};
			}
			if (wave == kt::LD_WAVE) {
				f32 const landed = *reinterpret_cast<f32 const *>(smem + kt::LD_OFFSET + slot * kt::LD_BYTES + lane * 4);
				f32 *cst = reinterpret_cast<f32 *>(smem + kt::CONST_OFFSET + buf * kt::CONST_BYTES);
				cst[kt::Q_PER_STEP + lane] = lane < 32 ? landed - LOG2_PROB_SCALE : landed;       // L - lg2 255 | D
				if (lane < 32) {
					u32 const qi = tile * kt::Q_PER_STEP + lane;
					u32 const visible = qi < wr ? qi : wr;
					cst[lane] = (BASE_TEMPERATURE * sfu::lg2(f32(visible + 4u))) * head_temperature;
				}
			}
		};

		// the first tiles are requested ahead of the wavefront's own operands (every walk has at least two tiles; where it has no
		// third, the second is requested again)
		__syncthreads();                      // the previous item's LDS is no longer read
		request_q(0, true);
		request_q(1, n_steps > 2);
		request_do(0, true);
		request_q(2, n_steps > 3);

		// ---- the wavefront's own operands
		v4i kf[K_SLICES];                    // "B" of S: lane = key, the 16 bytes 64 s + 16 group of its row
		X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
			kf[s] = v4i{0, 0, 0, 0};
			if (k_group_in_row) kf[s] = *reinterpret_cast<v4i const *>(kv_head + (size_t)key * KV_STRIDE + 64 * s + 16 * group);
		}
		v8bf vfrag[D_SLICES];                // "B" of dP: lane = key, dims 32 sl + 8 group + 0..7 as bf16, real values (code / 8)
		X17_UNROLL for (u32 sl = 0; sl < D_SLICES; ++sl) {
			v2u const raw = *reinterpret_cast<v2u const *>(kv_head + (size_t)key * KV_STRIDE + HD + 32 * sl + 8 * group);
			v2u const a = widen4(raw[0], 0.125f), b = widen4(raw[1], 0.125f);
			vfrag[sl] = __builtin_bit_cast(v8bf, (v4u{a[0], a[1], b[0], b[1]}));
		}
		v4f dk_acc[D_TILES], dv_acc[D_TILES];    // (dims x keys): lane = key, register r = dim 16 dt + 4 group + r
		X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
			dk_acc[dt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
			dv_acc[dt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
		}

		__builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
		prepare(tile_begin, 0, 0);

		// One pipeline step, common to all wavefronts of the workgroup.  SLOT: the step's position in the ring as a compile-time
		// number, or -1 for "compute it"; SLOT >= 0 also says that tile i + 4 exists (the caller's loop bound).
		auto advance = [&]<int SLOT>(u32 i) __attribute__((always_inline)) {
			u32 const slot = SLOT >= 0 ? (u32)SLOT : i % kt::RING;
			// this thread's requests for dO tile i and Q tile i + 1 have landed (those for Q tile i + 2, and its L and D, may be in
			// flight: the last one or two of step i - 1); its LDS traffic of step i - 1 is complete; after the barrier so is
			// everybody else's: tile i is visible, the slots of Q tile i - 1 and dO tile i - 1 are free
			if (wave == kt::LD_WAVE) {
				__builtin_amdgcn_s_waitcnt(kt::Q_STAGERS == kt::THREADS_PER_BLOCK ? 0x0F72 : 0x0F71);
			} else {
				__builtin_amdgcn_s_waitcnt(kt::Q_STAGERS == kt::THREADS_PER_BLOCK ? 0x0F71 : 0x0F70);      // (wavefronts that request no Q: all of dO)
			}
			__builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
			__builtin_amdgcn_s_barrier();
			request_do((slot + 1) & 1, SLOT >= 0 || i + 2 < n_steps);
			request_q((slot + 3) % kt::RING, SLOT >= 0 || i + 4 < n_steps);
		};
		auto prepare_next = [&]<int SLOT>(u32 i) __attribute__((always_inline)) {
			u32 const slot = SLOT >= 0 ? (u32)SLOT : i % kt::RING;
			prepare(tile_begin + i + 1, (slot + 1) % kt::RING, (slot + 1) & 1);
		};
		// the step's arithmetic for this wavefront's 16 keys
		auto compute = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
			u32 const slot = SLOT >= 0 ? (u32)SLOT : i % kt::RING;
			u8 const *q_raw = smem + kt::Q_RAW_OFFSET + slot * kt::Q_RAW_BYTES;
			u8 const *d_o = smem + kt::DO_OFFSET + (slot & 1) * kt::WIDE_BYTES;
			u8 const *q_wide = smem + kt::Q_WIDE_OFFSET + (slot & 1) * kt::WIDE_BYTES;
			u8 const *cst = smem + kt::CONST_OFFSET + (slot & 1) * kt::CONST_BYTES;
			u32 do_off = do_read_base, tr_off = tr_base, cst_off = 16 * group;
			asm volatile("" : "+v"(do_off), "+v"(tr_off));      // (keeps the flipped addresses out of registers that live across steps)
			u32 pw[2 * Q_TILES], ww[2 * Q_TILES];     // P and the dK weights as bf16 pairs: "B" operands, slots = this lane's 8 queries
			X17_UNROLL for (u32 qt = 0; qt < Q_TILES; ++qt) {
				// S and dP blocks: rows = 16 queries of the tile, columns = this wave's 16 keys
				v4i s_acc = {0, 0, 0, 0};
				X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
					v4i qa = *reinterpret_cast<v4i const *>(q_raw + q_read_off[qt][s]);
					if (!k_group_in_row) qa = v4i{0, 0, 0, 0};
					s_acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa, kf[s], s_acc, 0, 0, 0);
				}
				v4f dp_acc = {0.0f, 0.0f, 0.0f, 0.0f};
				auto multiply_dp = [&]() __attribute__((always_inline)) {
					X17_UNROLL for (u32 sl = 0; sl < D_SLICES; ++sl) {
						v8bf const da = *reinterpret_cast<v8bf const *>(d_o + (do_off ^ kt::dims_flip(32 * sl)) + qt * SIXTEEN_ROWS);
						dp_acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(da, vfrag[sl], dp_acc, 0, 0, 0);
					}
				};
				if constexpr (!DP_LATE) multiply_dp();
				// register r belongs to query 32 tile + 16 qt + 4 group + r; key j is visible to query i iff the distance
				// i - 1 - j, as an unsigned number, is at most W' - 1
				[[maybe_unused]] u32 const first = (tile_begin + i) * kt::Q_PER_STEP + 16 * qt + 4 * group - 1 - key;
				v4f const ct = *reinterpret_cast<v4f const *>(cst + cst_off + 64 * qt);
				v4f const cl = *reinterpret_cast<v4f const *>(cst + cst_off + 4 * kt::Q_PER_STEP + 64 * qt);
				f32 p[4], w[4];
				X17_UNROLL for (u32 r = 0; r < 4; ++r) {
					f32 pe = sfu::ex2(fmaf32(f32(s_acc[r]), ct[r], -cl[r]));
					if constexpr (MASKED) {
						pe = first + r <= vis_bound ? pe : 0.0f;
					}
					p[r] = pe;
				}
				asm volatile("" : "+v"(cst_off) : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]));
				if constexpr (DP_LATE) {
					asm volatile("" : "+v"(do_off) : "v"(cst_off));
					multiply_dp();
				}
				v4f const cd = *reinterpret_cast<v4f const *>(cst + cst_off + 8 * kt::Q_PER_STEP + 64 * qt);
				X17_UNROLL for (u32 r = 0; r < 4; ++r) w[r] = (p[r] * (dp_acc[r] - cd[r])) * ct[r];
				pw[2 * qt] = pack2_bf16_rne(p[0], p[1]);
				pw[2 * qt + 1] = pack2_bf16_rne(p[2], p[3]);
				ww[2 * qt] = pack2_bf16_rne(w[0], w[1]);
				ww[2 * qt + 1] = pack2_bf16_rne(w[2], w[3]);
			}
			prepare_next.template operator()<SLOT>(i);
			static_assert(Q_TILES == 2, "one 16 x 16 x 32 instruction contracts over the step's 32 queries");
			v8bf const pfrag = __builtin_bit_cast(v8bf, (v4u{pw[0], pw[1], pw[2], pw[3]}));
			v8bf const wfrag = __builtin_bit_cast(v8bf, (v4u{ww[0], ww[1], ww[2], ww[3]}));
			X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
				u32 const lo = tr_off ^ kt::dims_flip(16 * dt), hi = lo + SIXTEEN_ROWS;
				dv_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
					transposed_fragment(d_o + lo, d_o + hi), pfrag, dv_acc[dt], 0, 0, 0);
				dk_acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
					transposed_fragment(q_wide + lo, q_wide + hi), wfrag, dk_acc[dt], 0, 0, 0);
			}
		};
		auto step = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
			advance.template operator()<SLOT>(i);
			compute.template operator()<MASKED, SLOT>(i);
		};
		auto idle_step = [&](u32 i) __attribute__((always_inline)) {
			advance.template operator()<-1>(i);
			prepare_next.template operator()<-1>(i);
		};
		// A wavefront's keys are seen by the tiles [wave_tile_first, wave_tile_last] of the workgroup's walk: plain loops for
		// nothing to do, the diagonal, tiles all of whose queries see all of its keys, the window's edge, nothing to do
		// (around a skip the compiler moves the accumulators about once per step).  The long run is unrolled over the slots
		// of the ring, so that every LDS address is a register plus an immediate.
		u32 const lead = wave_tile_first - tile_begin;
		u32 const active_end = wave_tile_last + 1 - tile_begin < n_steps ? wave_tile_last + 1 - tile_begin : n_steps;
		u32 const full_tile = (key_wave0 + kt::KEYS_PER_WAVE + kt::Q_PER_STEP - 1) / kt::Q_PER_STEP - tile_begin;
		u32 const full_begin = full_tile < active_end ? full_tile : active_end;
		u32 const full_tile_end = wr >= seq_len ? active_end : (key_wave0 + wr + 1) / kt::Q_PER_STEP;      // (tiles up to its own keys': not before tile_begin)
		u32 const full_end = wr >= seq_len ? active_end : full_tile_end <= tile_begin + full_begin ? full_begin
		                   : (full_tile_end - tile_begin < active_end ? full_tile_end - tile_begin : active_end);
		u32 i = 0;
		for (; i < lead; ++i) idle_step(i);
		for (; i < full_begin; ++i) step.template operator()<true, -1>(i);
		for (; i < full_end && i % kt::RING != 0; ++i) step.template operator()<false, -1>(i);
		for (; i + kt::RING <= full_end && i + 2 * kt::RING <= n_steps; i += kt::RING) {
			step.template operator()<false, 0>(i);
			step.template operator()<false, 1>(i + 1);
			step.template operator()<false, 2>(i + 2);
			step.template operator()<false, 3>(i + 3);
		}
		for (; i < full_end; ++i) step.template operator()<false, -1>(i);
		for (; i < active_end; ++i) step.template operator()<true, -1>(i);
		for (; i < n_steps; ++i) idle_step(i);

		// ---- output: dk = 8 ln 2 * dk_acc, dv = dv_acc.  A key's dK and dV are one run of memory, a lane holds eight bytes of it at
		// a time: turned around in LDS they leave as whole rows, 16 bytes per lane (8-byte stores straight from the
		// registers, 32 bytes per row and instruction: a fifth of the launch at 4 x 8192 tokens).
		__builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0): the last requests write LDS
		__syncthreads();
		u32 out_lane = lane;
		asm volatile("" : "+v"(out_lane));    // (or the addresses below are kept in registers through the walk, and spilled)
		u32 const out_key = out_lane % 16, out_group = out_lane / 16;
		u8 *rows_lds = smem + wave * kt::OUT_BYTES_PER_WAVE;
		X17_UNROLL for (u32 dt = 0; dt < D_TILES; ++dt) {
			v2u const k_pair = {pack2_bf16_rne(dk_acc[dt][0] * EIGHT_LN2, dk_acc[dt][1] * EIGHT_LN2), pack2_bf16_rne(dk_acc[dt][2] * EIGHT_LN2, dk_acc[dt][3] * EIGHT_LN2)};
			v2u const v_pair = {pack2_bf16_rne(dv_acc[dt][0], dv_acc[dt][1]), pack2_bf16_rne(dv_acc[dt][2], dv_acc[dt][3])};
			*reinterpret_cast<v2u *>(rows_lds + kt::out_offset(out_key, 2 * dt + out_group / 2) + 8 * (out_group % 2)) = k_pair;
			*reinterpret_cast<v2u *>(rows_lds + kt::out_offset(out_key, HD / 8 + 2 * dt + out_group / 2) + 8 * (out_group % 2)) = v_pair;
		}
		u16 *dkv_rows = d_kv + (row_base + key_wave0) * KV_STRIDE + (size_t)head * 2 * HD;
		X17_UNROLL for (u32 j = 0; j < kt::OUT_BYTES_PER_WAVE / 1024; ++j) {
			u32 const n = 64 * j + out_lane, row = n / kt::OUT_CPR, c = n % kt::OUT_CPR;
			*reinterpret_cast<v4u *>(dkv_rows + (size_t)row * KV_STRIDE + 8 * c) = *reinterpret_cast<v4u const *>(rows_lds + kt::out_offset(row, c));
		}
	}
}
