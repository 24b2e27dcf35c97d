// attn_fwd_i8.hip -- int8 causal sliding-window flash-attention forward with a sink token and
// scalable-softmax temperature, for gfx950.
//
// Replaces the reference's AttnForward (cuda/attn_fwd_i8.cuh:30-620); the kernel entry and its
// parameters follow templates/attn/kernel.cu:9-33.  The arithmetic it reproduces, per head and
// query i (0-based position inside its sequence):
//   keys j in [max(0, i - W'), i - 1] plus one sink key/value; W' = window rounded up to 16
//   (0 = no window);  n = min(W', i) + 4;  temperature = f32(hd^-1/2 / 64) * lg2(n) * head_temp[h];
//   s_j = f32(q_i . k_j) * temperature (int32 dot);  running max starts at the sink score, the
//   partial sums at 4 x 63.75, O at 255 * sink_v;  per 16-key tile (ascending): rescale when the
//   max grows, p_j = ex2(s_j - max) * 255, four partial sums over key quads of the tile,
//   P_j = rne(p_j), O += f32(sum_j P_j v_j);  at the end sum = (s0+s1)+(s2+s3),
//   L = lg2(sum) + max, out = fixedi8(O / sum).
//
// Design, MI355X-first:
//   * One workgroup = 4 wavefronts = 128 queries of one head; a wavefront owns 32 queries.
//     Keys/values are staged 32 keys per step (two 16-key tiles) through rings in LDS.
//   * S^T = K . Q^T on v_mfma_i32_32x32x32_i8 with the KEYS as the MFMA "A" operand: a lane then
//     owns one query (lane % 32) and 8 keys of each 16-key tile; the other 8 keys sit in lane+32.
//     Row max needs one cross-lane exchange per tile; the four per-quad partial sums of the
//     reference fall two-and-two into the lane pair, so they need none until the very end.
//   * P stays in registers: packed to f16 it already IS the "B" operand of O^T = V^T . P^T.
//     PV runs on v_mfma_f32_32x32x16_f16: K = 16 is exactly one 16-key tile, P (0..255) and
//     int8 V are exact in f16 and every tile sum is below 2^24, so the f32 result equals the
//     reference's f32(int32 dot) bit for bit.  (CDNA4 has no unsigned x signed int8 MFMA; an
//     int8 PV would need two MFMAs per tile for the 8-bit probabilities.)
//   * K and V go global -> LDS directly, three 32-key steps ahead of their use.  V is widened to
//     f16 once per workgroup, LDS -> LDS, one step ahead (sign-bit flip, byte splice under the
//     exponent of 1024, subtract 1152: five instructions per four values) and fetched transposed
//     with ds_read_b64_tr_b16, so no register transposes.
//   * Three workgroups share a compute unit (register budget of 168 per lane), so one workgroup's
//     waits for its tiles and its barrier are covered by the others' arithmetic.
//   * X17_STRICT_MATH = 1: deterministic ex2 and one explicit f32 add per tile (parity build).  Same key loop as the
//     speed build (runs of steps per mask class, hand-written tile requests with constant waits: around the compiler's
//     own direct-to-LDS loads it waits for every load in flight before a step's LDS reads).  64 heads of 32, 16384
//     tokens, no window: 5300 us on a plain loop, 3440 us on this one with five wavefronts per SIMD.
//     X17_STRICT_MATH = 0: v_exp_f32 with the factor 255 folded into the exponent, accumulation
//     inside the PV MFMA, and lazy rescaling of O (speed build; results stay within one output code).
//
// common.h (generated per kernel) provides X17_N_HEADS, X17_HEAD_DIM, X17_Q_STRIDE,
// X17_KV_STRIDE, X17_O_STRIDE, X17_STRICT_MATH.
//
// Extension over the reference ABI: gridDim.z = number of independent sequences stacked along
// the rows of q / kv / out (each `seq_len` rows, own causal origin); L is [H, gridDim.z * seq_len].
//
// X17_ATTN_ROW_SCALES = 1 (no counterpart in the reference, whose codes share the constant scale 1/8):
// five more parameters give one f32 scale per (head, row) for q and k, a weight <= 1 per (head, row)
// for v (all three laid out [H, rows] like L), and per head the weight of the sink value and the output
// scale.  The recurrence becomes
//   tq = ((f32(hd^-1/2) * lg2(n)) * head_temp[h]) * q_scale[h, i],  s_j = (f32(q_i . k_j) * k_scale[h, j]) * tq,
//   sink score = f32(q_i . sink_k) * (tq * 0.125),  P_j = rne(p_j * v_weight[h, j]),
//   O starts at f32(255 * sink_v) * sink_v_weight[h],  out = store((O * rcp(sum)) * out_scale[h])
// and produces the bits of the plain kernel when every scale is 1/8 and every weight and out_scale is 1.
// X17_ATTN_OUT_BF16 = 1 stores bf16 real values (round to nearest even) instead of FixedI8 codes.

#include "common.h"
#include "x17_device.h"
#include "attn_tile.h"
#include "attn_parts.h"

using namespace x17;
namespace at = x17::attn_tile;
using namespace x17::attn_parts;

namespace {

constexpr u32 HD = X17_HEAD_DIM;
constexpr u32 N_HEADS = X17_N_HEADS;
constexpr u32 Q_STRIDE = X17_Q_STRIDE;
constexpr u32 KV_STRIDE = X17_KV_STRIDE;
constexpr u32 O_STRIDE = X17_O_STRIDE;
constexpr u32 HPK = at::HEADS_PER_KERNEL;
constexpr u32 K_SLICES = HD / 32;      // 32 bytes of head_dim per QK MFMA
constexpr u32 D_BLOCKS = HD / 32;      // 32 output dims per PV MFMA
constexpr u32 CPR = HD / 16;           // 16-byte chunks per key row
constexpr bool STRICT = X17_STRICT_MATH != 0;
constexpr bool ROW_SCALES = at::ROW_SCALES;
constexpr bool OUT_BF16 = X17_ATTN_OUT_BF16 != 0;
static_assert(ROW_SCALES || !OUT_BF16, "the bf16 output needs the row-scaled build (it supplies out_scale)");

static_assert(HD == 32 || HD == 64 || HD == 128, "head_dim must be 32, 64 or 128");
static_assert(N_HEADS % HPK == 0, "n_heads must be divisible by heads_per_kernel");

constexpr f32 BASE_TEMPERATURE = ROW_SCALES ? f32(constexpr_inv_sqrt(f64(HD)))
                                            : f32(constexpr_inv_sqrt(f64(HD)) / 64.0);   // :47, :447-449

typedef short v4s __attribute__((ext_vector_type(4)));

// V tile (f16): linear 32-byte granule n = key * CPR + c (16 dims) lives in 256-byte line n / 8
// at position (n % 8) ^ ((line & 3) << 1): the 4 keys x 2 granules that 32 lanes of a transposed
// read touch then cover all 64 banks exactly once (checked exhaustively for head_dim 32/64/128).
X17_DEV u32 v_granule_offset(u32 key, u32 c) {
	u32 n = key * CPR + c;
	u32 line = n >> 3;
	return (line << 8) | (((n & 7) ^ ((line & 3) << 1)) << 5);
}

// Strict build without row scales.  The reference's numbers at powers of two of its own scale, so that a score of a fully visible tile
// takes 17 vector instructions instead of 19 and the slow ones of them (conversion, comparison and select, rounding) go:
//  * Score accumulators start at the bits of DOT_START = 1 / 2 pi, which the matrix instruction takes as an inline constant: read as a
//    float the sum is DOT_START + dot * 2^-26 exactly (0x3E22F983 has 2 292 099 steps of 2^-26 below it in its binade and
//    more above, |dot| <= 128 * 128 * 128), one exact subtraction away from the dot product.
//  * Scores, and the maximum their probabilities refer to, at 2^-7: maximum - score is what ex2 takes, and the subtraction's own
//    clamp to [0, 1] keeps its argument above -128.
//  * ex2's polynomial at one half: a result below 2^-125, which the reference's ex2 flushes, then has an exponent field of 0 (an f32
//    denormal) or a negative one (a set sign bit, or a NaN).  The key loop runs with f32 denormals flushed, so that the multiplication by 255
//    takes the former for 0; its clamp makes 0 of the latter, of NaNs too.  The clamp wants probabilities below 1: they and the partial sums
//    are at 2^-8.  (What else could be denormal there has no bearing on the output: O and the sums, decayed by 2^-100 and
//    more, next to a sum of at least 63.)
//  * Adding 1.5 * 2^15 rounds p / 256 to the integer P and leaves it in the low half of the sum, where it is the f16 denormal
//    P * 2^-24: the matrix instructions multiply those exactly, O is at 2^-24.
// Powers of two change no rounding, so the bits are the reference's.  A head whose temperature is zero, not finite or outside
// 2^-40 .. 2^40 takes the masked steps throughout.  Bound by vector issue (2.5 clocks an instruction, by the counters):
// 64 heads of 32, 16384 tokens, no window 3219 -> 3047 us; 32 heads of 128, 8192 tokens 868 -> 831 (in turn, three times each).
constexpr bool SCALED_SUMS = STRICT && !ROW_SCALES;
constexpr u32 DOT_START_BITS = 0x3E22F983u;
static_assert((DOT_START_BITS & 0x7FFFFFu) >= 128 * 128 * HD && 0x7FFFFFu - (DOT_START_BITS & 0x7FFFFFu) >= 128 * 128 * HD, "every dot product stays in DOT_START's binade");
constexpr f32 DOT_START = __builtin_bit_cast(f32, DOT_START_BITS);
constexpr f32 SUM_SCALE = SCALED_SUMS ? 0.00390625f : 1.0f;                        // 2^-8
constexpr f32 SUM_PROB_SCALE = PROB_SCALE * SUM_SCALE;
constexpr f32 O_SCALE = SCALED_SUMS ? 5.9604644775390625e-08f : 1.0f;              // 2^-24
constexpr f32 ROUND_MAGIC = 49152.0f;                                               // 1.5 * 2^15: last place 2^-8
constexpr f32 EX2_MAGIC = 98304.0f;                                                 // 1.5 * 2^16: last place 2^-7
constexpr int F32_DENORMALS = 1 | 4 << 6 | 1 << 11;                                 // the register MODE, its bits 4 and 5
X17_DEV bool regular_temperature(f32 t) { return ((f2u(t) >> 23) & 0xFFu) - 87u <= 80u; }
// Constants of the fully visible step, kept in scalar registers (an addition then is four bytes of code, not eight)
struct StepConstants {
	f32 dot_start = DOT_START, ex2_magic = EX2_MAGIC, minus_ex2_magic = -EX2_MAGIC, round_magic = ROUND_MAGIC;
	X17_DEV f32 dot(i32 sum) const { return (u2f((u32)sum) - dot_start) * 67108864.0f; }      // exact
	X17_DEV void keep() { asm volatile("" : "+s"(dot_start), "+s"(ex2_magic), "+s"(minus_ex2_magic), "+s"(round_magic)); }
};

// 255 / 256 * strict::ex2(-128 * below), with f32 denormals flushed
X17_DEV f32 scaled_probability(f32 below, StepConstants const &c) {
	f32 const x = __builtin_amdgcn_fmed3f(below, 0.0f, 1.0f);      // (becomes the subtraction's clamp)
	f32 const t = c.ex2_magic - x;
	f32 const g = (t + c.minus_ex2_magic) + x;                      // -f / 128
	// strict::ex2's coefficients in powers of g, halved
	constexpr auto of_g = [](f32 coefficient, int power) { f32 v = 0.5f * coefficient; for (int i = 0; i < power; ++i) v *= -128.0f; return v; };
	f32 p = of_g(0.00015453163359779865f, 6);
	p = fmaf32(p, g, of_g(0.0013390863314270973f, 5));
	p = fmaf32(p, g, of_g(0.009618083015084267f, 4));
	p = fmaf32(p, g, of_g(0.055503569543361664f, 3));
	p = fmaf32(p, g, of_g(0.24022650718688965f, 2));
	p = fmaf32(p, g, of_g(0.6931471824645996f, 1));
	p = fmaf32(p, g, of_g(1.0f, 0));
	f32 const r = u2f(f2u(p) + (f2u(t) << 23));                     // (the bits of EX2_MAGIC above the integer leave in the shift)
	return __builtin_amdgcn_fmed3f(r * (2.0f * SUM_PROB_SCALE), 0.0f, 1.0f);      // (the multiplication's clamp)
}

X17_DEV u32 pack_f16(f32 lo, f32 hi) {
	// both values are integers below 2048: exact in f16 whatever the rounding mode
	return __builtin_bit_cast(u32, __builtin_amdgcn_cvt_pkrtz(lo, hi));
}

// One 16-byte-per-lane direct-to-LDS load: LDS destination in M0 (wave-uniform; lane l lands 16 * l bytes further),
// global source = a uniform 64-bit base in scalar registers + a 32-bit offset per lane (the compiler's own selection
// forms a 64-bit address per lane with a 64-bit vector add in front of every load).
X17_DEV void load_to_lds_16(u8 *lds_uniform, i8 const *src_uniform, u32 lane_offset) {
	// (the address is the same in every lane; reading it from the first one tells the compiler so)
	u32 const lds = __builtin_amdgcn_readfirstlane((u32)(size_t)X17_LDS_PTR(lds_uniform));
	// (gfx9 family: a scalar write of M0 needs one wait state before a direct-to-LDS load reads it; the compiler
	// inserts it for its own loads and cannot see into this string)
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
	             :: "s"(lds), "v"(lane_offset), "s"(src_uniform) : "memory", "m0");
}

} // namespace

extern "C" __global__ __launch_bounds__(at::THREADS_PER_BLOCK)
__attribute__((amdgpu_waves_per_eu(at::WAVES_PER_SIMD, at::WAVES_PER_SIMD)))
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

	u32 const wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);

	// Which (sequence, head group, query block) this workgroup takes.  The hardware starts workgroups in the order of
	// their linear index (and deals them round-robin to the 8 XCDs).  The query block is the slowest index of that
	// order and runs from the last block to the first: the workgroups in flight at one time are the same few query
	// blocks of every (sequence, head group) pair -- neighbouring blocks of a pair share most of their key/value
	// window in the L2 of the XCD the pair keeps landing on when the pairs are a multiple of 8 -- and the blocks with
	// the shortest windows (the first of each sequence) come last, where they fill the tail of the launch.
	// Measured against the other orders on both long workloads: 2-4 % faster than query blocks fastest
	// (4 x 8192 tokens, window 512), 7 % faster on 65536 tokens with a window of 4096.
	u32 const pairs = gridDim.y * gridDim.z;
	u32 const lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
	u32 const pair = lin % pairs;
	u32 const q_block_index = gridDim.x - 1 - lin / pairs;
	// heads of this workgroup, one behind the other: the grid says how many groups they were cut into (one group per head
	// by this library's launchers, groups of 128 / head_dim heads by src/device/cuda/attn.rs:60-66)
	u32 const heads_here = HPK == 1 ? 1 : N_HEADS / gridDim.y;
	u32 const head_group = pair % gridDim.y;
	u32 const seq = pair / gridDim.y;
	size_t const row_base = (size_t)seq * seq_len;          // first row of this sequence
	// position of the block's first query; a last block that would overhang the sequence (lengths are multiples of 64,
	// src/device/cuda/attn.rs:398-404) starts earlier and recomputes some of its neighbour's queries
	u32 const q_block0 = at::block_first_query(q_block_index, seq_len);
	u32 const q_wave0 = q_block0 + wave * at::Q_PER_WAVE;

	// cuda/attn_fwd_i8.cuh:408-412 -- window 0 means "no window"; otherwise rounded up to 16
	u32 const wr = at::rounded_window(window_size);
	u32 const vis_bound = wr - 1 < 0x7FFFFFFFu ? wr - 1 : 0x7FFFFFFFu;

	// key blocks (32 keys) the workgroup walks, and the sub-range this wave needs
	u32 const kb_begin = at::first_key_block(q_block0, wr);
	u32 const kb_end = at::end_key_block(q_block0);                          // exclusive
	u32 const wave_kb_first = at::first_key_block(q_wave0, wr);
	u32 const wave_kb_last = q_wave0 / at::KV_PER_STEP;                      // inclusive

	for (u32 hh = 0; hh < heads_here; ++hh) {
		u32 const head = head_group * heads_here + hh;
		// (opaque: what a head derives from it is derived anew for the next one, not kept in registers from here on)
		u32 tid = threadIdx.x;
		if constexpr (STRICT) asm volatile("" : "+v"(tid));
		u32 const lane = tid % 64;
		u32 const half = lane / 32;
		u32 const qlane = lane % 32;
		u32 const qi = q_wave0 + qlane;                     // this lane's query position
		i8 const *q_head = q + row_base * Q_STRIDE + (size_t)head * HD;
		i8 const *kv_head = kv + row_base * KV_STRIDE + (size_t)head * 2 * HD;

		// ---- staging helpers for one 32-key block.  Both K and V travel global -> LDS without passing
		// through registers (thread t fetches 16-byte chunk t of each tile), PREFETCH steps ahead; one step
		// before its use a V tile is widened LDS -> LDS by the threads that fetched it.
		bool const stager = at::is_stager(tid);
		u32 stage_k_src = 0, stage_v_src = 0, widen_dst = 0;
		if (stager) {
			// lane `tid` fills stored chunk `tid` of the K tile (attn_tile.h finds which logical chunk lives there)
			stage_k_src = at::stage_k_offset(tid, KV_STRIDE);
			stage_v_src = at::stage_v_offset(tid, KV_STRIDE);
			widen_dst = v_granule_offset(tid / CPR, tid % CPR);
		}
		u32 const stage_lds = wave * 1024;                // wave-uniform part of the direct-to-LDS address
		auto widen_v = [&](u32 slot, u32 tile) {
			if (CPR == 8 || stager) {          // (head_dim 128: every thread stages)
				v4u raw = *reinterpret_cast<v4u const *>(smem + at::RAW_V_RING_OFFSET + slot * at::RAW_V_TILE_BYTES + tid * 16);
				u32 w[8];
				widen16(raw, w);
				u8 *dst = smem + at::V_TILES_OFFSET + tile * at::V_TILE_BYTES + widen_dst;
				*reinterpret_cast<v4u *>(dst) = v4u{w[0], w[1], w[2], w[3]};
				*reinterpret_cast<v4u *>(dst + 16) = v4u{w[4], w[5], w[6], w[7]};
			}
		};
		static_assert(at::PREFETCH == 3, "the waits below are written for a prefetch distance of 3");

		// ---- per-query setup (cuda/attn_fwd_i8.cuh:444-517)
		v4i qf[K_SLICES];
		X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
			qf[s] = *reinterpret_cast<v4i const *>(q_head + (size_t)qi * Q_STRIDE + 32 * s + 16 * half);
		}
		u32 const visible = qi < wr ? qi : wr;
		f32 temperature = BASE_TEMPERATURE * strict::lg2(f32(visible + 4u));
		temperature = temperature * attn_temperature[head];
#if X17_ATTN_ROW_SCALES
		temperature = temperature * q_scale[(size_t)head * ((size_t)gridDim.z * seq_len) + row_base + qi];
#endif
		// (the sign is the head's: lg2(visible + 4) >= 2)
		bool const positive_temperature = __builtin_amdgcn_readfirstlane(f2u(attn_temperature[head])) - 1u < 0x7F7FFFFFu;

		i32 sink_dot = 0;
		X17_UNROLL for (u32 s = 0; s < K_SLICES; ++s) {
			v4i sk = *reinterpret_cast<v4i const *>(sink_k + (size_t)head * HD + 32 * s + 16 * half);
			X17_UNROLL for (int w = 0; w < 4; ++w) sink_dot = __builtin_amdgcn_sdot4(qf[s][w], sk[w], sink_dot, false);
		}
		sink_dot += partner_i32(sink_dot, half);

		f32 m = ROW_SCALES ? f32(sink_dot) * (temperature * 0.125f) : f32(sink_dot) * temperature;
		f32 lift = 1.0f;                     // speed build: 2^(m - the maximum O's scale refers to)
		v2h lift2 = {(_Float16)1.0f, (_Float16)1.0f};
		f32 sum_lo = 0.25f * SUM_PROB_SCALE;     // partial sum of key quad `half` of every tile
		f32 sum_hi = 0.25f * SUM_PROB_SCALE;     // partial sum of key quad `2 + half`
		// (the lane pair holds the reference's four partial sums two-and-two; each starts at 63.75)
		v16f o_acc[D_BLOCKS];                // O^T: lane = query, register r = dim 32*db + 8*(r/4) + 4*half + r%4
		if constexpr (!STRICT && !ROW_SCALES) {
			// Speed build: O starts at 255 * sink_v at the scale 2^-12 its accumulation starts from (see below), and the
			// matrix cores compute that as the outer product (sink_v) x (255 * 2^-12): key slot 0 of the V^T operand
			// holds the sink value of the lane's dim, key slot 0 of the P^T operand the constant, every other slot is
			// zero -- one product per element, exact.  (A few instructions per 32 dims instead of a conversion, a fused
			// multiply-add and a multiplication per element.)
			typedef short v8s __attribute__((ext_vector_type(8)));
			_Float16 const p0 = half == 0 ? (_Float16)(PROB_SCALE / 4096.0f) : (_Float16)0.0f;
			v8s pz = {0, 0, 0, 0, 0, 0, 0, 0};
			pz[0] = __builtin_bit_cast(short, p0);
			X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
				_Float16 const v0 = half == 0 ? (_Float16)(f32)(i32)sink_v[(size_t)head * HD + 32 * db + qlane] : (_Float16)0.0f;
				v8s vz = {0, 0, 0, 0, 0, 0, 0, 0};
				vz[0] = __builtin_bit_cast(short, v0);
				v16f const zero = {0};
				o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, vz), __builtin_bit_cast(v8h, pz), zero, 0, 0, 0);
			}
		} else
		X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
			X17_UNROLL for (int r4 = 0; r4 < 4; ++r4) {
				// 255 * v for the int8 byte v, through the unsigned byte v + 128 (one conversion and one fma per value, all exact)
				u32 const word = *reinterpret_cast<u32 const *>(sink_v + (size_t)head * HD + 32 * db + 8 * r4 + 4 * half) ^ 0x80808080u;
				X17_UNROLL for (int b = 0; b < 4; ++b) {
					o_acc[db][4 * r4 + b] = fmaf32(f32((word >> (8 * b)) & 0xFFu), 255.0f * O_SCALE, -32640.0f * O_SCALE);
				}
			}
		}
#if X17_ATTN_ROW_SCALES
		{
			f32 const sink_weight = sink_v_weight[head];
			X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
				X17_UNROLL for (int r = 0; r < 16; ++r) o_acc[db][r] = o_acc[db][r] * sink_weight;
			}
		}
#endif

		u32 const n_steps = kb_end - kb_begin;
		// ---- the key loop.  It is built around what the kernel turned out to be bound by: the number of instructions of ANY
		// kind a SIMD has to issue per step (scalar bookkeeping and waits count like vector arithmetic; with three
		// wavefronts per SIMD an instruction costs 1.5-2.5 ns of SIMD time whatever it does).  Both builds:
		//  * A wave's steps fall into runs -- nothing to do, masked (the window's edge), fully visible, the diagonal,
		//    nothing to do -- and each run is its own loop.  Every step requests a tile (past the end the last one
		//    again, into a slot nobody reads any more), so the waits are constants.
		//  * The long run (fully visible steps) is unrolled over the four phases of the tile ring: every LDS address
		//    is a register plus an immediate, and the ring arithmetic disappears from the scalar unit.
		//  * The tile requests take a scalar base and a lane offset; M0 is set by one scalar addition.
		// Speed build only:
		//  * The 8-bit probabilities are rounded and turned into f16 by one fused multiply-add and one byte shuffle per
		//    pair (PACK_MAGIC); the lift and the removal of the 1024 are one packed fma.
		//  * O and the partial sums live at the scale of a reference maximum kept HEADROOM above the running one
		//    whenever it is set: the lift of new probabilities then starts at 2^-12 (8-bit integers times it are still
		//    exact f16 values), a moving maximum costs one exponential, and O has to be brought down only after the
		//    maximum has grown by 17 (Gaussian scores move it by that much a few times per query block, not per tile).
		//  * The score accumulators start at the bits of 1.5 * 2^23 instead of zero: the int32 sum 0x4B400000 + dot,
		//    read as a float, is 12582912 + dot exactly (|dot| < 2^22), so no score is ever converted.  What refers to
		//    a maximum lives in that biased domain: `ext` is the running extreme of sgn * (12582912 + dot) (exact) and
		//    `mb` the subtrahend of the exponent, ext * |temperature| - lg2 255 rounded to a float.  That rounding (an
		//    ulp of 12582912 * temperature) would move the maximum the probabilities are rounded against; its exact
		//    remainder is therefore taken and 2^-remainder (`fine`) multiplies every probability inside operations that
		//    are needed anyway (the rounding addition is the fused multiply-add above, the sums' lift carries it).
		//  * The row maximum of a tile needs the partner lane's eight keys only when it moves: both lanes hold the same
		//    `ext`, and the tile's maximum exceeds it exactly when one of the two halves does.
		//  * Row-scaled build: a key's scale is not monotone in the dot product and the 16 registers of the bias words are
		//    not there to spend (they cost spills inside the loop), so the accumulators start at zero and
		//    z = f32(dot) * k_scale (a conversion and a multiplication per score); the
		//    extremes are taken over z as floats, and -- z being small -- the subtrahend ext * |t| - lg2 255 rounds to
		//    within 4e-6 of its value: no remainder is carried (`fine` is 1) and the value row's weight takes its place
		//    in the rounding fused multiply-add, P = rne(p * v_weight).  The first wavefront requests the step's 32 key
		//    scales and 32 value weights with the K tile (one more load in flight per prefetched step: its waits count
		//    three loads per step).  Scales are taken to be non-negative (absmax / 127): the sign of a query's
		//    temperature is then the head's.
		v16i s_bias;
		X17_UNROLL for (int r = 0; r < 16; ++r) s_bias[r] = SCALED_SUMS ? (i32)DOT_START_BITS : ROW_SCALES || STRICT ? 0 : 0x4B400000;
		if constexpr (!ROW_SCALES && !STRICT) {
			asm volatile("" : "+v"(s_bias));      // (kept in registers: rebuilding it per step would cost what it saves)
		}
		f32 const abs_t = __builtin_fabsf(temperature);
		// strict build, fully visible steps: what takes dot * 2^-26 to a score at 2^-7, and the maximum at 2^-7
		[[maybe_unused]] f32 const scaled_temperature = temperature * 524288.0f;
		[[maybe_unused]] f32 scaled_m = m * 0.0078125f;
		[[maybe_unused]] bool const regular = SCALED_SUMS && regular_temperature(u2f(__builtin_amdgcn_readfirstlane(f2u(attn_temperature[head]))));
		f32 const sgn = positive_temperature ? 1.0f : -1.0f;
		f32 ext = ROW_SCALES ? (f32(sink_dot) * 0.125f) * sgn : (f32(sink_dot) + DOT_BIAS) * sgn;
		[[maybe_unused]] f32 mb = 0.0f, fine = 1.0f;
		f32 ext_ref = ext;                        // O and the sums refer to the maximum HEADROOM above this extreme's score
		[[maybe_unused]] f32 sum_lift = 1.0f;
		[[maybe_unused]] v2h neg_bias2 = {(_Float16)(-1024.0f * LIFT0), (_Float16)(-1024.0f * LIFT0)};      // -1024 * lift2
		if constexpr (!STRICT) {
			set_subtrahend<ROW_SCALES>(ext, abs_t, mb, fine);
			lift = LIFT0;
			sum_lift = LIFT0 * fine;
			lift2 = v2h{(_Float16)LIFT0, (_Float16)LIFT0};
			sum_lo = sum_lo * LIFT0;
			sum_hi = sum_hi * LIFT0;
			if constexpr (ROW_SCALES) {
				X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
					X17_UNROLL for (int r = 0; r < 16; ++r) o_acc[db][r] = o_acc[db][r] * LIFT0;
				}
			}
		}
		u32 const first_active = wave_kb_first - kb_begin;
		u32 const diagonal = wave_kb_last - kb_begin;
		// first block that lies inside the window of all 32 queries: q_wave0 + 31 - 32 kb <= wr
		u32 const inside_kb = q_wave0 + 31 > wr ? (q_wave0 + 62 - wr) / 32 : 0;
		u32 const inside_clamped = inside_kb < wave_kb_first ? wave_kb_first : (inside_kb > wave_kb_last ? wave_kb_last : inside_kb);
		// (the speed build's fully visible steps take the row maximum over the scores' bits, which needs a positive
		// temperature, the strict build's scaled ones a regular one; with any other temperature every step goes the way of the masked ones)
		bool const all_masked = STRICT ? SCALED_SUMS && !regular : !positive_temperature;
		u32 const first_full = (all_masked ? wave_kb_last : inside_clamped) - kb_begin;

		// Tile requests.  Step s asks for K tile s + 3 and raw V tile s + 4, into the ring slots that K tile s - 1 and raw
		// V tile s have just left (a V tile is widened -- by the thread that fetched it -- during the step before its
		// use, so its slot is free one step earlier than a K slot): both tiles are on their way for three whole steps
		// before anything waits for them.  The requests of a thread complete in the order V0, (K0, V1), (K1, V2), ...;
		// step s needs the pair (K s, V s + 1), which leaves the two pairs behind it in flight.
		// `src` is the address of tile min(s + 3, last) when step s makes its requests; V tile s + 4 is one tile further
		// through a second lane offset, or the last tile again once the sequence ends.
		// SLOT: the step's position in the tile rings (s % RING) as a compile-time number, or -1 for "compute it".
		constexpr u32 TILE_STEP_BYTES = at::KV_PER_STEP * KV_STRIDE;
		i8 const *src = kv_head + (size_t)(kb_begin * at::KV_PER_STEP) * KV_STRIDE;
		u32 const stage_v_next = stage_v_src + TILE_STEP_BYTES;
		u32 const lds_wave = (u32)(size_t)X17_LDS_PTR(smem) + stage_lds;
		// SLOT >= 0 also says that tiles s + 3 and s + 4 both exist (the caller's loop bound)
		// row-scaled build, first wavefront: lane l < 32 fetches the scale of key l of the K tile being requested, lane
		// 32 + l the weight of its value row (4 bytes per lane, one 256-byte slot of the scale ring)
		[[maybe_unused]] f32 const *sc_src = nullptr;
#if X17_ATTN_ROW_SCALES
		sc_src = (half == 0 ? k_scale : v_weight) + (size_t)head * ((size_t)gridDim.z * seq_len) + row_base
		         + (size_t)kb_begin * at::KV_PER_STEP + qlane;
#endif
		// (by hand like the tile requests: in front of an LDS read the compiler waits for every direct-to-LDS load of its own,
		// and with it for all that were requested behind that one.  With the builtin the first wavefront drained its three
		// steps of prefetch every step: 65536 tokens, 32 heads of 128, window 4096: 3869 -> 3815 us; 1024 tokens, 8 heads
		// of 64: 15.5 -> 15.1 us)
		auto request_scales = [&](u32 ring_slot) __attribute__((always_inline)) {
			if (wave == 0) {
				asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, off"
				             :: "s"(lds_wave), "s"(at::SCALE_RING_OFFSET + ring_slot * at::SCALE_TILE_BYTES), "v"(sc_src) : "memory", "m0", "scc");
			}
		};
		auto request_tiles = [&]<int SLOT>(u32 s) __attribute__((always_inline)) {
			if constexpr (SLOT >= 0) {
				if constexpr (ROW_SCALES) {
					request_scales((SLOT + 3) % 4);
					sc_src += at::KV_PER_STEP;
				}
				if (CPR == 8 || stager) {
					asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
					             :: "s"(lds_wave), "i"(at::K_RING_OFFSET + ((SLOT + 3) % 4) * at::K_TILE_BYTES), "v"(stage_k_src), "s"(src) : "memory", "m0", "scc");
					asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
					             :: "s"(lds_wave), "i"(at::RAW_V_RING_OFFSET + SLOT * at::RAW_V_TILE_BYTES), "v"(stage_v_next), "s"(src) : "memory", "m0", "scc");
				}
				src += TILE_STEP_BYTES;
			} else {
				bool const more = at::further_tile_exists(s, n_steps);
				if constexpr (ROW_SCALES) {
					request_scales((s + 3) % at::RING);
					sc_src += __builtin_amdgcn_readfirstlane(more ? at::KV_PER_STEP : 0u);
				}
				if (CPR == 8 || stager) {
					load_to_lds_16(smem + at::K_RING_OFFSET + ((s + 3) % at::RING) * at::K_TILE_BYTES + stage_lds, src, stage_k_src);
					load_to_lds_16(smem + at::RAW_V_RING_OFFSET + (s % at::RING) * at::RAW_V_TILE_BYTES + stage_lds, src, more ? stage_v_next : stage_v_src);
				}
				if (more) {
					src += TILE_STEP_BYTES;
				}
			}
		};
		auto stage = [&]<int SLOT>(u32 i) __attribute__((always_inline)) {
			if (ROW_SCALES && wave == 0) {
				__builtin_amdgcn_s_waitcnt(0x0F76);      // vmcnt(6): three loads per step in the first wavefront
			} else {
				__builtin_amdgcn_s_waitcnt(0x0F74);      // vmcnt(4): K tile i and raw V tile i + 1 have landed
			}
			__builtin_amdgcn_s_waitcnt(0xC07F);          // lgkmcnt(0): own LDS traffic of step i-1 is complete
			__builtin_amdgcn_s_barrier();                // ... and so is everybody else's: tiles i are visible
			request_tiles.template operator()<SLOT>(i);
		};
		// raw V tile of step i + 1 -> f16 tile (i + 1) % 2
		auto widen_next = [&]<int SLOT>(u32 i) __attribute__((always_inline)) {
			if constexpr (SLOT >= 0) {
				widen_v((SLOT + 1) % at::RING, (SLOT + 1) & 1);
			} else {
				widen_v((i + 1) % at::RING, (i + 1) & 1);
			}
		};
		// maximum of a lane pair's two values, in both lanes
		auto pair_max_i32 = [](i32 x) {
			auto const r = __builtin_amdgcn_permlane32_swap((u32)x, (u32)x, false, false);
			return (i32)r[0] > (i32)r[1] ? (i32)r[0] : (i32)r[1];
		};

		// V^T operand of the 32 dims of block db: lane = dim 32 * db + lane % 32, slots = keys 16 * tile + {4 * half .. + 3,
		// 8 + 4 * half .. + 3}.  The lane's part of the address is the same for both tiles and both key groups
		// (they differ by whole 256-byte lines: 4096 bytes per tile, 2048 per group of 8 keys).
		// A key's granules fill CPR * 32 bytes; 16 keys further is always a whole number of 4-line groups further
		// (the swizzle key repeats), 8 keys further is one only when a key row has at least four granules.
		u32 v_lane_off[D_BLOCKS];
		[[maybe_unused]] u32 v_lane_off8[D_BLOCKS];
		{
			u32 const t = lane % 16, dh = (lane / 16) % 2;
			X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
				v_lane_off[db] = v_granule_offset(4 * half + (t >> 2), 2 * db + dh) + 8 * (t & 3);
				v_lane_off8[db] = v_granule_offset(8 + 4 * half + (t >> 2), 2 * db + dh) + 8 * (t & 3);
			}
		}
		auto v_fragment = [&](u8 const *v_tile, u32 tile, u32 db) __attribute__((always_inline)) {
			// (a key's granules fill whole lines of CPR * 32 bytes: 16 keys = one tile further, 8 keys = the other group)
			u8 const *p0 = v_tile + v_lane_off[db] + tile * (16 * CPR * 32);
			u8 const *p1 = CPR >= 4 ? p0 + 8 * CPR * 32 : v_tile + v_lane_off8[db] + tile * (16 * CPR * 32);
			v4s const lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)p0);
			v4s const hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *)p1);
			typedef short v8s __attribute__((ext_vector_type(8)));
			v8s const both = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
			return __builtin_bit_cast(v8h, both);
		};
		[[maybe_unused]] StepConstants step_constants;
		if constexpr (SCALED_SUMS) step_constants.keep();
		// Strict build, one 16-key tile: the reference's operations one by one.
		auto strict_tile = [&]<bool MASKED>(u32 i, u32 tile, v16i const &s_acc, u32 k_slot, u8 const *v_tile) __attribute__((always_inline)) {
			constexpr bool SCALED = !MASKED && SCALED_SUMS;      // scores at 2^-7
			f32 s[8];
			// row-scaled build: this lane's 8 keys of the tile are 4 * half + {0..3} and 8 + 4 * half + {0..3}
			[[maybe_unused]] f32 const *sc = nullptr;
			if constexpr (ROW_SCALES) {
				sc = reinterpret_cast<f32 const *>(smem + at::SCALE_RING_OFFSET + k_slot * at::SCALE_TILE_BYTES) + 16 * tile + 4 * half;
				v4f const k0 = *reinterpret_cast<v4f const *>(sc), k1 = *reinterpret_cast<v4f const *>(sc + 8);
				X17_UNROLL for (u32 r = 0; r < 8; ++r) s[r] = (f32(s_acc[8 * tile + r]) * (r < 4 ? k0[r % 4] : k1[r % 4])) * temperature;
			} else if constexpr (SCALED) {
				X17_UNROLL for (u32 r = 0; r < 8; ++r) s[r] = (u2f((u32)s_acc[8 * tile + r]) - step_constants.dot_start) * scaled_temperature;
			} else {
				X17_UNROLL for (u32 r = 0; r < 8; ++r) s[r] = step_constants.dot(s_acc[8 * tile + r]) * temperature;
			}
			if constexpr (MASKED) {
				// key j is visible iff j < qi and qi - j <= wr, i.e. iff the distance qi - 1 - j, taken as an
				// unsigned number, is at most wr - 1 (a key at or behind the query wraps to a huge distance;
				// the bound is capped at 2^31 - 1 so that an unlimited window cannot meet it)
				u32 const first = qi - 1 - ((kb_begin + i) * at::KV_PER_STEP + 16 * tile + 4 * half);
				X17_UNROLL for (u32 r = 0; r < 8; ++r) {
					u32 const distance = first - (8 * (r / 4) + (r % 4));
					s[r] = distance <= vis_bound ? s[r] : -__builtin_inff();
				}
			}
			f32 tmax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(s[0], s[1]), __builtin_fmaxf(s[2], s[3])),
			                           __builtin_fmaxf(__builtin_fmaxf(s[4], s[5]), __builtin_fmaxf(s[6], s[7])));
			// cuda/attn_fwd_i8.cuh:233-256 -- rescale only when some row's max grew (both lanes of a pair hold the same m:
			// the tile's maximum exceeds it exactly when one of the two halves does)
			f32 resc = 1.0f;
			if (__any(tmax > (SCALED ? scaled_m : m))) {
				tmax = __builtin_fmaxf(tmax, partner_f32(tmax, half));
				f32 const new_m = SCALED ? __builtin_fmaxf(tmax, scaled_m) * 128.0f : __builtin_fmaxf(tmax, m);
				resc = strict::ex2<true>(m - new_m);      // exactly 1 for rows whose max did not move
				m = new_m;
				if constexpr (SCALED_SUMS) scaled_m = m * 0.0078125f;
				X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
					X17_UNROLL for (int r = 0; r < 16; ++r) o_acc[db][r] = o_acc[db][r] * resc;
				}
			}
			// :265-290 -- p = ex2(s - max) * 255 (without row scales: at 2^-8); partial sums over key quads; P = rne(p)
			f32 p[8];
			if constexpr (SCALED) {
				X17_UNROLL for (u32 r = 0; r < 8; ++r) p[r] = scaled_probability(scaled_m - s[r], step_constants);
			} else {
				X17_UNROLL for (u32 r = 0; r < 8; ++r) p[r] = strict::ex2<true>(s[r] - m) * SUM_PROB_SCALE;
			}
			sum_lo = fmaf32(sum_lo, resc, (p[0] + p[1]) + (p[2] + p[3]));
			sum_hi = fmaf32(sum_hi, resc, (p[4] + p[5]) + (p[6] + p[7]));
			v4u pp;
			if constexpr (ROW_SCALES) {
				// the numerator takes the probabilities at the value rows' relative scales
				v4f const w0 = *reinterpret_cast<v4f const *>(sc + 32), w1 = *reinterpret_cast<v4f const *>(sc + 40);
				X17_UNROLL for (u32 r = 0; r < 8; ++r) p[r] = p[r] * (r < 4 ? w0[r % 4] : w1[r % 4]);
				X17_UNROLL for (int w = 0; w < 4; ++w) pp[w] = pack_f16(__builtin_rintf(p[2 * w]), __builtin_rintf(p[2 * w + 1]));
			} else {
				X17_UNROLL for (int w = 0; w < 4; ++w) {
					pp[w] = __builtin_amdgcn_perm(f2u(p[2 * w + 1] + step_constants.round_magic), f2u(p[2 * w] + step_constants.round_magic), 0x05040100u);
				}
			}
			v8h const pfrag = __builtin_bit_cast(v8h, pp);
			// :588-605 -- O += f32(P . V) for this 16-key tile (without row scales: at 2^-24)
			X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
				v16f const zero = {0};
				v16f const pv = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_fragment(v_tile, tile, db), pfrag, zero, 0, 0, 0);
				X17_UNROLL for (int r = 0; r < 16; ++r) o_acc[db][r] = o_acc[db][r] + pv[r];
			}
		};
		u32 k_lane_off[K_SLICES];
		X17_UNROLL for (u32 sl = 0; sl < K_SLICES; ++sl) k_lane_off[sl] = at::k_chunk_offset(qlane, 2 * sl + half);

		auto compute = [&]<bool MASKED, int SLOT>(u32 i) __attribute__((always_inline)) {
			u32 const k_slot = SLOT >= 0 ? (u32)SLOT : i % at::RING;
			u32 const v_slot = SLOT >= 0 ? (u32)SLOT & 1u : i & 1u;
			u8 const *k_tile = smem + at::K_RING_OFFSET + k_slot * at::K_TILE_BYTES;
			u8 const *v_tile = smem + at::V_TILES_OFFSET + v_slot * at::V_TILE_BYTES;
			v16i s_acc = s_bias;
			X17_UNROLL for (u32 sl = 0; sl < K_SLICES; ++sl) {
				v4i kf = *reinterpret_cast<v4i const *>(k_tile + k_lane_off[sl]);
				s_acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf, qf[sl], s_acc, 0, 0, 0);
			}
			widen_next.template operator()<SLOT>(i);      // (behind the matrix instructions, whose results are not ready yet)
			if constexpr (STRICT) {
				strict_tile.template operator()<MASKED>(i, 0, s_acc, k_slot, v_tile);
				strict_tile.template operator()<MASKED>(i, 1, s_acc, k_slot, v_tile);
				return;
			}
			X17_UNROLL for (u32 tile = 0; tile < 2; ++tile) {
				f32 y[8];
				[[maybe_unused]] bool vis[8];
				f32 tmax;
				// row-scaled build: this lane's 8 keys of the tile are 4 * half + {0..3} and 8 + 4 * half + {0..3}
				[[maybe_unused]] f32 const *sc = nullptr;
				[[maybe_unused]] f32 z[8];
				if constexpr (ROW_SCALES) {
					sc = reinterpret_cast<f32 const *>(smem + at::SCALE_RING_OFFSET + k_slot * at::SCALE_TILE_BYTES) + 16 * tile + 4 * half;
					v4f const k0 = *reinterpret_cast<v4f const *>(sc), k1 = *reinterpret_cast<v4f const *>(sc + 8);
					X17_UNROLL for (u32 r = 0; r < 4; ++r) {
						z[r] = f32(s_acc[8 * tile + r]) * k0[r];
						z[4 + r] = f32(s_acc[8 * tile + 4 + r]) * k1[r];
					}
				}
				if constexpr (!MASKED && ROW_SCALES) {
					// (non-negative temperature: sgn = 1)
					X17_UNROLL for (u32 r = 0; r < 8; ++r) y[r] = z[r];
					tmax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(y[0], y[1]), __builtin_fmaxf(y[2], y[3])),
					                       __builtin_fmaxf(__builtin_fmaxf(y[4], y[5]), __builtin_fmaxf(y[6], y[7])));
				} else if constexpr (!MASKED) {
					// (positive temperature: sgn = 1; the biased scores are positive floats: their order is the order
					// of their bits as integers)
					X17_UNROLL for (u32 r = 0; r < 8; ++r) y[r] = u2f((u32)s_acc[8 * tile + r]);
					i32 const *a = reinterpret_cast<i32 const *>(&s_acc) + 8 * tile;
					auto mx = [](i32 x, i32 y) { return x > y ? x : y; };
					i32 const imax = mx(mx(mx(mx(mx(mx(mx(a[0], a[1]), a[2]), a[3]), a[4]), a[5]), a[6]), a[7]);     // four max3-type operations
					tmax = u2f((u32)imax);
				} else {
					u32 const key0 = (kb_begin + i) * at::KV_PER_STEP;
					u32 const first = qi - 1 - (key0 + 16 * tile + 4 * half);
					f32 ym[8];
					X17_UNROLL for (u32 r = 0; r < 8; ++r) {
						u32 const distance = first - (8 * (r / 4) + (r % 4));
						vis[r] = distance <= vis_bound;
						y[r] = ROW_SCALES ? z[r] * sgn : u2f((u32)s_acc[8 * tile + r]) * sgn;
						ym[r] = vis[r] ? y[r] : -__builtin_inff();
					}
					tmax = __builtin_fmaxf(__builtin_fmaxf(__builtin_fmaxf(ym[0], ym[1]), __builtin_fmaxf(ym[2], ym[3])),
					                       __builtin_fmaxf(__builtin_fmaxf(ym[4], ym[5]), __builtin_fmaxf(ym[6], ym[7])));
				}
				if (__any(tmax > ext)) {
					if constexpr (!MASKED && !ROW_SCALES) {
						tmax = u2f((u32)pair_max_i32((i32)f2u(tmax)));
					} else {
						tmax = __builtin_fmaxf(tmax, partner_f32(tmax, half));
					}
					ext = tmax > ext ? tmax : ext;
					set_subtrahend<ROW_SCALES>(ext, abs_t, mb, fine);
					lift = hw::ex2(fmaf32(ext - ext_ref, abs_t, -HEADROOM));      // (the difference is exact)
					if (__any(lift > MAX_LIFT)) {
						// O and the partial sums come down to the scale of the new maximum
						f32 const down = hw::rcp(lift) * LIFT0;
						X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
							X17_UNROLL for (int r = 0; r < 16; ++r) o_acc[db][r] = o_acc[db][r] * down;
						}
						sum_lo = sum_lo * down;
						sum_hi = sum_hi * down;
						ext_ref = ext;
						lift = LIFT0;
					}
					lift2 = v2h{(_Float16)lift, (_Float16)lift};      // round to nearest
					neg_bias2 = lift2 * v2h{(_Float16)-1024.0f, (_Float16)-1024.0f};     // exact
					sum_lift = lift * fine;
				}
				f32 p[8];
				X17_UNROLL for (u32 r = 0; r < 8; ++r) {
					f32 const arg = fmaf32(y[r], abs_t, -mb);       // lg2 of 255 * 2^(score - maximum)
					if constexpr (!MASKED) {
						p[r] = hw::ex2(arg);
					} else {
						p[r] = hw::ex2(vis[r] ? arg : -__builtin_inff());
					}
				}
				sum_lo = fmaf32((p[0] + p[1]) + (p[2] + p[3]), sum_lift, sum_lo);
				sum_hi = fmaf32((p[4] + p[5]) + (p[6] + p[7]), sum_lift, sum_hi);
				v4u pp;
				[[maybe_unused]] f32 vw[8];
				if constexpr (ROW_SCALES) {
					v4f const w0 = *reinterpret_cast<v4f const *>(sc + 32), w1 = *reinterpret_cast<v4f const *>(sc + 40);
					X17_UNROLL for (u32 r = 0; r < 4; ++r) { vw[r] = w0[r]; vw[4 + r] = w1[r]; }
				}
				X17_UNROLL for (int w = 0; w < 4; ++w) {
					f32 const f_lo = ROW_SCALES ? vw[2 * w] : fine, f_hi = ROW_SCALES ? vw[2 * w + 1] : fine;
					u32 const lo16 = f2u(fmaf32(p[2 * w], f_lo, PACK_MAGIC)), hi16 = f2u(fmaf32(p[2 * w + 1], f_hi, PACK_MAGIC));
					u32 const pair = __builtin_amdgcn_perm(hi16, lo16, 0x05040100u);           // f16 (1024 + P) twice
					pp[w] = __builtin_bit_cast(u32, __builtin_elementwise_fma(__builtin_bit_cast(v2h, pair), lift2, neg_bias2));
				}
				v8h const pfrag = __builtin_bit_cast(v8h, pp);
				X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
					o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_fragment(v_tile, tile, db), pfrag, o_acc[db], 0, 0, 0);
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

		__syncthreads();                      // previous head's tiles are no longer read
		// (every workgroup walks at least four tiles: 0 .. 3 exist)
		if (CPR == 8 || stager) {
			load_to_lds_16(smem + at::RAW_V_RING_OFFSET + stage_lds, src, stage_v_src);
			X17_UNROLL for (u32 j = 0; j < 3; ++j) {
				if constexpr (ROW_SCALES) {
					request_scales(j);
					sc_src += at::KV_PER_STEP;
				}
				load_to_lds_16(smem + at::K_RING_OFFSET + j * at::K_TILE_BYTES + stage_lds, src + j * TILE_STEP_BYTES, stage_k_src);
				load_to_lds_16(smem + at::RAW_V_RING_OFFSET + (j + 1) * at::RAW_V_TILE_BYTES + stage_lds, src + j * TILE_STEP_BYTES, stage_v_next);
			}
		}
		src += 3 * TILE_STEP_BYTES;
		if (ROW_SCALES && wave == 0) {
			__builtin_amdgcn_s_waitcnt(0x0F79);   // vmcnt(9): raw V tile 0 has landed (three loads per later tile)
		} else {
			__builtin_amdgcn_s_waitcnt(0x0F76);   // vmcnt(6): raw V tile 0 has landed
		}
		widen_v(0, 0);
		if (regular) __builtin_amdgcn_s_setreg(F32_DENORMALS, 0);      // flushed
		u32 i = 0;
		for (; i < first_active; ++i) idle_step(i);
		for (; i < first_full; ++i) step.template operator()<true, -1>(i);
		if constexpr (!STRICT) {
			// the fully visible run: single steps up to a multiple of the ring, whole rings, single steps again.  (The strict
			// build's step is four times as long, the ring arithmetic does not show in it, and the registers of the unrolled
			// form would cost it a wavefront per SIMD.)
			for (; i < diagonal && i % at::RING != 0; ++i) step.template operator()<false, -1>(i);
			static_assert(at::RING == 4 && at::PREFETCH == 3, "the run below and the requests are written out for rings of four");
			for (; i + at::RING <= diagonal && i + 2 * at::RING <= n_steps; i += at::RING) {
				step.template operator()<false, 0>(i);
				step.template operator()<false, 1>(i + 1);
				step.template operator()<false, 2>(i + 2);
				step.template operator()<false, 3>(i + 3);
			}
		}
		for (; i < diagonal; ++i) step.template operator()<false, -1>(i);
		step.template operator()<true, -1>(i);
		for (++i; i < n_steps; ++i) idle_step(i);
		if constexpr (SCALED_SUMS) __builtin_amdgcn_s_setreg(F32_DENORMALS, 3);      // kept
		__builtin_amdgcn_s_waitcnt(0x0F70);   // the last requests write LDS: they land before the tiles are reused
		// speed build: the partial sums are at the scale of the maximum HEADROOM above ext_ref's score: the common ending below
		// takes them as if that were the maximum (sgn * ext_ref - 12582912 is that extreme's dot product, exactly)
		if constexpr (!STRICT) {
			m = ROW_SCALES ? fmaf32(ext_ref * sgn, temperature, HEADROOM) : fmaf32(fmaf32(ext_ref, sgn, -DOT_BIAS), temperature, HEADROOM);
		}

		// ---- finish (cuda/attn_fwd_i8.cuh:293-351): the lane pair holds partial sums (s0, s2) and (s1, s3)
		f32 other_lo = partner_f32(sum_lo, half);
		f32 other_hi = partner_f32(sum_hi, half);
		f32 s0 = half == 0 ? sum_lo : other_lo;
		f32 s1 = half == 0 ? other_lo : sum_lo;
		f32 s2 = half == 0 ? sum_hi : other_hi;
		f32 s3 = half == 0 ? other_hi : sum_hi;
		f32 total = ((s0 + s1) + (s2 + s3)) * (1.0f / SUM_SCALE);
		if (l_out != nullptr && half == 0) {
			l_out[(size_t)head * ((size_t)gridDim.z * seq_len) + row_base + qi] = sfu::lg2(total) + m;
		}
		f32 inv = sfu::rcp(total) * (1.0f / O_SCALE);
#if X17_ATTN_ROW_SCALES
		f32 const head_out_scale = out_scale[head];
		if constexpr (OUT_BF16) {
			u16 *o_row = reinterpret_cast<u16 *>(out) + (row_base + qi) * O_STRIDE + (size_t)head * HD;
			X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
				X17_UNROLL for (int g = 0; g < 4; ++g) {
					f32 b[4];
					X17_UNROLL for (int e = 0; e < 4; ++e) b[e] = (o_acc[db][4 * g + e] * inv) * head_out_scale;
					v2u pair = {pack2_bf16_rne(b[0], b[1]), pack2_bf16_rne(b[2], b[3])};
					*reinterpret_cast<v2u *>(o_row + 32 * db + 8 * g + 4 * half) = pair;
				}
			}
			continue;
		}
		X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
			X17_UNROLL for (int r = 0; r < 16; ++r) o_acc[db][r] = (o_acc[db][r] * inv) * head_out_scale;
		}
		inv = 1.0f;          // exact: the stores below multiply by it once more
#endif
		i8 *o_row = out + (row_base + qi) * O_STRIDE + (size_t)head * HD;
		X17_UNROLL for (u32 db = 0; db < D_BLOCKS; ++db) {
			// word g of this lane = dims 32*db + 8*g + 4*half .. +3
			u32 word[4];
			X17_UNROLL for (int g = 0; g < 4; ++g) {
				if constexpr (STRICT) {
					word[g] = pack4_fixedi8(o_acc[db][4 * g] * inv, o_acc[db][4 * g + 1] * inv,
					                        o_acc[db][4 * g + 2] * inv, o_acc[db][4 * g + 3] * inv);
				} else {
					word[g] = scaled_codes(o_acc[db][4 * g], o_acc[db][4 * g + 1], o_acc[db][4 * g + 2], o_acc[db][4 * g + 3], inv);
				}
			}
			// The lane pair (lane, lane + 32) holds the 32 bytes of this block interleaved word by word; two
			// cross-half swaps give the lower lane bytes 0..15 and the upper lane bytes 16..31, so that each
			// lane writes one 16-byte vector.
			auto a = __builtin_amdgcn_permlane32_swap(word[0], word[2], false, false);
			auto b = __builtin_amdgcn_permlane32_swap(word[1], word[3], false, false);
			v4u vec = {a[0], a[1], b[0], b[1]};
			*reinterpret_cast<v4u *>(o_row + 32 * db + 16 * half) = vec;
		}
	}
}
