// attn_parts.h -- arithmetic that attention kernels share: the two forms of the forward's speed build (attn_fwd_i8.hip,
// attn_fwd_i8_narrow.hip), which have to give the same bytes, and the backward with respect to q (attn_d_q_i8.hip).
// Needs common.h, x17_device.h and attn_tile.h.
#pragma once

namespace x17 { namespace attn_parts {

constexpr f32 PROB_SCALE = 255.0f;                                  // cuda/attn_fwd_i8.cuh:206
constexpr f32 LOG2_PROB_SCALE = 7.9943534368588578f;                // lg2(255)
// Speed build (attn_fwd_i8.hip explains them): O and the sums refer to a maximum HEADROOM above the running one whenever it is
// set, the lift of new probabilities starts at LIFT0 and O comes down when it passes MAX_LIFT ((1024 + 255) * 32 stays inside
// f16); without row scales score accumulators start at the bits of DOT_BIAS
constexpr f32 HEADROOM = 12.0f, LIFT0 = 1.0f / 4096.0f, MAX_LIFT = 32.0f, DOT_BIAS = 12582912.0f;
// p + PACK_MAGIC rounds p in [0, 256) to the nearest integer P (ties to even, as rintf) and leaves
// the f16 bit pattern of 1024 + P in the low half of the sum: 12582912 = 1.5 * 2^23 has an ulp of 1 and the bits
// 0x4B400000; adding 0x6400 = 25600 puts the f16 exponent of 1024 above the eight integer bits.
constexpr f32 PACK_MAGIC = 12582912.0f + 25600.0f;

// value of lane ^ 32
X17_DEV f32 partner_f32(f32 x, u32 half) {
	u32 u = f2u(x);
	auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
	return u2f(half == 0 ? r[1] : r[0]);
}
X17_DEV i32 partner_i32(i32 x, u32 half) {
	auto r = __builtin_amdgcn_permlane32_swap((u32)x, (u32)x, false, false);
	return (i32)(half == 0 ? r[1] : r[0]);
}

// sixteen int8 (four words) -> sixteen f16 (eight words), exact: flip the sign bit (b + 128 as an unsigned byte u),
// splice u under the f16 exponent of 1024 (0x6400 | u == 1024 + u), subtract 1152; or (EIGHTHS) an eighth of each code, its real
// value: under the exponent of 128, whose last place is an eighth, less 144
template <bool EIGHTHS = false>
X17_DEV void widen16(v4u raw, u32 (&w)[8]) {
	_Float16 const less = (_Float16)(EIGHTHS ? -144.0f : -1152.0f);
	u32 const exponent = EIGHTHS ? 0x58585858u : 0x64646464u;
	v2h const bias = {less, less};
	X17_UNROLL for (int i = 0; i < 4; ++i) {
		u32 const word = raw[i] ^ 0x80808080u;
		u32 const lo = __builtin_amdgcn_perm(exponent, word, 0x04010400u);
		u32 const hi = __builtin_amdgcn_perm(exponent, word, 0x04030402u);
		w[2 * i] = __builtin_bit_cast(u32, __builtin_bit_cast(v2h, lo) + bias);
		w[2 * i + 1] = __builtin_bit_cast(u32, __builtin_bit_cast(v2h, hi) + bias);
	}
}

// Speed build: what the exponent's subtrahend mb is for the running extreme, and 2^-(what mb's rounding leaves over), close to 1
template <bool ROW_SCALES>
X17_DEV void set_subtrahend(f32 ext, f32 abs_t, f32 &mb, f32 &fine) {
	if constexpr (ROW_SCALES) {
		mb = fmaf32(ext, abs_t, -LOG2_PROB_SCALE);
		fine = 1.0f;
	} else {
		// ext * |t| as a rounded product and its exact remainder; prod - mb is exact (neighbouring floats)
		f32 const prod = ext * abs_t;
		f32 const low = fmaf32(ext, abs_t, -prod);
		mb = prod - LOG2_PROB_SCALE;
		fine = hw::ex2(-(((prod - mb) - LOG2_PROB_SCALE) + low));
	}
}

// Speed build: four outputs as FixedI8 codes.  The scaling rides in the rounding addition; clamping the rounded value gives what
// rounding the clamped one gives
X17_DEV u32 scaled_codes(f32 a, f32 b, f32 c, f32 d, f32 scale) {
	constexpr f32 MAGIC = 12582912.0f;
	f32 const x[4] = {a, b, c, d};
	u32 u[4];
	X17_UNROLL for (int e = 0; e < 4; ++e) u[e] = f2u(__builtin_amdgcn_fmed3f(fmaf32(x[e], scale, MAGIC), MAGIC - 127.0f, MAGIC + 127.0f));
	return __builtin_amdgcn_perm(u[1], u[0], 0x0c0c0400u) | __builtin_amdgcn_perm(u[3], u[2], 0x04000c0cu);
}

}} // namespace x17::attn_parts
