// gemm_parts.h -- what the GEMM kernels over 8-bit operands share: the configuration of common.h as constants, the
// writers, operand fragments and their matrix instructions, and the hand-written tile request.
//
// The including kernel declares before this header the namespace alias `gt` of its tile geometry (WAVE_M, WAVE_N: tokens
// and raw columns of a wavefront; K_STEP: bytes of K per pipeline step and per LDS row) and LANE_COLS, the number of raw
// columns a lane hands to a writer at a time.
#pragma once

namespace {

constexpr u32 K_TOTAL = X17_A_COLS;
constexpr u32 N_RAW = X17_B_ROWS;
constexpr int A_KIND = X17_A_KIND;
constexpr int B_KIND = X17_B_KIND;
constexpr int STORE = X17_STORE;

// The writers that normalise whole heads (and the fused q + kv kernel, which contains one) keep the weight rows, in blocks
// of 32, in their natural order (blocks of 16: NaturalWriters16): a lane then owns, of every 32-column block, the columns whose (column % 8) / 4 equals
// lane / 32 -- exactly two of the reference's four partial sums of squares (cuda/gemm_b8.cuh:789-801), so a head's
// sum needs one exchange between the lanes of a pair whatever its width.  Every other writer takes 64 consecutive
// columns per lane (pairs and 16-byte output vectors stay inside a lane).
constexpr bool NATURAL_COLS = X17_EPILOGUE == 3 || X17_EPILOGUE == 5 || X17_EPILOGUE == 6;

// 0: int8 MFMA, 1: fp8 MFMA, 2: f16 MFMA after widening
constexpr int MMA = (A_KIND == 0 && B_KIND == 0) ? 0 : ((A_KIND == 1 && B_KIND == 1) ? 1 : 2);
constexpr bool ACC_F32 = MMA != 0;

constexpr u32 ROW_BYTES = gt::K_STEP;                       // one LDS row = one step of K
using Acc = __attribute__((ext_vector_type(16))) int;       // raw 16 registers; reinterpreted as f32 when ACC_F32

// ------------------------------------------------------------------ epilogues
// Each receives, for ONE token row, the accumulators of LANE_COLS (64, 32 or 16, a choice of the including kernel)
// consecutive raw columns starting at raw column `n`, already converted to f32 (i32 -> f32 is the
// reference's implicit RNE cast).

// A row's packed words leave `W` at a time: sixteen bytes, or eight where a lane has no more
template <int W>
X17_DEV void store_words(u8 *dst, u32 const (&w)[W]) {
	static_assert(W == 2 || W == 4);
	if constexpr (W == 2) {
		*reinterpret_cast<v2u *>(dst) = v2u{w[0], w[1]};
	} else {
		*reinterpret_cast<v4u *>(dst) = v4u{w[0], w[1], w[2], w[3]};
	}
}
constexpr int HALF_WORDS = LANE_COLS / 8 < 4 ? LANE_COLS / 8 : 4;   // per store of a writer that halves the columns

// ScaledMatrixWriter, cuda/gemm_b8.cuh:291-339
struct ScaleEpilogue {
	static constexpr f64 SCALE = f64(X17_INP_SCALE) * f64(X17_OUT_SCALE);
	static constexpr u32 OUT_COLS = N_RAW;
	X17_DEV static void run(f32 const (&x)[LANE_COLS], u8 *c, u32 row, u32 n, void const *) {
		u8 *dst = c + (size_t)row * OUT_COLS + n;
		// (a value of its own: a factor of 1 that folds away lets the compiler start on several rows at once, and it spills)
		f32 scale = f32(SCALE);
		asm("" : "+s"(scale));
		X17_UNROLL for (int v = 0; v < LANE_COLS / 16; ++v) {
			v4u pack;
			X17_UNROLL for (int w = 0; w < 4; ++w) {
				f32 y[4];
				X17_UNROLL for (int b = 0; b < 4; ++b) y[b] = x[16 * v + 4 * w + b] * scale;
				pack[w] = pack4_store<STORE>(y[0], y[1], y[2], y[3]);
			}
			*reinterpret_cast<v4u *>(dst + 16 * v) = pack;
		}
	}
};

// GeGluMatrixWriter, cuda/gemm_b8.cuh:341-441 with math::fast::gelu, cuda/utils_core.cuh:426-448
struct GeGluEpilogue {
	static constexpr f64 I = X17_INP_SCALE;
	static constexpr f64 O = X17_OUT_SCALE;
	static constexpr f64 INP2 = I * I;
	static constexpr f64 OUT2 = INP2 * (O * O);
	static constexpr f64 KK = constexpr_sqrt(INP2);
	static constexpr f64 CK = constexpr_sqrt(INP2 * 2.0 * INV_PI);
	static constexpr f64 CK3 = 0.044715 * CK * INP2;
	static constexpr f64 Y = 0.5 * constexpr_sqrt(OUT2 * 1.0) * KK;
	static constexpr u32 OUT_COLS = N_RAW / 2;

	X17_DEV static f32 gate(f32 x) {
		f32 x2 = x * x;
		f32 s = fmaf32(f32(CK3) * x, x2, f32(CK) * x);
		f32 t = sfu::tanh(s);
		return fmaf32(f32(Y) * x, t, f32(Y) * x);
	}
	// gate(g) * v.  The speed build uses 1 + tanh(s) = 2 / (1 + 2^(-2 s lg e)) and folds the constants:
	// g * v / (c + c * 2^(g * (A1 + A3 g^2))), c = 1 / (2 Y) -- two transcendentals and seven plain
	// operations; an overflowing exponential gives +inf and a quotient of zero, the right limit.
	static constexpr f64 LOG2E = 1.4426950408889634;
	X17_DEV static f32 gated(f32 g, f32 v) {
		if constexpr (X17_STRICT_MATH != 0) {
			return gate(g) * v;
		} else {
			f32 g2 = g * g;
			f32 t = fmaf32(g2, f32(-2.0 * LOG2E * CK3), f32(-2.0 * LOG2E * CK));
			f32 e = hw::ex2(t * g);
			f32 d = fmaf32(e, f32(0.5 / Y), f32(0.5 / Y));
			return (g * v) * hw::rcp(d);
		}
	}
	X17_DEV static void run(f32 const (&x)[LANE_COLS], u8 *c, u32 row, u32 n, void const *) {
		u8 *dst = c + (size_t)row * OUT_COLS + n / 2;
		X17_UNROLL for (int v = 0; v < LANE_COLS / (8 * HALF_WORDS); ++v) {
			u32 pack[HALF_WORDS];
			X17_UNROLL for (int w = 0; w < HALF_WORDS; ++w) {
				f32 y[4];
				X17_UNROLL for (int b = 0; b < 4; ++b) {
					int j = 4 * (HALF_WORDS * v + w) + b;
					y[b] = gated(x[2 * j], x[2 * j + 1]);
				}
				pack[w] = pack4_store<STORE>(y[0], y[1], y[2], y[3]);
			}
			store_words(dst + 4 * HALF_WORDS * v, pack);
		}
	}
};

// ResidualMatrixWriter, cuda/gemm_b8.cuh:443-622; sigmoid_base4 / imprecise_softplus_base4,
// cuda/utils_core.cuh:397-405, 468-483
struct ResidualEpilogue {
	static constexpr f64 I = X17_INP_SCALE;
	static constexpr f64 O = X17_OUT_SCALE;
	static constexpr f64 SG_HALF = 0.5 * (1.0 / 8.0);
	static constexpr f64 SG_IN = LN2 * (-I);
	static constexpr f64 SP_INP = I;
	static constexpr f64 SP_OUT = I * O;
	static constexpr f32 SP_INP_SCALE = f32(SP_INP * 2.0);
	static constexpr f32 SP_OUT_SCALE = f32(SP_OUT / 2.0);
	static constexpr f32 SP_LINE = f32(SP_INP * SP_OUT);
	static constexpr u32 OUT_COLS = N_RAW / 2;

	X17_DEV static f32 mix(f32 g, f32 v, f32 r) {
		if constexpr (X17_STRICT_MATH == 0) {
			// Speed build: both weights from one exponential.  With u = 2 I g and E = 2^-|u|:
			//   1 + tanh(-I ln2 g) = 2 / (1 + 2^u) = 2 (u >= 0 ? E : 1) / (1 + E)       -> old_w
			//   lg2(1 + 2^-|u|)    = lg2(1 + E)                                          -> new_w
			// three transcendentals (ex2, rcp, lg2) instead of four.
			f32 const u = g * SP_INP_SCALE;
			f32 const e = hw::ex2(-__builtin_fabsf(u));
			f32 const d = 1.0f + e;
			f32 const old_w = (f32(2.0 * SG_HALF) * hw::rcp(d)) * (u >= 0.0f ? e : 1.0f);
			f32 line = __builtin_fmaxf(0.0f, g);
			if constexpr (SP_LINE != 1.0f) {
				line = line * SP_LINE;
			}
			f32 const new_w = fmaf32(hw::lg2(d), SP_OUT_SCALE, line);
			return fmaf32(new_w, v, old_w * r);
		}
		f32 old_w = fmaf32(f32(SG_HALF), sfu::tanh(f32(SG_IN) * g), f32(SG_HALF));
		f32 line = __builtin_fmaxf(0.0f, g);
		if constexpr (SP_LINE != 1.0f) {
			line = line * SP_LINE;
		}
		f32 new_w = fmaf32(sfu::lg2(1.0f + sfu::ex2(-__builtin_fabsf(g * SP_INP_SCALE))), SP_OUT_SCALE, line);
		return fmaf32(new_w, v, old_w * r);
	}
	X17_DEV static void run(f32 const (&x)[LANE_COLS], u8 *c, u32 row, u32 n, void const *extra) {
		size_t off = (size_t)row * OUT_COLS + n / 2;
		i8 const *res = reinterpret_cast<i8 const *>(extra) + off;
		u8 *dst = c + off;
		X17_UNROLL for (int v = 0; v < LANE_COLS / (8 * HALF_WORDS); ++v) {
			using Words = __attribute__((ext_vector_type(HALF_WORDS))) u32;
			Words const rv = *reinterpret_cast<Words const *>(res + 4 * HALF_WORDS * v);
			u32 pack[HALF_WORDS];
			X17_UNROLL for (int w = 0; w < HALF_WORDS; ++w) {
				f32 y[4];
				X17_UNROLL for (int b = 0; b < 4; ++b) {
					int j = 4 * (HALF_WORDS * v + w) + b;
					f32 r = f32((i32)(i8)((rv[w] >> (8 * b)) & 0xFFu));
					y[b] = mix(x[2 * j], x[2 * j + 1], r);
				}
				pack[w] = pack4_store<STORE>(y[0], y[1], y[2], y[3]);
			}
			store_words(dst + 4 * HALF_WORDS * v, pack);
		}
	}
};

// Dequantising writer: per-row (token) and per-column (output channel) f32 scales, bf16 output, optional
// GeGLU over column pairs.  The reference folds its scales into compile-time constants; this is the
// run-time-scale superset for symmetric per-row / per-channel int8 quantisation (bf16 store precedent:
// cuda/gemm_b16.cuh:264-294).  t = (x * row_scale) * col_scale, two f32 multiplies in that order.
#if X17_EPILOGUE == 4
struct DequantEpilogue {
	static constexpr bool GEGLU = X17_DEQ_GEGLU != 0;
	static constexpr u32 OUT_COLS = GEGLU ? N_RAW / 2 : N_RAW;
	X17_DEV static void run(f32 const (&x)[LANE_COLS], u8 *c, u32 row, u32 n, f32 const *row_scale, f32 const *col_scale) {
		f32 const rs = row_scale[row];
		f32 t[LANE_COLS];
		X17_UNROLL for (int v = 0; v < LANE_COLS / 4; ++v) {
			v4f cs = *reinterpret_cast<v4f const *>(col_scale + n + 4 * v);
			X17_UNROLL for (int i = 0; i < 4; ++i) t[4 * v + i] = (x[4 * v + i] * rs) * cs[i];
		}
		if constexpr (GEGLU) {
			u8 *dst = c + ((size_t)row * OUT_COLS + n / 2) * 2;
			X17_UNROLL for (int v = 0; v < LANE_COLS / 16; ++v) {
				u32 pack[4];
				X17_UNROLL for (int w = 0; w < 4; ++w) {
					int j = 8 * v + 2 * w;
					pack[w] = pack2_bf16_rne(GeGluEpilogue::gated(t[2 * j], t[2 * j + 1]), GeGluEpilogue::gated(t[2 * j + 2], t[2 * j + 3]));
				}
				store_words(dst + 16 * v, pack);
			}
		} else {
			u8 *dst = c + ((size_t)row * OUT_COLS + n) * 2;
			X17_UNROLL for (int v = 0; v < LANE_COLS / 8; ++v) {
				u32 pack[4];
				X17_UNROLL for (int w = 0; w < 4; ++w) {
					int j = 8 * v + 2 * w;
					pack[w] = pack2_bf16_rne(t[j], t[j + 1]);
				}
				store_words(dst + 16 * v, pack);
			}
		}
	}
};
#endif

// ---- writers over the natural column order (l2norm, qnorm and the fused q + kv kernel).
// For ONE token row a lane holds x[16 * b + r] = raw column 32 * b + 8 * (r / 4) + 4 * (lane / 32) + r % 4 of its
// wave's 128 columns (b = 32-column block, r = accumulator register).
#if X17_EPILOGUE == 3 || X17_EPILOGUE == 5 || X17_EPILOGUE == 6
static_assert(LANE_COLS == 64 || LANE_COLS == 32, "the head-normalising writers are written for 128-column waves");
constexpr u32 HEAD_DIM = X17_HEAD_DIM;
static_assert(HEAD_DIM == 32 || HEAD_DIM == 64 || HEAD_DIM == 128, "head_dim must be 32, 64 or 128");
struct NaturalWriters {
	static constexpr f32 EPS = f32(f64(X17_EPS));
	static constexpr f32 HEAD_SCALE = f32(f64(X17_HEAD_SCALE));
	static constexpr int HB = HEAD_DIM / 32;                    // 32-column blocks per head

	// value of lane ^ 32
	X17_DEV static f32 partner(f32 v, u32 half) {
		u32 const u = f2u(v);
		auto const r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
		return u2f(half == 0 ? r[1] : r[0]);
	}
	// The lane pair (lane, lane + 32) holds the 32 output bytes of a block interleaved word by word (word g of a lane
	// = columns 8 g + 4 half .. + 3); two cross-half swaps give the lower lane bytes 0..15 and the upper lane bytes
	// 16..31, so that each lane writes one 16-byte vector.
	X17_DEV static void store_block(u8 *block, u32 const (&w)[4], u32 half) {
		auto const a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
		auto const b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
		*reinterpret_cast<v4u *>(block + 16 * half) = v4u{a[0], a[1], b[0], b[1]};
	}
	// kv_helpers::l2_norm, cuda/gemm_b8.cuh:767-830: the sum of squares of the head made of blocks [B0, B0 + HB).
	// The reference's partial sum q owns the columns with (column % 8) / 2 == q in increasing order; the lower lane
	// of a pair runs the chains of q = 0 and 1, the upper lane those of 2 and 3, total (s0 + s1) + (s2 + s3).
	template <int B0>
	X17_DEV static f32 head_scale(f32 const (&x)[64], u32 half) {
		f32 p0 = 0.0f, p1 = 0.0f;
		X17_UNROLL for (int b = B0; b < B0 + HB; ++b) {
			X17_UNROLL for (int g = 0; g < 4; ++g) {
				p0 = fmaf32(x[16 * b + 4 * g], x[16 * b + 4 * g], p0);
				p0 = fmaf32(x[16 * b + 4 * g + 1], x[16 * b + 4 * g + 1], p0);
				p1 = fmaf32(x[16 * b + 4 * g + 2], x[16 * b + 4 * g + 2], p1);
				p1 = fmaf32(x[16 * b + 4 * g + 3], x[16 * b + 4 * g + 3], p1);
			}
		}
		f32 const mine = p0 + p1;
		f32 const other = partner(mine, half);
		f32 const total = half == 0 ? mine + other : other + mine;
		return strict::rsq(total + EPS) * HEAD_SCALE;
	}
	// block b of the row times `scale` (and, with learned scales, times the bf16 scale of each column, in that order:
	// cuda/gemm_b8.cuh:819-820) -> FixedI8, 16 bytes per lane.  `dst` and `dyn` point at the wave's first column.
	template <bool DYN>
	X17_DEV static void emit_block(f32 const (&x)[64], int b, f32 scale, u8 *dst, u16 const *dyn, u32 half) {
		u32 w[4];
		X17_UNROLL for (int g = 0; g < 4; ++g) {
			f32 y[4];
			X17_UNROLL for (int e = 0; e < 4; ++e) y[e] = x[16 * b + 4 * g + e] * scale;
			if constexpr (DYN) {
				v2u const d = *reinterpret_cast<v2u const *>(dyn + 32 * b + 8 * g + 4 * half);
				y[0] = y[0] * u2f(d[0] << 16);
				y[1] = y[1] * u2f(d[0] & 0xFFFF0000u);
				y[2] = y[2] * u2f(d[1] << 16);
				y[3] = y[3] * u2f(d[1] & 0xFFFF0000u);
				// The old writer hands its f32 values to a base writer built with SCALE = 1 / sqrt(MODEL_DIM)
				// (cuda/qkvg_fwd_i8.cuh:151-159); that base class is gone from the tree, and the live scaled writer's f32
				// overload multiplies by its SCALE unless it is 1 (cuda/gemm_b8.cuh:307-324).  X17_INP_SCALE carries that
				// factor (1.0: stored as is).
				if constexpr (f32(f64(X17_INP_SCALE)) != 1.0f) {
					X17_UNROLL for (int e = 0; e < 4; ++e) y[e] = y[e] * f32(f64(X17_INP_SCALE));
				}
			}
			w[g] = pack4_fixedi8(y[0], y[1], y[2], y[3]);
		}
		store_block(dst + 32 * b, w, half);
	}
#if X17_EPILOGUE == 3 || X17_EPILOGUE == 6
	// L2NormMatrixWriter, cuda/gemm_b8.cuh:861-949: per head the columns are [K (hd) | V (hd)]; K is normalised,
	// V only scaled, rrms[row, head] = the K scale.  `col0` = the wave's first raw column of the kv matrix.
	static constexpr f32 SEP_SCALE = f32(f64(X17_SEP_SCALE));
	X17_DEV static void l2norm_row(f32 const (&x)[64], u8 *c, f32 *rrms, u32 row, u32 col0, u32 kv_cols, u32 half) {
		u8 *dst = c + (size_t)row * kv_cols + col0;
		f32 *rr = rrms + (size_t)row * (kv_cols / (2 * HEAD_DIM));
		if constexpr (HEAD_DIM == 32) {
			f32 const scale0 = head_scale<0>(x, half);
			emit_block<false>(x, 0, scale0, dst, nullptr, half);
			emit_block<false>(x, 1, SEP_SCALE, dst, nullptr, half);
			f32 const scale1 = head_scale<2>(x, half);
			emit_block<false>(x, 2, scale1, dst, nullptr, half);
			emit_block<false>(x, 3, SEP_SCALE, dst, nullptr, half);
			if (half == 0) {
				rr[col0 / 64] = scale0;
				rr[col0 / 64 + 1] = scale1;
			}
		} else if constexpr (HEAD_DIM == 64) {
			f32 const scale = head_scale<0>(x, half);
			emit_block<false>(x, 0, scale, dst, nullptr, half);
			emit_block<false>(x, 1, scale, dst, nullptr, half);
			emit_block<false>(x, 2, SEP_SCALE, dst, nullptr, half);
			emit_block<false>(x, 3, SEP_SCALE, dst, nullptr, half);
			if (half == 0) rr[col0 / 128] = scale;
		} else {
			// the wave's 128 columns are the K half or the V half of one head
			if ((col0 / 128) % 2 == 0) {
				f32 const scale = head_scale<0>(x, half);
				X17_UNROLL for (int b = 0; b < 4; ++b) emit_block<false>(x, b, scale, dst, nullptr, half);
				if (half == 0) rr[col0 / 256] = scale;
			} else {
				X17_UNROLL for (int b = 0; b < 4; ++b) emit_block<false>(x, b, SEP_SCALE, dst, nullptr, half);
			}
		}
	}
#endif
#if X17_EPILOGUE == 5
	// QMatrixWriter, cuda/qkvg_fwd_i8.cuh:145-219: every head_dim columns are one normalised head
	template <int B0>
	X17_DEV static void qnorm_heads(f32 const (&x)[64], u8 *dst, u16 const *dyn, u32 half) {
		if constexpr (B0 < 4) {
			f32 const scale = head_scale<B0>(x, half);
			X17_UNROLL for (int b = B0; b < B0 + HB; ++b) emit_block<true>(x, b, scale, dst, dyn, half);
			qnorm_heads<B0 + HB>(x, dst, dyn, half);
		}
	}
	X17_DEV static void qnorm_row(f32 const (&x)[64], u8 *c, u16 const *dyn, u32 row, u32 col0, u32 half) {
		qnorm_heads<0>(x, c + (size_t)row * N_RAW + col0, dyn + col0, half);
	}
#endif
#if X17_EPILOGUE == 6
	// ScaledMatrixWriter (cuda/gemm_b8.cuh:291-339) over the natural column order, for the q columns
	X17_DEV static void scale_row(f32 const (&x)[64], u8 *c, u32 row, u32 col0, u32 q_cols, u32 half) {
		u8 *dst = c + (size_t)row * q_cols + col0;
		X17_UNROLL for (int b = 0; b < 4; ++b) emit_block<false>(x, b, f32(f64(X17_Q_SCALE)), dst, nullptr, half);
	}
	X17_DEV static void qkv_row(f32 const (&x)[64], u8 *c, u8 *c_kv, f32 *rrms, u32 row, u32 col0, u32 half) {
		constexpr u32 Q_COLS = X17_Q_COLS;
		if (col0 < Q_COLS) {
			scale_row(x, c, row, col0, Q_COLS, half);
		} else {
			l2norm_row(x, c_kv, rrms, row, col0 - Q_COLS, N_RAW - Q_COLS, half);
		}
	}
#endif
};

// The same writers for blocks of 16 x 16: lane group g (lane / 16) holds x[4 * bn + r] = raw column 16 * bn + 8 * (r / 2) + 2 * g + r % 2 of
// its token row, which is the reference's partial sum g of every head, in its order.
struct NaturalWriters16 {
	static constexpr int HB = HEAD_DIM / 32;
	// (a scale in a register of its own: see ScaleEpilogue)
	X17_DEV static f32 opaque(f32 v) {
		asm("" : "+s"(v));
		return v;
	}
	// the sum over the four lanes of a row: (0 + 1) + (2 + 3)
	X17_DEV static f32 over_groups(f32 v) {
		auto const a = __builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false);
		f32 const pair = u2f(a[0]) + u2f(a[1]);
		auto const b = __builtin_amdgcn_permlane32_swap(f2u(pair), f2u(pair), false, false);
		return u2f(b[0]) + u2f(b[1]);
	}
	// kv_helpers::l2_norm, cuda/gemm_b8.cuh:767-830, of the head made of 32-column blocks [B0, B0 + HB)
	template <int B0>
	X17_DEV static f32 head_scale(f32 const (&x)[32]) {
		f32 p = 0.0f;
		X17_UNROLL for (int i = 8 * B0; i < 8 * (B0 + HB); ++i) p = fmaf32(x[i], x[i], p);
		return strict::rsq(over_groups(p) + NaturalWriters::EPS) * NaturalWriters::HEAD_SCALE;
	}
	// The row times `scale` per 32-column block (and, with learned scales, as in NaturalWriters::emit_block) -> FixedI8.  A lane's words hold
	// two columns of every eight: an exchange of words between the four lanes gives each the 32 bytes of one block.
	template <bool DYN>
	X17_DEV static void emit(f32 const (&x)[32], f32 const (&scale)[4], u8 *dst, u16 const *dyn, u32 group) {
		u32 w[8];
		X17_UNROLL for (int bn = 0; bn < 8; ++bn) {
			f32 y[4];
			X17_UNROLL for (int e = 0; e < 4; ++e) y[e] = x[4 * bn + e] * scale[bn / 2];
			if constexpr (DYN) {
				X17_UNROLL for (int h = 0; h < 2; ++h) {
					u32 const d = *reinterpret_cast<u32 const *>(dyn + 16 * bn + 8 * h + 2 * group);
					y[2 * h] = y[2 * h] * u2f(d << 16);
					y[2 * h + 1] = y[2 * h + 1] * u2f(d & 0xFFFF0000u);
				}
				if constexpr (f32(f64(X17_INP_SCALE)) != 1.0f) {
					X17_UNROLL for (int e = 0; e < 4; ++e) y[e] = y[e] * f32(f64(X17_INP_SCALE));
				}
			}
			w[bn] = pack4_fixedi8(y[0], y[1], y[2], y[3]);
		}
		X17_UNROLL for (int e = 0; e < 2; ++e) {
			auto const even = __builtin_amdgcn_permlane32_swap(w[e], w[4 + e], false, false);
			auto const odd = __builtin_amdgcn_permlane32_swap(w[2 + e], w[6 + e], false, false);
			auto const t01 = __builtin_amdgcn_permlane16_swap(even[0], odd[0], false, false);      // word 2 * group + e of lane groups 0, 1
			auto const t23 = __builtin_amdgcn_permlane16_swap(even[1], odd[1], false, false);      // of lane groups 2, 3
			*reinterpret_cast<v4u *>(dst + 32 * group + 16 * e) = v4u{
				__builtin_amdgcn_perm(t01[1], t01[0], 0x05040100u), __builtin_amdgcn_perm(t23[1], t23[0], 0x05040100u),
				__builtin_amdgcn_perm(t01[1], t01[0], 0x07060302u), __builtin_amdgcn_perm(t23[1], t23[0], 0x07060302u)};
		}
	}
#if X17_EPILOGUE == 3 || X17_EPILOGUE == 6
	// the scales of the K heads among the columns, whose first is column col0 of the kv matrix
	X17_DEV static void key_scales(f32 const (&x)[32], f32 (&scale)[4], f32 *rrms, u32 row, u32 col0, u32 kv_cols, u32 group) {
		f32 *rr = rrms + (size_t)row * (kv_cols / (2 * HEAD_DIM));
		if constexpr (HEAD_DIM == 32) {
			scale[0] = head_scale<0>(x);
			scale[2] = head_scale<2>(x);
			if (group == 0) {
				rr[col0 / 64] = scale[0];
				rr[col0 / 64 + 1] = scale[2];
			}
		} else if (HEAD_DIM == 64 || (col0 / 128) % 2 == 0) {       // (head_dim 128: the wave's columns are K or V of one head)
			scale[0] = head_scale<0>(x);
			X17_UNROLL for (int b = 1; b < HB; ++b) scale[b] = scale[0];
			if (group == 0) rr[col0 / (2 * HEAD_DIM)] = scale[0];
		}
	}
	X17_DEV static void l2norm_row(f32 const (&x)[32], u8 *c, f32 *rrms, u32 row, u32 col0, u32 kv_cols, u32 group) {
		f32 const sep = opaque(NaturalWriters::SEP_SCALE);
		f32 scale[4] = {sep, sep, sep, sep};
		key_scales(x, scale, rrms, row, col0, kv_cols, group);
		emit<false>(x, scale, c + (size_t)row * kv_cols + col0, nullptr, group);
	}
#endif
#if X17_EPILOGUE == 5
	X17_DEV static void qnorm_row(f32 const (&x)[32], u8 *c, u16 const *dyn, u32 row, u32 col0, u32 group) {
		f32 scale[4];
		scale[0] = head_scale<0>(x);
		if constexpr (HB == 4) {
			scale[1] = scale[2] = scale[3] = scale[0];
		} else {
			scale[2] = head_scale<2>(x);
			if constexpr (HB == 2) {
				scale[1] = scale[0];
				scale[3] = scale[2];
			} else {
				scale[1] = head_scale<1>(x);
				scale[3] = head_scale<3>(x);
			}
		}
		emit<true>(x, scale, c + (size_t)row * N_RAW + col0, dyn + col0, group);
	}
#endif
#if X17_EPILOGUE == 6
	// q columns or kv columns of the fused kernel: one copy of the writer (two spill)
	X17_DEV static void qkv_row(f32 const (&x)[32], u8 *c, u8 *c_kv, f32 *rrms, u32 row, u32 col0, u32 group) {
		constexpr u32 Q_COLS = X17_Q_COLS, KV_COLS = N_RAW - Q_COLS;
		bool const q = col0 < Q_COLS;
		f32 const all = opaque(q ? f32(f64(X17_Q_SCALE)) : NaturalWriters::SEP_SCALE);
		f32 scale[4] = {all, all, all, all};
		if (!q) key_scales(x, scale, rrms, row, col0 - Q_COLS, KV_COLS, group);
		emit<false>(x, scale, q ? c + (size_t)row * Q_COLS + col0 : c_kv + (size_t)row * KV_COLS + (col0 - Q_COLS), nullptr, group);
	}
#endif
};
#endif

// ------------------------------------------------------------------ requests, fragments, matrix instructions

// One 16-byte-per-lane direct-to-LDS load: LDS destination in M0 (wave-uniform; lane l lands 16 * l bytes further),
// global source = uniform 64-bit base in scalar registers + a 32-bit offset per lane.  Written out because the
// compiler's own selection forms a 64-bit address per lane in ONE vector register pair for every load: a 64-bit
// vector add per load, each waiting until the previous load has read the pair (measured 3-5 % of the kernel).
X17_DEV void load_to_lds_16(u8 *lds_uniform, u8 const *src_uniform, u32 lane_offset) {
	// (gfx9 family: a scalar write of M0 needs one wait state before a direct-to-LDS load reads it; the compiler
	// inserts it for its own loads and cannot see into this string)
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
	             :: "s"((u32)(size_t)X17_LDS_PTR(lds_uniform)), "v"(lane_offset), "s"(src_uniform) : "memory", "m0");
}

// s_waitcnt vmcnt(N) with the other counters left alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14)
template <u32 N>
X17_DEV void wait_vmcnt() {
	static_assert(N < 64);
	__builtin_amdgcn_s_waitcnt((N & 15u) | ((N >> 4) << 14) | 0x0F70u);
}
// One 16-byte operand chunk: row `row_off` (bytes), logical chunk `kc` of the row.
X17_DEV v4i lds_chunk(u8 const *tile, u32 row_off, u32 kc, u32 swz) {
	return *reinterpret_cast<v4i const *>(tile + row_off + ((kc ^ swz) << 4));
}

// Eight 8-bit values (two registers) -> eight f16, exact for both kinds.
//   e4m3: the gfx950 packed fp8 -> f16 conversion (scale 1).  It reads OCP e4m3; the codes the
//         reference's encoder produces (no subnormals, no NaN, no -0) mean the same in both.
//   int8: flip the sign bit (b + 128 as an unsigned byte u), splice u under the f16 exponent of 1024
//         (0x6400 | u == 1024 + u) and subtract 1152 -- five instructions per four bytes.
[[maybe_unused]] X17_DEV v8h widen8(u32 lo, u32 hi, int kind) {
	v2h p[4];
	if (kind == 1) {
		p[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false);
		p[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true);
		p[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false);
		p[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true);
	} else {
		v2h const bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
		u32 w[2] = {lo ^ 0x80808080u, hi ^ 0x80808080u};
		X17_UNROLL for (int i = 0; i < 2; ++i) {
			u32 l = __builtin_amdgcn_perm(0x64646464u, w[i], 0x04010400u);
			u32 h = __builtin_amdgcn_perm(0x64646464u, w[i], 0x04030402u);
			p[2 * i] = __builtin_bit_cast(v2h, l) + bias;
			p[2 * i + 1] = __builtin_bit_cast(v2h, h) + bias;
		}
	}
	return v8h{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// Operand fragments of one K slice (what one round of 4 x BM MFMA blocks consumes) and the MFMAs
// themselves, per arithmetic: 32 bytes of K for int8 and for the f16-widened mix, 64 for e4m3.
constexpr u32 SLICE_BYTES = MMA == 1 ? 64 : 32;
constexpr u32 SLICES = gt::K_STEP / SLICE_BYTES;
constexpr u32 CHUNKS_PER_FRAG = SLICE_BYTES / 32;           // 16-byte chunks a lane fetches per operand row

constexpr int BM = gt::WAVE_M / 32;                         // 32-token MFMA blocks per wave
constexpr int BN = gt::WAVE_N / 32;                         // 32-column MFMA blocks per wave

struct Frags {
	v4i w[BN][CHUNKS_PER_FRAG];
	v4i x[BM][CHUNKS_PER_FRAG];
};

X17_DEV void load_frags(Frags &f, u8 const *w_tile, u8 const *x_tile, u32 s, u32 half, u32 swz) {
	// in the order the MFMAs of a slice want them: w0, every x, then the other w
	u32 const kc0 = CHUNKS_PER_FRAG * (2 * s + half);
	X17_UNROLL for (u32 c = 0; c < CHUNKS_PER_FRAG; ++c) f.w[0][c] = lds_chunk(w_tile, 0, kc0 + c, swz);
	X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
		X17_UNROLL for (u32 c = 0; c < CHUNKS_PER_FRAG; ++c) f.x[bm][c] = lds_chunk(x_tile, bm * 32 * ROW_BYTES, kc0 + c, swz);
	}
	X17_UNROLL for (int bn = 1; bn < BN; ++bn) {
		X17_UNROLL for (u32 c = 0; c < CHUNKS_PER_FRAG; ++c) f.w[bn][c] = lds_chunk(w_tile, bn * 32 * ROW_BYTES, kc0 + c, swz);
	}
}

X17_DEV void mma_slice(Frags const &f, Acc (&acc)[BN][BM]) {
	if constexpr (MMA == 0) {
		X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
			X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
				acc[bn][bm] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.w[bn][0], f.x[bm][0], acc[bn][bm], 0, 0, 0);
			}
		}
	} else if constexpr (MMA == 1) {
		v8i wf[BN], xf[BM];
		X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
			v4i l = f.w[bn][0], h = f.w[bn][CHUNKS_PER_FRAG - 1];
			wf[bn] = v8i{l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
		}
		X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
			v4i l = f.x[bm][0], h = f.x[bm][CHUNKS_PER_FRAG - 1];
			xf[bm] = v8i{l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
		}
		X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
			X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
				v16f r = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
					wf[bn], xf[bm], __builtin_bit_cast(v16f, acc[bn][bm]), 0, 0, 0, 0, 0, 0);
				acc[bn][bm] = __builtin_bit_cast(Acc, r);
			}
		}
	} else {
		X17_UNROLL for (int h = 0; h < 2; ++h) {                // two f16 MFMAs of K = 16
			v8h wf[BN], xf[BM];
			X17_UNROLL for (int bn = 0; bn < BN; ++bn) wf[bn] = widen8(f.w[bn][0][2 * h], f.w[bn][0][2 * h + 1], B_KIND);
			X17_UNROLL for (int bm = 0; bm < BM; ++bm) xf[bm] = widen8(f.x[bm][0][2 * h], f.x[bm][0][2 * h + 1], A_KIND);
			X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
				X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
					v16f r = __builtin_amdgcn_mfma_f32_32x32x16_f16(
						wf[bn], xf[bm], __builtin_bit_cast(v16f, acc[bn][bm]), 0, 0, 0);
					acc[bn][bm] = __builtin_bit_cast(Acc, r);
				}
			}
		}
	}
}

} // namespace
