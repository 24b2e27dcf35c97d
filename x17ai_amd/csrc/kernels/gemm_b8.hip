// gemm_b8.hip -- C[M, N] = epilogue(A[M, K] . B[N_raw, K]^T) for 8-bit operands on gfx950.
//
// Replaces the reference's b8::Gemm (cuda/gemm_b8.cuh:624-755: i8 x i8 -> i32) and b16::Gemm
// (cuda/gemm_b16.cuh:436-567: any e4m3 operand, f32 accumulate) together with their four fused
// writers (Scaled :291-339, GeGlu :341-441, Residual :443-622, L2Norm :861-949).  The kernel
// entry and its parameters follow templates/basic_gemm/kernel.cu:9-32.
//
// Design, MI355X-first (nothing here is derived from the SM80 kernel):
//   * One workgroup = a 256 (tokens) x 256 (raw columns) output tile, by default 8 wavefronts of
//     64 x 128 (two per SIMD); gemm_tile.h can also build 8 wavefronts of 128 x 64 or 4 wavefronts of 128 x 128
//     (256 accumulator registers per lane, one wavefront per SIMD: what the host picks whenever an operand is e4m3).
//   * The WEIGHTS are the MFMA "A" operand and the TOKENS the "B" operand, i.e. the matrix
//     cores compute C^T.  A lane then owns one token and, per MFMA block, 4 output columns (16 of a 32 x 32 block);
//     weight rows are permuted on their way into LDS so that those are 32 (64)
//     CONSECUTIVE columns across the blocks.  Gate/value pairs, whole K|V heads and 16-byte output
//     vectors all live inside one lane: the epilogues need no cross-lane shuffles (the SM80
//     code needs a 4x4 shuffle transpose per 32x32 tile, cuda/gemm_b8.cuh:411, 570, 592).
//   * Global -> LDS goes through the gfx950 16-byte direct-to-LDS load (no register staging) into
//     rings of LDS tiles (gemm_tile.h: K_STEP bytes of K per step; by default three token tiles and two
//     weight tiles of 32 KB, which is all 160 KB of a compute unit), one barrier per step;
//     16-byte chunks are XOR-swizzled so that ds_read_b128 is conflict-free.  In the int8 and e4m3 kernels the
//     issue order of a K step is pinned: each MFMA is followed by its share of the LDS reads and tile requests
//     (and, in the mixed arithmetic, of the next round's conversions to f16).
//   * int8: v_mfma_i32_16x16x64_i8.  e4m3 x e4m3: v_mfma_f32_16x16x128_f8f6f4 (the 32 x 32 forms of both with fewer than three
//     K steps, for e4m3 below K = 2048 and in the kv writer at head_dim 32: gemm_tile.h).  Mixed
//     e4m3 x int8: both widened exactly to f16 in registers, v_mfma_f32_32x32x16_f16
//     (int8 codes need 7 significand bits, e4m3 has 4; every e4m3 value is a normal f16).
//   * Workgroup ids are remapped so that each XCD (own L2) works on a compact block of tiles.
//
// common.h (generated per kernel by the host-side kernel builder) provides:
//   X17_A_COLS (K), X17_B_ROWS (N_raw), X17_A_KIND / X17_B_KIND (0 = int8, 1 = e4m3),
//   X17_EPILOGUE (0 scale, 1 geglu, 2 residual, 3 l2norm, 4 dequant, 5 qnorm, 6 fused q + kv), X17_STORE
//   (0 FixedI8, 1 e4m3; dequant always stores bf16), X17_DEQ_GEGLU (dequant only: 0 plain, 1 GeGLU over column
//   pairs), X17_INP_SCALE, X17_OUT_SCALE, for l2norm / qnorm / fused X17_HEAD_DIM, X17_EPS, X17_HEAD_SCALE,
//   X17_SEP_SCALE (doubles), for fused X17_Q_COLS (the first raw columns belong to q) and X17_Q_SCALE,
//   X17_STRICT_MATH.
//
// Epilogue 5 (qnorm) is the reference's older Q writer with learned scales (cuda/qkvg_fwd_i8.cuh:145-219; the
// hook is still in the live header: kv_helpers::l2_norm<USE_DYN_SCALE>, cuda/gemm_b8.cuh:761-824): every head_dim
// raw columns are L2-normalised like the K halves of epilogue 3 and multiplied by a bf16 scale per column.
// Epilogue 6 computes the q and the kv projection of src/main.rs:387-493 in ONE launch over the same token tiles
// (raw columns [0, X17_Q_COLS) from the q weights through the Scale writer into q, the rest from the kv weights
// through the L2-norm writer into kv and rrms): the writer is chosen per output tile, x is read once.

#include "common.h"
#include "x17_device.h"
#include "gemm_tile.h"

using namespace x17;
namespace gt = x17::gemm_tile;
namespace {
constexpr int LANE_COLS = gt::WAVE_N / gt::GROUPS;          // consecutive raw columns a lane ends up with
}
#include "gemm_parts.h"

// The compiler fully unrolls a K loop of up to 8 steps and then runs out of registers; longer loops it
// unrolls by a small factor on its own, which measures 5 % faster than a rolled loop.
#if (X17_A_COLS / X17_GEMM_K_STEP) <= 8
#define X17_K_LOOP_PRAGMA _Pragma("clang loop unroll(disable)")
#else
#define X17_K_LOOP_PRAGMA
#endif

namespace {

static_assert(K_TOTAL % gt::K_STEP == 0, "K must be a multiple of 128");
static_assert((gt::max_offset_row(NATURAL_COLS) + 1ull) * K_TOTAL <= 1ull << 32, "a lane's operand offsets fit 32 bits");
static_assert(N_RAW % 128 == 0 && N_RAW >= gt::N_PER_BLOCK, "raw output columns: a multiple of 128, at least one tile");

constexpr u32 X_TILE_BYTES = gt::M_PER_BLOCK * ROW_BYTES;   // tokens
constexpr u32 W_TILE_BYTES = gt::N_PER_BLOCK * ROW_BYTES;   // weights
constexpr u32 XS = gt::X_STAGES;                             // ring depth of the token tiles
constexpr u32 WS = gt::STAGES;                               // ring depth of the weight tiles
constexpr u32 W_RING_OFFSET = XS * X_TILE_BYTES;             // LDS: XS token tiles, then WS weight tiles
constexpr u32 K_STEPS = K_TOTAL / gt::K_STEP;

constexpr u32 WAVES = gt::WAVES_M * gt::WAVES_N;

constexpr bool BLOCKS16 = gt::BLOCKS16;
#if X17_EPILOGUE == 3 || X17_EPILOGUE == 5 || X17_EPILOGUE == 6
template <bool> struct NaturalOf { using Writers = NaturalWriters; };
template <> struct NaturalOf<true> { using Writers = NaturalWriters16; };
using Natural = NaturalOf<BLOCKS16>::Writers;
#endif
constexpr int XB = gt::WAVE_M / 16, WB = gt::WAVE_N / 16, WH = WB / 2;      // blocks of 16 tokens, of 16 columns, of half the columns
constexpr u32 CH = MMA == 1 ? 2 : 1;                         // 16-byte chunks a lane fetches per operand row
constexpr u32 SLICES16 = gt::K_STEP / (64 * CH);             // slices of a K step

// ------------------------------------------------------------------ tile loads

// LDS rows hold K_STEP bytes = CHUNKS chunks of 16; logical chunk c of row r is stored at position c ^ gt::swizzle(r): with 128-byte
// rows two rows share a line of the 64 four-byte banks, so the row PAIR is what has to be mixed in, with 64-byte rows the row QUAD.
constexpr u32 CHUNKS = gt::CHUNKS;
constexpr u32 UNIT_ROWS = gt::UNIT_ROWS;                    // rows one 64-lane x 16-byte direct-to-LDS load fills
// With eight waves, two per SIMD, only the first of each pair (waves 0 .. 3) requests tiles.  The arbiter serves
// that wave first: with the loads shared evenly it ended its step early and sat at the barrier while its partner,
// the same loads to issue between its MFMAs, finished alone.  (Splitting the weight units 6:2, 4:4, 2:6 or 0:8
// between the two measured the same as 8:0.)
constexpr u32 LOADER_WAVES = gt::LOADER_WAVES;            // (a four-wave workgroup has one wave per SIMD)
constexpr u32 X_UNITS = gt::X_UNITS;                      // such loads per loading wave, step and tile
constexpr u32 W_UNITS = gt::W_UNITS;
constexpr u32 LOADS_PER_STAGE = X_UNITS + W_UNITS;
static_assert((X_UNITS * UNIT_ROWS) % 16 == 0 && (W_UNITS * UNIT_ROWS) % 16 == 0, "a wave's share must keep the swizzle phase");

// A wave that has a SIMD to itself has registers to spare: it keeps one lane offset per load unit, the unit's
// own row offset included, and all loads of a tile share ONE scalar base (no scalar add per load, two scalar
// register pairs instead of sixteen).
constexpr bool LANE_UNIT_OFFSETS = gt::WAVES_PER_SIMD == 1;
constexpr u32 X_OFFSETS = LANE_UNIT_OFFSETS ? X_UNITS : 2;
constexpr u32 W_OFFSETS = LANE_UNIT_OFFSETS ? W_UNITS : 2;
X17_DEV constexpr u32 w_unit_row(u32 r0) {   // weight row that LDS weight row r0 (a multiple of the unit) starts from
	return gt::w_unit_row(r0, NATURAL_COLS);
}
struct LaneOffsets {
	u32 x_src[X_OFFSETS];   // per-lane byte offset into A for a direct-to-LDS load (even / odd load unit, or per unit)
	u32 w_src[W_OFFSETS];   // per-lane byte offset into B
	u32 frag_row;   // (lane % BLOCK) * ROW_BYTES
	u32 half;       // lane / BLOCK
	u32 swz;        // swizzle key of the fragment row this lane reads
};

// Direct-to-LDS loads of a loading wave's share of one token tile / one weight tile: loading wave w copies
// token rows [X_UNITS * UNIT_ROWS * w, +X_UNITS * UNIT_ROWS) and as many LDS weight rows.
// Which weight row an LDS weight row holds: gt::w_unit_row.  A 32 x 32 matrix instruction hands output row
// i = 8*(r/4) + 4*(lane/32) + r%4 to register r, so with WN = WAVE_N columns per wave a lane collects columns
// (WN/2)*(lane/32) + 16*bn + r; a 16 x 16 one row i = 4*(lane/16) + r, and columns (WN/4)*(lane/16) + 4*bn + r.  For the
// rows of one load unit the lane-dependent part is constant.
template <u32 U>
X17_DEV void issue_x_load(u8 const *a_tile, u8 *x_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	u8 *x_lds = x_tile + (wave * X_UNITS + U) * UNIT_ROWS * ROW_BYTES;
	if constexpr (LANE_UNIT_OFFSETS) {
		load_to_lds_16(x_lds, a_tile + (size_t)(wave * X_UNITS * UNIT_ROWS) * K_TOTAL + k0, lo.x_src[U]);
	} else {
		u8 const *x_src = a_tile + (size_t)((wave * X_UNITS + U) * UNIT_ROWS) * K_TOTAL + k0;
		load_to_lds_16(x_lds, x_src, lo.x_src[U & 1]);
	}
}
template <u32 U>
X17_DEV void issue_w_load(u8 const *b_tile, u8 *w_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	u32 r0 = (wave * W_UNITS + U) * UNIT_ROWS;
	u8 *w_lds = w_tile + r0 * ROW_BYTES;
	if constexpr (LANE_UNIT_OFFSETS) {
		load_to_lds_16(w_lds, b_tile + (size_t)w_unit_row(wave * W_UNITS * UNIT_ROWS) * K_TOTAL + k0, lo.w_src[U]);
	} else {
		u8 const *w_src = b_tile + (size_t)w_unit_row(r0) * K_TOTAL + k0;
		load_to_lds_16(w_lds, w_src, lo.w_src[U & 1]);
	}
}
// this wave's share of one token tile / one weight tile of one step
template <u32 FIRST = 0, u32 LAST = X_UNITS>
X17_DEV void issue_x_units(u8 const *a_tile, u8 *x_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	if constexpr (FIRST < LAST) {
		issue_x_load<FIRST>(a_tile, x_tile, k0, wave, lo);
		issue_x_units<FIRST + 1, LAST>(a_tile, x_tile, k0, wave, lo);
	}
}
template <u32 FIRST = 0>
X17_DEV void issue_w_units(u8 const *b_tile, u8 *w_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	if constexpr (FIRST < W_UNITS) {
		issue_w_load<FIRST>(b_tile, w_tile, k0, wave, lo);
		issue_w_units<FIRST + 1>(b_tile, w_tile, k0, wave, lo);
	}
}
// (the other waves have nothing in flight: their waits on the load counter fall through)
X17_DEV void issue_x_loads(u8 const *a_tile, u8 *x_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	if (wave < LOADER_WAVES) {
		issue_x_units(a_tile, x_tile, k0, wave, lo);
	}
}
X17_DEV void issue_w_loads(u8 const *b_tile, u8 *w_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	if (wave < LOADER_WAVES) {
		issue_w_units(b_tile, w_tile, k0, wave, lo);
	}
}

// Loads complete in issue order.  Behind every barrier a wave issues its share of one weight tile (step + WS)
// and then of one token tile (step + XS).  The tiles of step ks+1 are awaited with everything issued after
// the weight tile of that step still allowed in flight: the token tile issued with it when the token ring
// is the deeper one, and `later` whole steps.
X17_DEV void wait_step(u32 later, bool token_tile_behind) {
	if constexpr (WS >= 4) {
		if (later >= 2) {
			if (XS > WS && token_tile_behind) { wait_vmcnt<2 * LOADS_PER_STAGE + X_UNITS>(); } else { wait_vmcnt<2 * LOADS_PER_STAGE>(); }
			return;
		}
	}
	if constexpr (WS >= 3) {
		if (later >= 1) {
			if (XS > WS && token_tile_behind) { wait_vmcnt<LOADS_PER_STAGE + X_UNITS>(); } else { wait_vmcnt<LOADS_PER_STAGE>(); }
			return;
		}
	}
	if (XS > WS && token_tile_behind) { wait_vmcnt<X_UNITS>(); } else { wait_vmcnt<0>(); }
}

static_assert(SLICES % 2 == 0, "the fragment double buffer needs an even number of slices per step");

// Pin the issue order of one slice: the LDS reads of the next fragments and this slice's share of the
// next stage's global loads are spread evenly between the MFMAs.  LDS latency then hides under
// matrix-core time, and a wave never sits in a burst of loads waiting for the memory pipeline to
// accept them (instructions issue in order: a queued load would hold back the MFMAs behind it).
template <u32 N_LOADS>
X17_DEV void interleave_slice(bool with_reads) {
	if constexpr (MMA != 2) {
		constexpr int READS = (BN + BM) * CHUNKS_PER_FRAG;
		constexpr int MFMAS = BN * BM;
		constexpr int GROUPS = MFMAS < READS ? MFMAS : READS;
		if (with_reads) {
			X17_UNROLL for (int i = 0; i < GROUPS; ++i) {
				__builtin_amdgcn_sched_group_barrier(0x008, MFMAS / GROUPS, 0);
				__builtin_amdgcn_sched_group_barrier(0x100, READS / GROUPS, 0);
				if (i < (int)N_LOADS) {
					__builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
				}
			}
		} else {
			__builtin_amdgcn_sched_group_barrier(0x008, MFMAS, 0);
		}
	}
}

// ---- the paced form of a slice (int8 and e4m3 arithmetic): every MFMA is followed by its share of the next
// fragments' LDS reads and of the tile requests, and nothing may move across the group boundaries, so a
// wave that has a SIMD to itself for a while keeps the matrix core fed instead of issuing requests in a burst.
constexpr int MFMAS_PER_SLICE = BN * BM;
constexpr int READS_PER_SLICE = (BN + BM) * (int)CHUNKS_PER_FRAG;

template <int I>
X17_DEV void mma_one(Frags const &f, Acc (&acc)[BN][BM]) {
	constexpr int bn = I / BM, bm = I % BM;
	if constexpr (MMA == 0) {
		acc[bn][bm] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.w[bn][0], f.x[bm][0], acc[bn][bm], 0, 0, 0);
	} else {
		v4i wl = f.w[bn][0], wh = f.w[bn][CHUNKS_PER_FRAG - 1];
		v4i xl = f.x[bm][0], xh = f.x[bm][CHUNKS_PER_FRAG - 1];
		v8i wf = v8i{wl[0], wl[1], wl[2], wl[3], wh[0], wh[1], wh[2], wh[3]};
		v8i xf = v8i{xl[0], xl[1], xl[2], xl[3], xh[0], xh[1], xh[2], xh[3]};
		v16f r = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf, xf, __builtin_bit_cast(v16f, acc[bn][bm]), 0, 0, 0, 0, 0, 0);
		acc[bn][bm] = __builtin_bit_cast(Acc, r);
	}
}
// read number J of a slice's fragments, in the order the MFMAs want them: w0, every x, then the other w
template <int J>
X17_DEV void read_one(Frags &f, u8 const *w_tile, u8 const *x_tile, u32 s, LaneOffsets const &lo) {
	constexpr int q = J / (int)CHUNKS_PER_FRAG;
	constexpr u32 c = J % CHUNKS_PER_FRAG;
	u32 const kc = CHUNKS_PER_FRAG * (2 * s + lo.half) + c;
	if constexpr (q == 0) {
		f.w[0][c] = lds_chunk(w_tile, 0, kc, lo.swz);
	} else if constexpr (q <= BM) {
		f.x[q - 1][c] = lds_chunk(x_tile, (q - 1) * 32 * ROW_BYTES, kc, lo.swz);
	} else {
		f.w[q - BM][c] = lds_chunk(w_tile, (q - BM) * 32 * ROW_BYTES, kc, lo.swz);
	}
}
template <int FIRST, int LAST>
X17_DEV void read_range(Frags &f, u8 const *w_tile, u8 const *x_tile, u32 s, LaneOffsets const &lo) {
	if constexpr (FIRST < LAST) {
		read_one<FIRST>(f, w_tile, x_tile, s, lo);
		read_range<FIRST + 1, LAST>(f, w_tile, x_tile, s, lo);
	}
}
template <u32 FIRST, u32 LAST>
X17_DEV void issue_w_range(u8 const *b_tile, u8 *w_tile, u32 k0, u32 wave, LaneOffsets const &lo) {
	if constexpr (FIRST < LAST) {
		issue_w_load<FIRST>(b_tile, w_tile, k0, wave, lo);
		issue_w_range<FIRST + 1, LAST>(b_tile, w_tile, k0, wave, lo);
	}
}
// KIND 0: no requests, 1: token units [FIRST, FIRST + COUNT), 2: weight units [FIRST, FIRST + COUNT)
template <int I, bool READS, int KIND, u32 FIRST, u32 COUNT>
X17_DEV void paced_slice(Frags const &cur, Frags &next, u8 const *nw, u8 const *nx, u32 ns, LaneOffsets const &lo,
                         Acc (&acc)[BN][BM], u8 const *src, u8 *dst, u32 k0, u32 wave) {
	if constexpr (I < MFMAS_PER_SLICE) {
		mma_one<I>(cur, acc);
		if constexpr (READS) {
			constexpr int R0 = I * READS_PER_SLICE / MFMAS_PER_SLICE, R1 = (I + 1) * READS_PER_SLICE / MFMAS_PER_SLICE;
			read_range<R0, R1>(next, nw, nx, ns, lo);
		}
		constexpr u32 L0 = FIRST + I * COUNT / MFMAS_PER_SLICE, L1 = FIRST + (I + 1) * COUNT / MFMAS_PER_SLICE;
		if constexpr (KIND == 1) {
			issue_x_units<L0, L1>(src, dst, k0, wave, lo);
		} else if constexpr (KIND == 2) {
			issue_w_range<L0, L1>(src, dst, k0, wave, lo);
		}
		__builtin_amdgcn_sched_barrier(0);
		paced_slice<I + 1, READS, KIND, FIRST, COUNT>(cur, next, nw, nx, ns, lo, acc, src, dst, k0, wave);
	}
}

// ---- the paced form for the mixed arithmetic (e4m3 x int8 widened to f16; one wave per SIMD).  A slice of 32 bytes
// of K is two rounds of BN x BM f16 MFMAs (K = 16 each).  The operands of a round are widened one round ahead, a
// piece of four bytes behind each MFMA, so the conversions run in the shadow of the matrix core instead of in
// front of it; the raw fragments of the next slice are read during the first round, tiles requested in the second.
struct Wide {
	v8h w[BN];
	v8h x[BM];
};
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// four 8-bit values -> four f16, exact (see widen8)
X17_DEV v4h widen4(u32 word, int kind) {
	v2h lo2, hi2;
	if (kind == 1) {
		lo2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(word, 1.0f, false);
		hi2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(word, 1.0f, true);
	} else {
		v2h const bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
		u32 const u = word ^ 0x80808080u;
		lo2 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias;
		hi2 = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias;
	}
	return v4h{lo2[0], lo2[1], hi2[0], hi2[1]};
}
constexpr int WIDEN_PIECES = 2 * (BN + BM);      // per round: every fragment in two pieces of four bytes
// piece P of the operands of round H (0 / 1: bytes 0..7 / 8..15 of the lane's 16) of the raw fragments `f`,
// fragments in the order the MFMAs want them: w0, every x, then the other w
template <int P, int H>
X17_DEV void widen_piece(Wide &wd, Frags const &f) {
	constexpr int q = P / 2, p = P % 2, dw = 2 * H + p;
	if constexpr (q == 0 || q > BM) {
		constexpr int bn = q == 0 ? 0 : q - BM;
		v4h const r = widen4((u32)f.w[bn][0][dw], B_KIND);
		X17_UNROLL for (int i = 0; i < 4; ++i) wd.w[bn][4 * p + i] = r[i];
	} else {
		v4h const r = widen4((u32)f.x[q - 1][0][dw], A_KIND);
		X17_UNROLL for (int i = 0; i < 4; ++i) wd.x[q - 1][4 * p + i] = r[i];
	}
}
template <int FIRST, int LAST, int H>
X17_DEV void widen_range(Wide &wd, Frags const &f) {
	if constexpr (FIRST < LAST) {
		widen_piece<FIRST, H>(wd, f);
		widen_range<FIRST + 1, LAST, H>(wd, f);
	}
}
// One round.  NEXT_H < 0: nothing to widen (the tile's last round); else the next round's operands are round NEXT_H
// of `raw`.  READS: the raw fragments `rd` of slice `ns` of tiles (nw, nx) are read behind the first MFMAs.
// KIND / FIRST / COUNT: tile requests as in paced_slice.
template <int I, int NEXT_H, bool READS, int KIND, u32 FIRST, u32 COUNT>
X17_DEV void mixed_round(Wide const &cur, Wide &nxt, Frags const &raw, Frags &rd, u8 const *nw, u8 const *nx, u32 ns,
                         LaneOffsets const &lo, Acc (&acc)[BN][BM], u8 const *src, u8 *dst, u32 k0, u32 wave) {
	if constexpr (I < MFMAS_PER_SLICE) {
		constexpr int bn = I / BM, bm = I % BM;
		v16f const r = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.w[bn], cur.x[bm], __builtin_bit_cast(v16f, acc[bn][bm]), 0, 0, 0);
		acc[bn][bm] = __builtin_bit_cast(Acc, r);
		if constexpr (NEXT_H >= 0) {
			widen_range<I * WIDEN_PIECES / MFMAS_PER_SLICE, (I + 1) * WIDEN_PIECES / MFMAS_PER_SLICE, NEXT_H>(nxt, raw);
		}
		if constexpr (READS) {
			constexpr int R0 = I * READS_PER_SLICE / MFMAS_PER_SLICE, R1 = (I + 1) * READS_PER_SLICE / MFMAS_PER_SLICE;
			read_range<R0, R1>(rd, nw, nx, ns, lo);
		}
		constexpr u32 L0 = FIRST + I * COUNT / MFMAS_PER_SLICE, L1 = FIRST + (I + 1) * COUNT / MFMAS_PER_SLICE;
		if constexpr (KIND == 1) {
			issue_x_units<L0, L1>(src, dst, k0, wave, lo);
		} else if constexpr (KIND == 2) {
			issue_w_range<L0, L1>(src, dst, k0, wave, lo);
		}
		__builtin_amdgcn_sched_barrier(0);
		mixed_round<I + 1, NEXT_H, READS, KIND, FIRST, COUNT>(cur, nxt, raw, rd, nw, nx, ns, lo, acc, src, dst, k0, wave);
	}
}

// ---- 16 x 16 blocks (int8 x int8 and e4m3 x e4m3).  What bounds these kernels is the power the chip may draw: it lowers the clock
// until they fit, and per product the 16 x 16 instructions cost less of it than the 32 x 32 ones (half the accumulator traffic).  Loops
// of nothing but matrix instructions on Gaussian operands: int8 3.71 -> 4.29 POP/s, e4m3 4.16 -> 4.46.  us in turn, blocks of 32 / of 16:
//   int8, K = 2048, 16384 columns with the GeGLU writer, 32768 rows 865 / 795 (by the counters 1.69 -> 1.80 GHz and 1.5 % more cycles)
//   int8, run-time scales, K = 8192, 2048 columns, 8192 rows 115 / 104     e4m3, K = 16384, 8192 columns, 16384 rows 1485 / 1471,
//   4096 rows 358 / 345; K = 4096, 32768 columns, 16384 rows 1463 / 1442 (ten of eleven e4m3 products 1-4 % faster, one equal)
// The bytes are those of the 32 x 32 instructions.  int32 sums are exact; a 16x16x128 instruction adds sixteen products of every lane
// group at a time, in the groups' order, and so goes through K as two 32x32x64 instructions do if group g takes the chunks
// chunk16 names (no difference in 400 thousand sums of 2048 products each).
struct Frags16 {
	v4i x[XB][CH];
	v4i w[2][WH][CH];          // the wavefront's columns in two halves
};
// 16-byte chunk of a K step that is chunk c of slice s in lane group `group`'s fragments
X17_DEV u32 chunk16(u32 s, u32 c, u32 group) {
	return MMA == 0 ? 4 * s + group : 4 * c + ((group & 1) << 1 | group >> 1);
}
// chunk C of token block B, of slice s; chunk I of a half's column blocks
template <int B, u32 C>
X17_DEV void read_x16(Frags16 &f, u8 const *x_tile, u32 s, LaneOffsets const &lo) {
	f.x[B][C] = lds_chunk(x_tile, B * 16 * ROW_BYTES, chunk16(s, C, lo.half), lo.swz);
}
template <int HALF, int I>
X17_DEV void read_w16(Frags16 &f, u8 const *w_tile, u32 s, LaneOffsets const &lo) {
	f.w[HALF][I / CH][I % CH] = lds_chunk(w_tile, (HALF * WH + I / CH) * 16 * ROW_BYTES, chunk16(s, I % CH, lo.half), lo.swz);
}
template <int I>
X17_DEV void read_first16(Frags16 &f, u8 const *w_tile, u8 const *x_tile, LaneOffsets const &lo) {
	if constexpr (I < XB * (int)CH) {
		if constexpr (I < WH * (int)CH) read_w16<0, I>(f, w_tile, 0, lo);
		read_x16<I / (int)CH, I % (int)CH>(f, x_tile, 0, lo);
		read_first16<I + 1>(f, w_tile, x_tile, lo);
	}
}
X17_DEV v4i mma16(v4i const (&w)[CH], v4i const (&x)[CH], v4i acc) {
	if constexpr (MMA == 0) {
		return __builtin_amdgcn_mfma_i32_16x16x64_i8(w[0], x[0], acc, 0, 0, 0);
	} else {
		v4i const w1 = w[CH - 1], x1 = x[CH - 1];
		v8i const wf = {w[0][0], w[0][1], w[0][2], w[0][3], w1[0], w1[1], w1[2], w1[3]};
		v8i const xf = {x[0][0], x[0][1], x[0][2], x[0][3], x1[0], x1[1], x1[2], x1[3]};
		return __builtin_bit_cast(v4i, __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, __builtin_bit_cast(v4f, acc), 0, 0, 0, 0, 0, 0));
	}
}
constexpr bool w_units_alike() {
	for (u32 wave = 0; wave < LOADER_WAVES; ++wave) {
		for (u32 u = 0; u < W_UNITS; ++u) {
			if (w_unit_row((wave * W_UNITS + u) * UNIT_ROWS) - w_unit_row(wave * W_UNITS * UNIT_ROWS) != w_unit_row(u * UNIT_ROWS)) return false;
		}
	}
	return true;
}
static_assert(w_units_alike(), "a loading wave's weight rows lie alike whichever wave it is");
// (a pointer that is the same in every lane; reading it from the first one tells the compiler so)
X17_DEV u8 const *uniform(u8 const *p) {
	u64 const a = (u64)p;
	return (u8 const *)((u64)(u32)__builtin_amdgcn_readfirstlane((u32)(a >> 32)) << 32 | (u32)__builtin_amdgcn_readfirstlane((u32)a));
}
// Tile request U of a loading wave: a buffer load (base of the step's rows, lane offset, the unit's rows as a scalar offset) to the
// unit's part of `lds`.  (A scalar write of M0 needs one wait state before a direct-to-LDS load reads it.)
template <bool WEIGHTS, u32 U>
X17_DEV void request16(v4u rows, u32 lds, LaneOffsets const &lo) {
	constexpr u32 row = LANE_UNIT_OFFSETS ? 0 : WEIGHTS ? w_unit_row(U * UNIT_ROWS) : U * UNIT_ROWS;
	u32 const lane_offset = WEIGHTS ? lo.w_src[LANE_UNIT_OFFSETS ? U : U & 1] : lo.x_src[LANE_UNIT_OFFSETS ? U : U & 1];
	asm volatile("s_add_i32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
	             :: "s"(lds), "i"(U * UNIT_ROWS * ROW_BYTES), "v"(lane_offset), "s"(rows), "s"(row * K_TOTAL) : "memory", "m0", "scc");
}
X17_DEV v4u rows_resource(u8 const *p) {
	return v4u{(u32)(u64)p, (u32)((u64)p >> 32), (u32)gt::RESOURCE_BYTES, 0x00020000u};
}
// One part of a step: slice Q / 2 of K, all tokens, half Q % 2 of the columns.  Its reads are the other half's columns (of `w_tile`) and,
// behind a slice's last use of a token block, that block of the next slice (of `x_tile`), into the same registers.  Behind a matrix instruction
// comes one read, one request or a piece of the next step's addresses (`between`), not several: a wavefront issues an
// instruction in about nine clocks, a matrix instruction takes 16 (int8) or 32.
template <int Q, int I, bool READS, int KIND, u32 FIRST, u32 COUNT, class Between>
X17_DEV void paced16(Frags16 &f, u8 const *w_tile, u8 const *x_tile, LaneOffsets const &lo, v4i (&acc)[WB][XB], v4u rows, u32 lds, Between const &between) {
	constexpr int MFMAS = XB * WH, HALF = Q % 2, NEXT = HALF == 0 ? Q / 2 : (Q / 2 + 1) % (int)SLICES16;
	if constexpr (I < MFMAS) {
		constexpr int b = I / WH, j = I % WH;
		constexpr int EVERY = MFMAS / (int)COUNT, SLOT = HALF == 0 ? I - 1 : I;
		static_assert(MFMAS % COUNT == 0, "requests at even distances");
		acc[HALF * WH + j][b] = mma16(f.w[HALF][j], f.x[b], acc[HALF * WH + j][b]);
		__builtin_amdgcn_sched_barrier(0);      // (a token block's read stays behind the instruction above: it takes its operand's registers)
		if constexpr (READS) {
			// columns: behind every other instruction from the first one; in a slice's second half behind the second and (two chunks) third
			// of a token block's four
			constexpr int W_READS = WH * (int)CH;
			constexpr int W = HALF == 0 ? (I % 2 == 0 ? I / 2 : W_READS) : j == 1 ? b * (int)CH : j == 2 && CH == 2 ? b * 2 + 1 : W_READS;
			if constexpr (W < W_READS) read_w16<1 - HALF, W>(f, w_tile, NEXT, lo);
			if constexpr (HALF == 1) {
				// tokens: first chunks behind the block's last instruction, second ones where the columns' reads were
				if constexpr (j == WH - 1) read_x16<b, 0>(f, x_tile, NEXT, lo);
				constexpr int LATE = CH == 1 ? XB : b >= XB / 2 && (j == 1 || j == 2) ? 2 * (b - XB / 2) + j - 1 : I == MFMAS - 1 ? XB - 1 : XB;
				if constexpr (LATE < (I == MFMAS - 1 ? XB : XB - 1)) read_x16<LATE, CH - 1>(f, x_tile, NEXT, lo);
			}
		}
		if constexpr (KIND != 0) {
			if constexpr (SLOT >= 0 && SLOT % EVERY == 0) request16<KIND == 2, FIRST + SLOT / EVERY>(rows, lds, lo);
		}
		between.template operator()<I>();
		__builtin_amdgcn_sched_barrier(0);
		paced16<Q, I + 1, READS, KIND, FIRST, COUNT>(f, w_tile, x_tile, lo, acc, rows, lds, between);
	}
}

} // namespace

extern "C" __global__ __launch_bounds__(gt::THREADS_PER_BLOCK)
__attribute__((amdgpu_waves_per_eu(gt::WAVES_PER_SIMD, gt::WAVES_PER_SIMD)))
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
	, u16 const *q_norm_scales          // bf16 [N_raw]
#elif X17_EPILOGUE == 6
	// a, b = q weights [X17_Q_COLS, K], c = q [M, X17_Q_COLS]; then:
	, f32 *rrms, u8 const *b_kv /* [N_raw - X17_Q_COLS, K] */, u8 *c_kv /* [M, N_raw - X17_Q_COLS] */
#endif
) {
	extern __shared__ __attribute__((aligned(1024))) u8 smem[];
	(void)b_rows;   // known at compile time, as in templates/basic_gemm/kernel.cu:18-21

	// ---- which tiles.  The kernel is persistent: workgroup g of G works on tiles g, g + G, ... and
	// any grid shape is accepted (with one workgroup per tile, as the reference launches it, every
	// workgroup runs the loop once).  The linear tile id is remapped so that each XCD (own L2) gets a
	// compact block of tiles -- the hardware deals workgroups round-robin to the 8 XCDs -- and tiles
	// are walked in bands of token-tiles so that co-resident tiles share weight and token panels.
	// A shape that is not a whole number of tiles (src/device/cuda/gemm.rs:605-614 accepts rows % 64 == 0 and raw
	// columns % 128 == 0) is covered by moving the last tile of a row or column of tiles back until it ends at the
	// matrix edge: it recomputes a few rows or columns of its neighbour and stores the same bytes again, and nothing
	// in the kernel needs a predicate.  (tile_coords hands out a tile's first row and first raw column.)
	u32 const tiles_m = (a_rows + gt::M_PER_BLOCK - 1) / gt::M_PER_BLOCK;
	constexpr u32 tiles_n = (N_RAW + gt::N_PER_BLOCK - 1) / gt::N_PER_BLOCK;
	u32 const total = tiles_m * tiles_n;
	u32 const n_groups = gridDim.x * gridDim.y * gridDim.z;
	u32 const group = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
	auto tile_coords = [&](u32 lin, u32 &tile_m, u32 &tile_n) {
		gt::TileOrigin const o = gt::tile_origin(lin, a_rows, N_RAW, gt::BAND);
		tile_m = o.m;
		tile_n = o.n;
	};
	if (group >= total) {
		return;
	}

	u32 const tid = threadIdx.x;
	u32 const lane = tid % 64;
	u32 const wave = __builtin_amdgcn_readfirstlane(tid / 64);
	u32 const wm = wave / gt::WAVES_N;
	u32 const wn = wave % gt::WAVES_N;

	LaneOffsets lo;
	{
		// (row inside a load unit and logical chunk of the stored chunk position: gemm_tile.h)
		u32 even_odd_x[2], even_odd_w[2];
		X17_UNROLL for (u32 odd = 0; odd < 2; ++odd) {
			u32 const chunk = gt::lane_chunk(lane, odd);
			even_odd_x[odd] = gt::x_lane_row(lane) * K_TOTAL + 16 * chunk;
			even_odd_w[odd] = gt::w_lane_row(lane, NATURAL_COLS) * K_TOTAL + 16 * chunk;
		}
		if constexpr (LANE_UNIT_OFFSETS) {
			u32 const w_first = wave * W_UNITS * UNIT_ROWS;
			X17_UNROLL for (u32 u = 0; u < X_UNITS; ++u) lo.x_src[u] = even_odd_x[u & 1] + u * UNIT_ROWS * K_TOTAL;
			X17_UNROLL for (u32 u = 0; u < W_UNITS; ++u) {
				lo.w_src[u] = even_odd_w[u & 1] + (w_unit_row(w_first + u * UNIT_ROWS) - w_unit_row(w_first)) * K_TOTAL;
			}
		} else {
			X17_UNROLL for (u32 odd = 0; odd < 2; ++odd) {
				lo.x_src[odd] = even_odd_x[odd];
				lo.w_src[odd] = even_odd_w[odd];
			}
		}
		lo.frag_row = (lane % gt::BLOCK) * ROW_BYTES;
		lo.half = lane / gt::BLOCK;
		lo.swz = gt::swizzle(lane % gt::BLOCK);
	}

	// ---- main loop.  Rings of XS token tiles and WS weight tiles in LDS; step ks consumes ring positions
	// ks % XS and ks % WS while the tiles of the following steps are in flight.  The one barrier per step sits
	// before the last slice's MFMAs, when every wave holds the last fragments of the step in registers: behind
	// it both positions are free, so the weight tile of step ks+WS and the token tile of step ks+XS are
	// requested there, and the first fragments of step ks+1 are fetched, so LDS latency is covered by
	// matrix-core time across the step boundary too.  The load stream runs across tile boundaries: the last
	// steps of a tile already fetch the first steps of the workgroup's next tile, which land while the epilogue
	// runs.  (a K shorter than the ring cannot prefetch across tiles: each tile then starts with its own prologue)
	static_assert(XS == WS || WS == 2, "a deeper token ring is supported on top of a two-deep weight ring");
	constexpr bool CROSS_TILE = K_STEPS >= XS;
	// Paced form: a step requests its token tile (step + XS - 1, into the position the PREVIOUS step's barrier
	// freed) during its first slices and its weight tile (step + WS) behind its own barrier, every request behind
	// an MFMA.  The pattern is the same in every step of every tile -- where nothing is left to fetch the request
	// is repeated from the tile's start into a position that no step reads again -- so no branch sits between
	// the MFMAs and the wait before a barrier is always "all but the token tile just requested".
	// (e4m3 fragments are twice the size: two such waves per SIMD do not fit the pinned order into 256 registers)
	constexpr bool PACED = WS == 2 && XS == 3 && CROSS_TILE && SLICES >= 2 && (MMA == 0 || gt::WAVES_PER_SIMD == 1);
	u32 const x_off = wm * gt::WAVE_M * ROW_BYTES + lo.frag_row;
	u32 const w_off = W_RING_OFFSET + wn * gt::WAVE_N * ROW_BYTES + lo.frag_row;

	// the weight rows of the tile whose first raw column is `col`: one matrix, or (fused q + kv) the q weights
	// followed by the kv weights
	auto weight_tile = [&](u32 col) -> u8 const * {
#if X17_EPILOGUE == 6
		static_assert(X17_Q_COLS % gt::N_PER_BLOCK == 0 && N_RAW - X17_Q_COLS >= gt::N_PER_BLOCK, "q and kv parts are whole tiles / at least a tile");
		return col < X17_Q_COLS ? b + (size_t)col * K_TOTAL : b_kv + (size_t)(col - X17_Q_COLS) * K_TOTAL;
#else
		return b + (size_t)col * K_TOTAL;
#endif
	};
	u32 tile_m, tile_n;
	tile_coords(group, tile_m, tile_n);
	u8 const *a_tile = a + (size_t)tile_m * K_TOTAL;
	u8 const *b_tile = weight_tile(tile_n);
	// the first steps of a tile nobody prefetched, in the order the waits of the main loop assume
	// (token tile s, weight tile s, ..., then the extra token tile of a deeper token ring)
	auto prologue = [&]() __attribute__((always_inline)) {
		X17_UNROLL for (u32 s = 0; s < WS; ++s) {
			if (s < K_STEPS) {
				issue_x_loads(a_tile, smem + s * X_TILE_BYTES, s * gt::K_STEP, wave, lo);
				issue_w_loads(b_tile, smem + W_RING_OFFSET + s * W_TILE_BYTES, s * gt::K_STEP, wave, lo);
			}
		}
		if constexpr (XS > WS && CROSS_TILE && !PACED) {
			issue_x_loads(a_tile, smem + WS * X_TILE_BYTES, WS * gt::K_STEP, wave, lo);
		}
		wait_vmcnt<0>();
		step_barrier();
	};
	prologue();

	u32 xb = 0, wb = 0;                            // ring positions of the step being consumed
	for (u32 lin = group; lin < total; lin += n_groups) {
		bool const first_tile = lin == group;
		bool const more_tiles = lin + n_groups < total;
		bool const has_next = CROSS_TILE && more_tiles;      // prefetch the next tile's first steps
		u32 next_m = 0, next_n = 0;
		if (more_tiles) {
			tile_coords(lin + n_groups, next_m, next_n);
		}
		u8 const *a_next = a + (size_t)next_m * K_TOTAL;
		u8 const *b_next = weight_tile(next_n);
		if constexpr (!CROSS_TILE) {
			if (!first_tile) {
				step_barrier();      // nobody still reads the previous tile's buffers
				xb = 0;
				wb = 0;
				prologue();
			}
		}

		[[maybe_unused]] v4i acc16[WB][XB];
		if constexpr (BLOCKS16) {
			X17_UNROLL for (int bn = 0; bn < WB; ++bn) {
				X17_UNROLL for (int bm = 0; bm < XB; ++bm) acc16[bn][bm] = v4i{0, 0, 0, 0};
			}
			Frags16 f;
			read_first16<0>(f, smem + wb * W_TILE_BYTES + w_off, smem + xb * X_TILE_BYTES + x_off, lo);
			auto k_loop = [&]<bool LOADER>() __attribute__((always_inline)) {
				constexpr u32 PARTS = 2 * SLICES16, X_PARTS = PARTS / 2;        // parts of a step; those that carry token requests
				size_t const x_wave = (size_t)(wave * X_UNITS * UNIT_ROWS) * K_TOTAL, w_wave = (size_t)w_unit_row(wave * W_UNITS * UNIT_ROWS) * K_TOTAL;
				u8 const *const a_rows_here = uniform(a_tile + x_wave), *const a_rows_next = uniform(a_next + x_wave);
				u8 const *const b_rows_here = uniform(b_tile + w_wave), *const b_rows_next = uniform(b_next + w_wave);
				u32 const lds0 = (u32)(size_t)X17_LDS_PTR(smem);
				u32 const lds_wave_x = lds0 + wave * X_UNITS * UNIT_ROWS * ROW_BYTES, lds_wave_w = lds0 + W_RING_OFFSET + wave * W_UNITS * UNIT_ROWS * ROW_BYTES;
				bool const hn = has_next;
				// a step's tiles, the rows its requests take and where they go; the next step's are computed a piece at a time in this one
				struct Step { u8 const *w_tile, *x_tile, *lx, *lw; u32 x_lds, w_lds; } now, next;
				u32 next_xb = xb, next_wb = wb;
				auto tiles = [&](Step &s) __attribute__((always_inline)) {
					s.w_tile = smem + next_wb * W_TILE_BYTES + w_off;
					s.x_tile = smem + next_xb * X_TILE_BYTES + x_off;
				};
				u32 x_k0 = 0, w_k0 = 0;
				auto offsets = [&](u32 ks) __attribute__((always_inline)) {
					u32 const x_step = ks + XS - 1, w_step = ks + WS;
					x_k0 = (x_step < K_STEPS ? x_step : (hn ? x_step - K_STEPS : 0)) * gt::K_STEP;
					w_k0 = (w_step < K_STEPS ? w_step : (hn ? w_step - K_STEPS : 0)) * gt::K_STEP;
				};
				// (values, not the captured variables: a choice between two captured pointers would keep them in memory)
				auto token_rows = [&](Step &s, u32 ks) __attribute__((always_inline)) {
					u8 const *const here = a_rows_here, *const after = a_rows_next;
					s.lx = (ks + XS - 1 < K_STEPS || !hn ? here : after) + x_k0;
				};
				auto weight_rows = [&](Step &s, u32 ks) __attribute__((always_inline)) {
					u8 const *const here = b_rows_here, *const after = b_rows_next;
					s.lw = (ks + WS < K_STEPS || !hn ? here : after) + w_k0;
				};
				auto token_destination = [&](Step &s) __attribute__((always_inline)) {
					s.x_lds = __builtin_amdgcn_readfirstlane(lds_wave_x + (next_xb == 0 ? XS - 1 : next_xb - 1) * X_TILE_BYTES);
				};
				auto weight_destination = [&](Step &s) __attribute__((always_inline)) {
					s.w_lds = __builtin_amdgcn_readfirstlane(lds_wave_w + next_wb * W_TILE_BYTES);
				};
				tiles(now);
				offsets(0);
				token_rows(now, 0);
				weight_rows(now, 0);
				token_destination(now);
				weight_destination(now);
				auto const nothing = [&]<int I>() __attribute__((always_inline)) {};
				auto step = [&]<bool LAST_STEP>(u32 ks) __attribute__((always_inline)) {
					auto const addresses = [&]<int I>() __attribute__((always_inline)) {
						constexpr int FROM = XB * WH / 2;      // behind the part's reads
						if constexpr (I == FROM) {
							next_xb = next_xb + 1 == XS ? 0 : next_xb + 1;
							next_wb = next_wb + 1 == WS ? 0 : next_wb + 1;
						} else if constexpr (I == FROM + 1 && !LAST_STEP) {
							tiles(next);
						} else if constexpr (I == FROM + 2 && !LAST_STEP) {
							offsets(ks + 1);
						} else if constexpr (I == FROM + 3 && !LAST_STEP) {
							token_rows(next, ks + 1);
						} else if constexpr (I == FROM + 4 && !LAST_STEP) {
							weight_rows(next, ks + 1);
						} else if constexpr (I == FROM + 5 && !LAST_STEP) {
							token_destination(next);
						} else if constexpr (I == FROM + 6 && !LAST_STEP) {
							weight_destination(next);
						}
					};
					v4u const x_rows = rows_resource(now.lx), w_rows = rows_resource(now.lw);
					auto parts = [&]<u32 Q>(auto &&self) __attribute__((always_inline)) {
						if constexpr (Q + 1 < PARTS) {
							constexpr u32 FIRST = (Q < X_PARTS ? Q : X_PARTS) * X_UNITS / X_PARTS, LAST = (Q + 1 < X_PARTS ? Q + 1 : X_PARTS) * X_UNITS / X_PARTS;
							constexpr int KIND = LOADER && Q < X_PARTS ? 1 : 0;
							constexpr u32 COUNT = KIND != 0 ? LAST - FIRST : 1;
							if constexpr (Q + 2 < PARTS) paced16<Q, 0, true, KIND, FIRST, COUNT>(f, now.w_tile, now.x_tile, lo, acc16, x_rows, now.x_lds, nothing);
							else paced16<Q, 0, true, KIND, FIRST, COUNT>(f, now.w_tile, now.x_tile, lo, acc16, x_rows, now.x_lds, addresses);
							self.template operator()<Q + 1>(self);
						} else {
							// the next step's tiles have landed once all but the token tile just requested have; this wave is done
							// reading this step's tiles
							wait_vmcnt<X_UNITS>();
							step_barrier();
							paced16<Q, 0, !LAST_STEP, LOADER ? 2 : 0, 0, W_UNITS>(f, next.w_tile, next.x_tile, lo, acc16, w_rows, now.w_lds, nothing);
						}
					};
					parts.template operator()<0>(parts);
				};
				// (the last step, which reads nothing ahead, behind the loop: a choice inside makes copies of the accumulators)
				_Pragma("clang loop unroll(disable)")
				for (u32 ks = 0; ks + 1 < K_STEPS; ++ks) {
					step.template operator()<false>(ks);
					now = next;
				}
				step.template operator()<true>(K_STEPS - 1);
				if constexpr (gt::NATURAL) {
					// (one register each where the loading wavefronts' loop and the others' meet: with places of their own in either, up to
					// eight spill in the q + kv writer at head_dim 64)
					X17_UNROLL for (int bn = 0; bn < WB; ++bn) {
						X17_UNROLL for (int bm = 0; bm < XB; ++bm) asm volatile("" : "+v"(acc16[bn][bm]));
					}
				}
				xb = next_xb;
				wb = next_wb;
			};
			if (WAVES == LOADER_WAVES || wave < LOADER_WAVES) {
				k_loop.template operator()<true>();
			} else {
				k_loop.template operator()<false>();
			}
		}
		[[maybe_unused]] Acc acc[BN][BM];   // [bn][bm]
		if constexpr (!BLOCKS16) {
		X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
			X17_UNROLL for (int bm = 0; bm < BM; ++bm) {
				X17_UNROLL for (int r = 0; r < 16; ++r) acc[bn][bm][r] = 0;
			}
		}

		// (step 0 of this tile is visible: the wait and the barrier were the previous tile's last ones)
		Frags frags[2];
		load_frags(frags[0], smem + wb * W_TILE_BYTES + w_off, smem + xb * X_TILE_BYTES + x_off, 0, lo.half, lo.swz);
		[[maybe_unused]] Wide wide[2];
		if constexpr (PACED && MMA == 2) {
			widen_range<0, WIDEN_PIECES, 0>(wide[0], frags[0]);      // (the only conversions of a tile no MFMA covers)
		}

		auto paced_k_loop = [&]<bool LOADER>() __attribute__((always_inline)) {
			constexpr u32 X_SLICES = SLICES >= 4 ? 2 : 1;                 // slices that carry token requests
			constexpr u32 X_PER_SLICE = X_UNITS / X_SLICES;
			// (values, not the captured variables: a choice between two captured pointers would keep them in memory)
			u8 const *const at = a_tile, *const an = a_next, *const bt = b_tile, *const bnx = b_next;
			bool const hn = has_next;
			// (no unroll pragma here: with the issue order pinned, unrolling a short loop completely costs no registers,
			// and the rolled form of this loop spills)
			for (u32 ks = 0; ks < K_STEPS; ++ks) {
				u32 const next_xb = xb + 1 == XS ? 0 : xb + 1;
				u32 const next_wb = wb + 1 == WS ? 0 : wb + 1;
				u32 const prev_xb = xb == 0 ? XS - 1 : xb - 1;
				u32 const x_step = ks + XS - 1, w_step = ks + WS;
				bool const x_here = x_step < K_STEPS, w_here = w_step < K_STEPS;
				u8 const *lx = (x_here || !hn) ? at : an;
				u8 const *lw = (w_here || !hn) ? bt : bnx;
				u32 const x_k0 = (x_here ? x_step : (hn ? x_step - K_STEPS : 0)) * gt::K_STEP;
				u32 const w_k0 = (w_here ? w_step : (hn ? w_step - K_STEPS : 0)) * gt::K_STEP;
				u8 *x_dst = smem + prev_xb * X_TILE_BYTES;
				u8 *w_dst = smem + W_RING_OFFSET + wb * W_TILE_BYTES;
				u8 const *w_tile = smem + wb * W_TILE_BYTES + w_off;
				u8 const *x_tile = smem + xb * X_TILE_BYTES + x_off;
				u8 const *nw_tile = smem + next_wb * W_TILE_BYTES + w_off;
				u8 const *nx_tile = smem + next_xb * X_TILE_BYTES + x_off;
				auto slices = [&]<u32 S>(auto &&self) __attribute__((always_inline)) {
					if constexpr (MMA == 2) {
						// first round: the operands of the second round are widened from the same raw fragments, the
						// next slice's raw fragments are read (behind the step's barrier when they belong to the next
						// step); second round: the next slice's first operands are widened, tiles are requested
						constexpr bool LAST = S + 1 == SLICES;
						constexpr int KIND = !LOADER ? 0 : (LAST ? 2 : (S < X_SLICES ? 1 : 0));
						constexpr u32 FIRST = LAST ? 0 : S * X_PER_SLICE, COUNT = LAST ? W_UNITS : X_PER_SLICE;
						u8 const *src = LAST ? lw : lx;
						u8 *dst = LAST ? w_dst : x_dst;
						u32 const k0 = LAST ? w_k0 : x_k0;
						if constexpr (LAST) {
							wait_vmcnt<X_UNITS>();
							step_barrier();
							// (the same code in a tile's last step, where what it reads and widens is never used: two
							// copies of the rounds would have to agree on where 256 accumulators live when they meet)
							mixed_round<0, 1, true, 0, 0, 0>(wide[0], wide[1], frags[S & 1], frags[(S + 1) & 1], nw_tile, nx_tile, 0, lo, acc, src, dst, k0, wave);
							mixed_round<0, 0, false, KIND, FIRST, COUNT>(wide[1], wide[0], frags[(S + 1) & 1], frags[S & 1], nw_tile, nx_tile, 0, lo, acc, src, dst, k0, wave);
						} else {
							mixed_round<0, 1, true, 0, 0, 0>(wide[0], wide[1], frags[S & 1], frags[(S + 1) & 1], w_tile, x_tile, S + 1, lo, acc, src, dst, k0, wave);
							mixed_round<0, 0, false, KIND, FIRST, COUNT>(wide[1], wide[0], frags[(S + 1) & 1], frags[S & 1], w_tile, x_tile, S + 1, lo, acc, src, dst, k0, wave);
							self.template operator()<S + 1>(self);
						}
					} else if constexpr (S + 1 < SLICES) {
						constexpr int KIND = LOADER && S < X_SLICES ? 1 : 0;
						paced_slice<0, true, KIND, S * X_PER_SLICE, X_PER_SLICE>(
							frags[S & 1], frags[(S + 1) & 1], w_tile, x_tile, S + 1, lo, acc, lx, x_dst, x_k0, wave);
						self.template operator()<S + 1>(self);
					} else {
						// the next step's tiles have landed once all but the token tile just requested have;
						// this wave is done reading this step's tiles
						wait_vmcnt<X_UNITS>();
						step_barrier();
						constexpr int KIND = LOADER ? 2 : 0;
						if (ks + 1 < K_STEPS) {
							paced_slice<0, true, KIND, 0, W_UNITS>(
								frags[S & 1], frags[(S + 1) & 1], nw_tile, nx_tile, 0, lo, acc, lw, w_dst, w_k0, wave);
						} else {
							paced_slice<0, false, KIND, 0, W_UNITS>(
								frags[S & 1], frags[(S + 1) & 1], nw_tile, nx_tile, 0, lo, acc, lw, w_dst, w_k0, wave);
						}
					}
				};
				slices.template operator()<0>(slices);
				xb = next_xb;
				wb = next_wb;
			}
		};
		if constexpr (PACED) {
			if (WAVES == LOADER_WAVES || wave < LOADER_WAVES) {
				paced_k_loop.template operator()<true>();
			} else {
				paced_k_loop.template operator()<false>();
			}
		} else {
		X17_K_LOOP_PRAGMA
		for (u32 ks = 0; ks < K_STEPS; ++ks) {
			u32 const next_xb = xb + 1 == XS ? 0 : xb + 1;
			u32 const next_wb = wb + 1 == WS ? 0 : wb + 1;
			// the tiles requested behind this step's barrier: weight step ks+WS, token step ks+XS (of this
			// output tile or of the workgroup's next one)
			u32 const w_step = ks + WS, x_step = ks + XS;
			bool const w_here = w_step < K_STEPS, x_here = x_step < K_STEPS;
			u8 const *lw = w_here ? b_tile : b_next;
			u8 const *lx = x_here ? a_tile : a_next;
			u32 const w_k0 = (w_here ? w_step : w_step - K_STEPS) * gt::K_STEP;
			u32 const x_k0 = (x_here ? x_step : x_step - K_STEPS) * gt::K_STEP;
			u8 const *w_tile = smem + wb * W_TILE_BYTES + w_off;
			u8 const *x_tile = smem + xb * X_TILE_BYTES + x_off;
			X17_UNROLL for (u32 s = 0; s < SLICES; ++s) {
				bool reads = true;
				if (s + 1 < SLICES) {
					load_frags(frags[(s + 1) & 1], w_tile, x_tile, s + 1, lo.half, lo.swz);
				} else if (ks + 1 < K_STEPS || has_next) {
					// Step ks+1 (or the next tile's step 0) must have landed; what was requested after its weight
					// tile may stay in flight: the token tile of step ks+2 when the token ring is the deeper one,
					// and up to WS-2 whole steps.  After an epilogue its stores share the counter with the loads:
					// wait for everything then.
					u32 const later_steps = has_next ? WS - 2 : (K_STEPS - 2 - ks < WS - 2 ? K_STEPS - 2 - ks : WS - 2);
					bool const token_tile_behind = has_next || ks + 2 < K_STEPS;
					bool const stores_pending = !first_tile && ks + 1 < WS;
					if (stores_pending) {
						wait_vmcnt<0>();
					} else {
						wait_step(later_steps, token_tile_behind);
					}
					step_barrier();      // this wave is done reading this step's tiles
					if (w_here || has_next) {
						issue_w_loads(lw, smem + W_RING_OFFSET + wb * W_TILE_BYTES, w_k0, wave, lo);
					}
					if (x_here || has_next) {
						issue_x_loads(lx, smem + xb * X_TILE_BYTES, x_k0, wave, lo);
					}
					if (ks + 1 < K_STEPS) {
						load_frags(frags[(s + 1) & 1], smem + next_wb * W_TILE_BYTES + w_off, smem + next_xb * X_TILE_BYTES + x_off, 0, lo.half, lo.swz);
					} else {
						reads = false;
					}
				} else {
					reads = false;
				}
				mma_slice(frags[s & 1], acc);
				if (s + 1 < SLICES) {
					interleave_slice<0>(reads);
				} else {
					interleave_slice<LOADS_PER_STAGE>(reads);
				}
			}
			xb = next_xb;
			wb = next_wb;
		}
		}

		}
	// ---- epilogue.  Lane owns token (BLOCK*bm + lane%BLOCK) of its wave and raw columns LANE_COLS*(lane/BLOCK) + 16*bn + r
	// (blocks of 16: 4*bn + r) of its wave, r = accumulator register index.
	u32 here = lane;
	if constexpr (BLOCKS16 && gt::NATURAL) {
		// (asked for anew: what these writers derive from the lane would live through the K loop, and spills)
		u32 every = ~0u;
		asm volatile("" : "+s"(every));
		here = __builtin_amdgcn_mbcnt_hi(every, __builtin_amdgcn_mbcnt_lo(every, 0));
	}
	u32 const part = here / gt::BLOCK;
	u32 const row0 = tile_m + wm * gt::WAVE_M + here % gt::BLOCK;
	u32 const n0 = tile_n + wn * gt::WAVE_N + LANE_COLS * part;

	X17_UNROLL for (int bm = 0; bm < (BLOCKS16 ? XB : BM); ++bm) {
		if constexpr (gt::WAVES_PER_SIMD == 1) {
			// Accumulators in the second half of the register file (where the vector ALU cannot read them) are copied
			// out row by row: pinning the later rows where they are keeps the register allocator from copying all
			// 256 out at once behind the K loop, which leaves no register for anything else.
			X17_UNROLL for (int later = bm + 1; later < (BLOCKS16 ? XB : BM); ++later) {
				X17_UNROLL for (int bn = 0; bn < (BLOCKS16 ? WB : BN); ++bn) {
					if constexpr (BLOCKS16) asm volatile("" : "+a"(acc16[bn][later]));
					else asm volatile("" : "+a"(acc[bn][later]));
				}
			}
		}
		u32 row = row0 + gt::BLOCK * bm;
		f32 x[LANE_COLS];
		if constexpr (BLOCKS16) {
			X17_UNROLL for (int bn = 0; bn < WB; ++bn) {
				v4f const as_f32 = __builtin_bit_cast(v4f, acc16[bn][bm]);
				X17_UNROLL for (int r = 0; r < 4; ++r) x[4 * bn + r] = ACC_F32 ? as_f32[r] : f32(acc16[bn][bm][r]);
			}
		} else
		X17_UNROLL for (int bn = 0; bn < BN; ++bn) {
			// (bit-casting a single vector element in place reads element 0; cast the whole vector first)
			v16f const as_f32 = __builtin_bit_cast(v16f, acc[bn][bm]);
			X17_UNROLL for (int r = 0; r < 16; ++r) {
				if constexpr (ACC_F32) {
					x[16 * bn + r] = as_f32[r];
				} else {
					x[16 * bn + r] = f32(acc[bn][bm][r]);
				}
			}
		}
#if X17_EPILOGUE == 0
		ScaleEpilogue::run(x, c, row, n0, nullptr);
#elif X17_EPILOGUE == 1
		GeGluEpilogue::run(x, c, row, n0, nullptr);
#elif X17_EPILOGUE == 2
		ResidualEpilogue::run(x, c, row, n0, residual);
#elif X17_EPILOGUE == 4
		DequantEpilogue::run(x, c, row, n0, row_scale, col_scale);
#elif X17_EPILOGUE == 3
		Natural::l2norm_row(x, c, rrms, row, tile_n + wn * gt::WAVE_N, N_RAW, part);
#elif X17_EPILOGUE == 5
		Natural::qnorm_row(x, c, q_norm_scales, row, tile_n + wn * gt::WAVE_N, part);
#else
		Natural::qkv_row(x, c, c_kv, rrms, row, tile_n + wn * gt::WAVE_N, part);
#endif
	}

		tile_m = next_m;
		tile_n = next_n;
		a_tile = a_next;
		b_tile = b_next;
	}
	// the paced form's last requests go nowhere useful, but they write LDS: they must land before the workgroup ends
	wait_vmcnt<0>();
}
