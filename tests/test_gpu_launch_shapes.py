"""Launch geometries that the operator layer's own launchers do not use but the kernels accept, driven through the raw
shim: attention grids with groups of heads per workgroup (src/device/cuda/attn.rs:60-66, 413-415: grid.y counts groups of
128 / head_dim heads) give the bytes of the one-head-per-workgroup launch, forward and backward."""
import ctypes
import json
import math
import os

import numpy as np
import pytest

import x17ai_amd as X
from x17ai_amd import _ffi, recipes
from tests.gpu_common import e4m3_bytes, e4m3_compare, i8_codes, rng_for
from tests.test_gpu_shim import P, SZ, _ok, _value, shim  # noqa: F401  (shim is a fixture)

pytestmark = pytest.mark.gpu


def _launch(shim, directory, meta, grid, slots):
	"""One launch of a built code object with `grid`, on a stream of its own."""
	ctx = _value(shim, shim.x17ai_hip_open_context(0))
	stream = _value(shim, shim.x17ai_hip_open_stream(ctx))
	module = _value(shim, shim.x17ai_hip_load_module(ctx, os.path.join(directory, "kernel.hsaco").encode()))
	function = _value(shim, shim.x17ai_hip_get_kernel(module, b"kernel", meta["SMEM_BYTES"]))
	values = [ctypes.c_uint64(s.device_ptr() if isinstance(s, X.Tensor) else s) for s in slots]
	args = (P * len(values))(*[ctypes.cast(ctypes.byref(v), P) for v in values])
	_ok(shim, shim.x17ai_hip_launch_kernel(stream, function, *grid, meta["THREADS_PER_BLOCK"], 1, 1, meta["SMEM_BYTES"], args))
	_ok(shim, shim.x17ai_hip_synchronize(stream))
	_ok(shim, shim.x17ai_hip_del_module(module))
	_ok(shim, shim.x17ai_hip_close_stream(stream))
	_ok(shim, shim.x17ai_hip_close_context(ctx))


def _launch_groups(shim, kernel, grid, slots):
	_launch(shim, os.path.join(_ffi.kernel_cache_dir(), kernel.name), kernel.metadata, grid, slots)


@pytest.mark.parametrize("h,hd,seq,batch,window", [(4, 32, 192, 2, 48), (2, 64, 256, 1, 0)])
def test_head_groups_in_the_grid(shim, h, hd, seq, batch, window):  # noqa: F811
	dev = X.Device(0)
	rng = rng_for("head groups", h, hd, seq, batch, window)
	rows, width = seq * batch, h * hd
	t = lambda a, dtype: X.Tensor.from_numpy(dev, a, dtype)
	q, kv = t(i8_codes(rng, (rows, width)), X.INT8), t(i8_codes(rng, (rows, 2 * width)), X.INT8)
	sk, sv = t(i8_codes(rng, (h, hd)), X.INT8), t(i8_codes(rng, (h, hd)), X.INT8)
	temp = t((0.5 + rng.random(h)).astype(np.float32), X.F32)
	d_out = t((rng.standard_normal((rows, width)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16), X.BF16)
	new = lambda shape, dtype: [X.Tensor(dev, shape, dtype) for _ in range(2)]
	out, l, d_q, d, d_kv = new((rows, width), X.INT8), new((h, rows), X.F32), new((rows, width), X.BF16), new((h, rows), X.F32), new((rows, 2 * width), X.BF16)
	fwd, bq, bkv = (make(dev, h, hd, True) for make in (recipes.attn_kernel, recipes.attn_d_q_kernel, recipes.attn_d_kv_kernel))
	fwd.launch(q, kv, sk, sv, temp, out[0], l[0], window, batch)
	bq.launch_d_q(q, kv, sk, sv, temp, out[0], d_out, d_q[0], l[0], d[0], window, batch)
	bkv.launch_d_kv(q, kv, temp, d_out, l[0], d[0], d_kv[0], window, batch)
	dev.synchronize()
	grid = ((seq + 127) // 128, h // (128 // hd), batch)
	_launch_groups(shim, fwd, grid, [seq, q, kv, sk, sv, temp, out[1], l[1], window])
	_launch_groups(shim, bq, grid, [seq, q, kv, sk, sv, temp, out[0], d_out, d_q[1], l[0], d[1], window])
	_launch_groups(shim, bkv, grid, [seq, q, kv, temp, d_out, l[0], d[0], d_kv[1], window])
	for name, pair in (("out", out), ("l", l), ("d_q", d_q), ("d", d), ("d_kv", d_kv)):
		a, b = (x.download() for x in pair)
		assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), name


@pytest.mark.parametrize("n,window,row_scales,threads", [
	(8, 256, False, 256), (8, 512, False, 512), (8, 4096, True, 1024),        # at most one workgroup per compute unit
	(9, 1040, False, 512), (9, 1024, True, 512), (32, 128, False, 256), (32, 1024, False, 256),
	(33, 128, True, 128), (33, 256, False, 128), (33, 528, False, 256), (33, 2048, False, 512),      # more than four
])
def test_decode_workgroup_widths(n, window, row_scales, threads):
	"""Every width the launcher picks (32 heads of 128, capacity 4096), ragged lengths including 0, 1 and the capacity:
	bit-equal to the oracle on sampled (sequence, head) slices."""
	from oracle import strict as S
	dev = X.Device(0)
	h, hd, cap = 32, 128, 4096
	rng = rng_for("decode widths", n, window, row_scales)
	lens = rng.integers(2, cap, n).astype(np.uint32)
	lens[:3] = 0, 1, cap
	q, sk, sv = i8_codes(rng, (n, h * hd)), i8_codes(rng, (h, hd)), i8_codes(rng, (h, hd))
	one = i8_codes(rng, (2, cap, 2 * h * hd))
	cache = one[np.arange(n) % 2]
	temp = (0.5 + rng.random(h)).astype(np.float32)
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)
	out, l = X.Tensor(dev, (n, h * hd), X.BF16 if row_scales else X.INT8), X.Tensor(dev, (n, h), X.F32)
	args = (t(q, X.INT8), t(cache, X.INT8), t(lens.view(np.float32), X.F32), t(sk, X.INT8), t(sv, X.INT8), t(temp, X.F32), out, l, window)
	if row_scales:
		qs, ks, vs = (0.125 * (0.75 + 0.5 * rng.random(s)).astype(np.float32) for s in ((n, h), (n, h, cap), (n, h, cap)))
		vw, sw, osc = recipes.attn_row_scale_operands(vs, X.BF16)
		kernel = recipes.attn_decode_row_scaled_kernel(dev, h, hd, cap, X.BF16, True)
		kernel.launch_row_scaled(*args, *(t(a, X.F32) for a in (qs, ks, vw, sw, osc)))
	else:
		kernel = recipes.attn_decode_kernel(dev, h, hd, cap, True)
		kernel.launch(*args)
	assert kernel.threads(n, window) == threads
	got, got_l = out.download(), l.download()
	seqs, heads = np.array([0, 1, 2, n - 1]), np.array([0, h - 1])
	cols = np.concatenate([np.arange(x * hd, (x + 1) * hd) for x in heads])
	kv_cols = np.concatenate([np.arange(x * 2 * hd, (x + 1) * 2 * hd) for x in heads])
	sub = (q[seqs][:, cols], cache[seqs][:, :, kv_cols], lens[seqs], sk[heads], sv[heads], temp[heads], len(heads), hd, window)
	sub = tuple(np.ascontiguousarray(a) if isinstance(a, np.ndarray) else a for a in sub)
	if row_scales:
		pick = lambda a: np.ascontiguousarray(a[seqs][:, heads])
		want, want_l = S.attn_decode_i8_row_scaled(*sub, pick(qs), pick(ks), pick(vw), sw[heads], osc[heads], out_bf16=True)
	else:
		want, want_l = S.attn_decode_i8(*sub)
	assert np.array_equal(got[seqs][:, cols], want)
	assert np.array_equal(got_l[seqs][:, heads].view(np.uint32), want_l.view(np.uint32))


# (kernel, K, raw columns, result per row, operand types): every writer, each operand mix
GEMM_FORMS = [
	("scale", lambda: recipes.attn_q_kernel(None, 512, 384), 512, 384),
	("geglu", lambda: recipes.ffn_f_kernel(None, 512, 384, True, X.E4M3), 512, 384),
	("geglu_i8_fast", lambda: recipes.ffn_f_kernel(None, 2048, 1024, False, X.INT8), 2048, 1024),
	("residual", lambda: recipes.attn_y_kernel(None, 192, 512, True, X.E4M3), 512, 384),
	("l2norm_32", lambda: recipes.attn_kv_kernel(None, 512, 384, 32), 512, 384),
	("l2norm_64", lambda: recipes.attn_kv_kernel(None, 512, 384, 64), 512, 384),
	("l2norm_128", lambda: recipes.attn_kv_kernel(None, 512, 512, 128), 512, 512),
	("dequant", lambda: recipes.dequant_gemm_kernel(None, 512, 384, X.INT8, X.INT8, False, True), 512, 384),
	("dequant_geglu", lambda: recipes.dequant_gemm_kernel(None, 512, 384, X.INT8, X.INT8, True, True), 512, 384),
	("qnorm", lambda: recipes.attn_q_norm_kernel(None, 512, 384, 64, 0.0), 512, 384),
	("qnorm_32", lambda: recipes.attn_q_norm_kernel(None, 512, 512, 32, 0.0), 512, 512),
	("qnorm_128", lambda: recipes.attn_q_norm_kernel(None, 512, 512, 128, 0.0), 512, 512),
	("qnorm_post", lambda: recipes.attn_q_norm_kernel(None, 512, 512, 64, 0.0, True, 1.0 / math.sqrt(512)), 512, 512),
	("qkv", lambda: recipes.attn_qkv_kernel(None, 512, 256, 384, 64), 512, 640),
	("qkv_32", lambda: recipes.attn_qkv_kernel(None, 512, 256, 512, 32), 512, 768),
	("qkv_128", lambda: recipes.attn_qkv_kernel(None, 512, 256, 512, 128), 512, 768),
	("mixed", lambda: recipes.mixed_gemm_kernel(None, 512, 384, False), 512, 384),
	("mixed_residual", lambda: recipes.ffn_y_kernel(None, 128, 512, True, X.E4M3, X.INT8), 512, 256),
	("e4m3", lambda: recipes.ffn_f_f8_kernel(None, 512, 256, True), 512, 256),
	# (the least K whose 256 x 256 tiles are blocks of 16 x 16, and an overhanging column tile)
	("e4m3", lambda: recipes.ffn_f_f8_kernel(None, 2048, 384, True), 2048, 384),
	("one_step", lambda: recipes.attn_q_kernel(None, 128, 256), 128, 256),
]


def _head_dim(name):
	"""The width of a head where the writer has any: "l2norm_32", "qkv_128"; 64 where the name has no number."""
	return next((int(part) for part in name.split("_") if part.isdigit()), 64)


def _oracle(name, k, n, q_cols, a, b, b_kv, residual, scales, learned):
	"""What the oracle gives for a launch of GEMM_FORMS, in the order of the launch's outputs."""
	from oracle import strict as S
	inp = 1.0 / math.sqrt(k) / 64.0
	if name in ("mixed", "mixed_residual", "e4m3"):
		acc = S.gemm_f32_seq(a, True, b, name == "e4m3")
		if name == "mixed":
			return [S.epilogue_scale(acc, 1.0 / math.sqrt(k) / 8.0, 8.0)]
		if name == "e4m3":
			return [S.epilogue_geglu(acc, 1.0 / math.sqrt(k), 1.0, S.STORE_E4M3)]
		return [S.epilogue_residual(acc, residual, math.sqrt(recipes.GELU_VAR_FIX_2 / k) / 8.0, 1.0, S.STORE_E4M3)]
	acc = S.gemm_i32(a, b)
	if name in ("scale", "one_step"):
		return [S.epilogue_scale(acc, inp, 8.0)]
	if name.startswith("geglu"):
		return [S.epilogue_geglu(acc, inp, 8.0 if name == "geglu_i8_fast" else 1.0, S.STORE_I8 if name == "geglu_i8_fast" else S.STORE_E4M3)]
	if name == "residual":
		return [S.epilogue_residual(acc, residual, inp, 1.0, S.STORE_E4M3)]
	if name.startswith("l2norm"):
		return list(S.epilogue_l2norm(acc, _head_dim(name), recipes.L2_NORM_EPS, inp, 8.0))
	if name.startswith("dequant"):
		return [S.epilogue_dequant(acc, *scales, name == "dequant_geglu")]
	if name.startswith("qnorm"):
		return [S.epilogue_qnorm(acc, _head_dim(name), 0.0, 8.0, learned, post_scale=1.0 / math.sqrt(k) if name == "qnorm_post" else 1.0)]
	kv, rrms = S.epilogue_l2norm(S.gemm_i32(a, b_kv), _head_dim(name), recipes.L2_NORM_EPS, inp, 8.0)
	return [S.epilogue_scale(acc, inp, 8.0), rrms, kv]


@pytest.mark.parametrize("name,make,k,n", GEMM_FORMS, ids=[f[0] for f in GEMM_FORMS])
@pytest.mark.parametrize("rows", [256, 320, 448, 2368])
def test_every_tile_size_gives_the_same_product(shim, name, make, k, n, rows):  # noqa: F811
	"""The 256 x 256 kernel against the oracle -- overhanging rows and columns moved back, every writer; launch() takes
	small tiles at these sizes -- and the 64 x 64 and 128 x 128 forms against it: the same bytes, also with e4m3
	operands, whose float32 sums every form adds in the same order.  (2368 rows: a partly filled band of tiles.)  The
	outputs hold another byte pattern before each launch."""
	dev = X.Device(0)
	rng = rng_for("tile sizes", name, rows)
	e4 = name in ("mixed", "mixed_residual", "e4m3")
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)
	a = e4m3_bytes(rng, (rows, k)) if e4 else i8_codes(rng, (rows, k))
	weights = lambda r: e4m3_bytes(rng, (r, k)) if name == "e4m3" else i8_codes(rng, (r, k))
	kernel = make()
	pairs = "geglu" in name or "residual" in name or name == "e4m3"
	out_cols, out_type = n // 2 if pairs else n, X.BF16 if "dequant" in name else X.E4M3 if pairs and name != "geglu_i8_fast" else X.INT8
	residual = i8_codes(rng, (rows, out_cols))
	scales = (0.01 + 0.01 * rng.random(rows)).astype(np.float32), (0.01 + 0.01 * rng.random(n)).astype(np.float32)
	learned = (16.0 * rng.standard_normal(n) if name == "qnorm_post" else rng.standard_normal(n)).astype(np.float32)
	learned = (learned.view(np.uint32) >> 16).astype(np.uint16)
	qkv = name.startswith("qkv")
	q_cols = 256 if qkv else n
	b, b_kv = weights(q_cols), weights(max(n - q_cols, 128))
	heads = (n - q_cols if qkv else n) // (2 * _head_dim(name))
	ta, tb, tb_kv = t(a, X.E4M3 if e4 else X.INT8), *(t(w, X.E4M3 if name == "e4m3" else X.INT8) for w in (b, b_kv))
	extras = t(residual, X.INT8), [t(v, X.F32) for v in scales], t(learned, X.BF16)
	results = {}
	base = os.path.join(_ffi.kernel_cache_dir(), kernel.name)
	for pattern, form in ((0x5A, ""), (0x3C, "s64x4"), (0xA7, "s128x4"), (0xC9, "s128x2")):
		if form == "s64x4" and k % 256 != 0:
			continue
		with open(os.path.join(base, form, "meta.json")) as f:
			meta = json.load(f)

		def poisoned(shape, dtype):
			size = {X.INT8: 1, X.E4M3: 1, X.BF16: 2, X.F32: 4}[dtype]
			return t(np.full(shape[:-1] + (shape[-1] * size,), pattern, np.uint8).view({1: np.uint8, 2: np.uint16, 4: np.float32}[size]), dtype)
		c = poisoned((rows, q_cols if qkv else out_cols), out_type)
		c_kv, rrms = poisoned((rows, max(n - q_cols, 128)), X.INT8), poisoned((rows, max(heads, 1)), X.F32)
		outputs = [c]
		slots = [ta, rows, tb, n, c]
		if name.startswith("l2norm"):
			slots.append(rrms)
			outputs.append(rrms)
		elif "residual" in name:
			slots.append(extras[0])
		elif "dequant" in name:
			slots.extend(extras[1])
		elif name.startswith("qnorm"):
			slots.append(extras[2])
		elif qkv:
			slots.extend([rrms, tb_kv, c_kv])
			outputs.extend([rrms, c_kv])
		dev.synchronize()
		tiles = -(-rows // meta["M_PER_BLOCK"]) * -(-n // meta["N_PER_BLOCK"])
		_launch(shim, os.path.join(base, form), meta, (tiles, 1, 1), slots)
		results[form] = [x.download() for x in outputs]
	for got, want in zip(results[""], _oracle(name, k, n, q_cols, a, b, b_kv, residual, scales, learned)):
		if not e4 and name != "geglu_i8_fast":
			assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), name
		elif out_type == X.E4M3:           # (the oracle adds f32 products one by one: another order, one step at most)
			differ, beyond = e4m3_compare(got, want)
			assert differ < 0.005 and beyond == 0.0, (name, differ, beyond)
		else:                              # likewise; hardware transcendentals: one code
			d = np.abs(got.astype(np.int32) - want.astype(np.int32))
			assert d.max() <= 1 and np.mean(d != 0) < 0.005, name
	for form, got in results.items():
		for x, y in zip(got, results[""]):
			assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (form, name)


def test_the_persistent_walk_over_more_tiles_than_workgroups(shim):  # noqa: F811
	"""The 256 x 256 kernel alone, whatever launch() takes at these sizes: 256 workgroups walk 260 tiles of K = 384 (three
	steps: every request of a tile's last two belongs to the workgroup's next tile), int8 and in the four-wavefront e4m3
	form, and 264 tiles through the L2-norm writer, whose rrms stores are in flight next to the next tile's loads.  e4m3 at K = 384 and
	the L2-norm writer at K = 256 are blocks of 32 x 32; at K = 2048 and 384 they are blocks of 16."""
	from oracle import strict as S
	dev = X.Device(0)
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)

	def launch(kernel, rows, n, slots):
		dev.synchronize()
		assert -(-rows // 256) * (n // 256) > 256
		_launch(shim, os.path.join(_ffi.kernel_cache_dir(), kernel.name), kernel.metadata, (256, 1, 1), slots)

	rng = rng_for("persistent walk")
	m, k, n = 256 * 65, 384, 1024
	a, b = i8_codes(rng, (m, k)), i8_codes(rng, (n, k))
	c = t(np.full((m, n), 0x5A, np.int8), X.INT8)
	launch(recipes.attn_q_kernel(None, k, n), m, n, [t(a, X.INT8), m, t(b, X.INT8), n, c])
	assert np.array_equal(c.download(), S.epilogue_scale(S.gemm_i32(a, b), 1.0 / math.sqrt(k) / 64.0, 8.0))

	m, n = 256 * 130, 512
	for k, every in ((384, 1), (2048, 5)):      # (the oracle's rows: all, or some of every tile)
		a8, b8 = e4m3_bytes(rng, (m, k)), e4m3_bytes(rng, (n, k))
		c = t(np.full((m, n // 2), 0x5A, np.uint8), X.E4M3)
		launch(recipes.ffn_f_f8_kernel(None, k, n, True), m, n, [t(a8, X.E4M3), m, t(b8, X.E4M3), n, c])
		want = S.epilogue_geglu(S.gemm_f32_seq(np.ascontiguousarray(a8[::every]), True, b8, True), 1.0 / math.sqrt(k), 1.0, S.STORE_E4M3)
		differ, beyond = e4m3_compare(c.download()[::every], want)
		assert differ < 5e-3 and beyond == 0.0, (k, differ, beyond)

	m, n = 256 * 33, 2048
	for k in (256, 384):
		a, b = i8_codes(rng, (m, k)), i8_codes(rng, (n, k))
		for hd in (64, 128):
			c, rrms = t(np.full((m, n), 0x5A, np.int8), X.INT8), t(np.full((m, n // (2 * hd)), 7.5, np.float32), X.F32)
			launch(recipes.attn_kv_kernel(None, k, n, hd), m, n, [t(a, X.INT8), m, t(b, X.INT8), n, c, rrms])
			want_c, want_r = S.epilogue_l2norm(S.gemm_i32(a, b), hd, recipes.L2_NORM_EPS, 1.0 / math.sqrt(k) / 64.0, 8.0)
			assert np.array_equal(c.download(), want_c) and np.array_equal(rrms.download().view(np.uint32), want_r.view(np.uint32)), (k, hd)


@pytest.mark.parametrize("name,make,out_type", [
	("e4m3 x e4m3", lambda dev: recipes.dequant_gemm_kernel(dev, 4096, 384, X.E4M3, X.E4M3, False, True), X.BF16),
	("e4m3 x int8", lambda dev: recipes.dequant_gemm_kernel(dev, 4096, 384, X.E4M3, X.INT8, False, True), X.BF16),
	("e4m3 x int8, residual", lambda dev: recipes.ffn_y_kernel(dev, 256, 4096, True), X.E4M3),
])
def test_a_row_of_an_e4m3_product_does_not_depend_on_the_rows_launched_with_it(name, make, out_type):
	"""float32 sums depend on their order: whatever tile size a launch takes, a token row's result is, byte for byte, what
	a large launch gives it.  Large and small values take turns along K, and its second half takes the first half's
	products away again, up to its last 128 columns, which are small: what the large partial sums lost to rounding shows
	in the result."""
	dev = X.Device(0)
	rng = rng_for("batch invariance", name)
	m, k, n = 16384, 4096, 512 if out_type == X.E4M3 else 384
	out_cols = n // 2 if out_type == X.E4M3 else n
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)
	a = e4m3_bytes(rng, (m, k), 0.05)
	a[:, :k // 2:2] = e4m3_bytes(rng, (m, k // 4), 200.0)
	w = e4m3_bytes(rng, (n, k)) if name == "e4m3 x e4m3" else i8_codes(rng, (n, k))
	half = k // 2 - 128
	a[:, k // 2:k - 128] = a[:, :half]
	w[:, k // 2:k - 128] = -w[:, :half] if w.dtype == np.int8 else np.where(w[:, :half] == 0, 0, w[:, :half] ^ 0x80)
	a[:, half:k // 2] = 0
	b = t(w, X.INT8 if w.dtype == np.int8 else X.E4M3)
	residual, rs, cs = i8_codes(rng, (m, out_cols)), (0.01 + 0.01 * rng.random(m)).astype(np.float32), (0.01 + 0.01 * rng.random(n)).astype(np.float32)
	kernel = make(dev)

	def launch(rows):
		c = X.Tensor(dev, (rows, out_cols), out_type)
		if out_type == X.E4M3:
			kernel.launch(t(a[:rows], X.E4M3), b, c, t(residual[:rows], X.INT8))
		else:
			kernel.launch_dequant(t(a[:rows], X.E4M3), b, c, t(rs[:rows], X.F32), t(cs, X.F32))
		return c.download()

	whole = launch(m)
	for rows in (256, 320, 448, 1024, 2368, 8192):
		assert np.array_equal(launch(rows), whole[:rows]), (name, rows)


@pytest.mark.parametrize("k", [256, 768, 1280])
@pytest.mark.parametrize("rows", [256, 320])
def test_weights_widened_once_per_workgroup(shim, k, rows):  # noqa: F811
	"""The 64 x 64 form of e4m3 x int8 at K steps (of 128 bytes) short of, equal to and past its rings of six, and with an
	overhanging token tile: the 256 x 256 kernel's bytes, and within a bf16 step (2^-8) plus float32 summation (K roundings
	of 2^-24 of the terms' magnitudes, in any order) of the product in 64 bits."""
	dev = X.Device(0)
	rng = rng_for("widened once", k, rows)
	n = 384
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)
	a, b = e4m3_bytes(rng, (rows, k)), i8_codes(rng, (n, k))
	rs, cs = (0.01 + 0.01 * rng.random(rows)).astype(np.float32), (0.01 + 0.01 * rng.random(n)).astype(np.float32)
	kernel = recipes.dequant_gemm_kernel(None, k, n, X.E4M3, X.INT8, False, True)
	ta, tb, trs, tcs = t(a, X.E4M3), t(b, X.INT8), t(rs, X.F32), t(cs, X.F32)
	results = []
	for form in ("", "s64x4"):
		path = os.path.join(_ffi.kernel_cache_dir(), kernel.name, form)
		with open(os.path.join(path, "meta.json")) as f:
			meta = json.load(f)
		c = t(np.full((rows, n), 0x5A5A, np.uint16), X.BF16)
		dev.synchronize()
		_launch(shim, path, meta, (-(-rows // meta["M_PER_BLOCK"]) * -(-n // meta["N_PER_BLOCK"]), 1, 1), [ta, rows, tb, n, c, trs, tcs])
		results.append(np.ascontiguousarray(c.download()).view(np.uint16))
	assert np.array_equal(results[0], results[1])
	values = np.zeros(a.shape)
	exponent, mantissa = (a >> 3 & 15).astype(np.int32), (a & 7).astype(np.float64)
	normal = exponent > 0
	values[normal] = ((1 + mantissa / 8) * np.exp2(exponent - 7))[normal]
	values[a >= 128] *= -1
	scale = rs[:, None].astype(np.float64) * cs
	want = values @ b.T.astype(np.float64) * scale
	magnitude = np.abs(values) @ np.abs(b.T.astype(np.float64)) * scale
	got = (results[1].astype(np.uint32) << 16).view(np.float32).reshape(rows, n)
	assert np.all(np.abs(got - want) <= np.abs(want) * 2.0 ** -8 + magnitude * k * 2.0 ** -24)


# (head_dim, heads, row scales, bf16 out, tokens, batch, window)
QUERY_WIDTHS = [
	(64, 8, True, True, 1024, 1, 256), (64, 8, False, False, 576, 2, 0), (64, 2, False, False, 192, 3, 16), (64, 2, True, False, 448, 1, 48),
	(32, 4, False, False, 768, 2, 64), (32, 4, True, False, 320, 1, 0),
	(128, 16, False, False, 256, 3, 512), (128, 2, False, False, 1088, 1, 112), (128, 2, True, True, 640, 2, 0), (128, 2, True, False, 128, 1, 0),
]


@pytest.mark.parametrize("hd,h,row_scales,out_bf16,seq,batch,window", QUERY_WIDTHS)
@pytest.mark.parametrize("spread", [0.25, 1.0, 3.0], ids=["flat", "gaussian", "peaked"])
def test_a_querys_attention_does_not_depend_on_the_queries_a_wavefront_takes(shim, hd, h, row_scales, out_bf16, seq, batch, window, spread):  # noqa: F811
	"""The speed build's two code objects give the same bytes, outputs and log-sum-exp: scores flat enough never to bring the
	accumulators down and peaked enough to do it many times, some heads at a negative temperature and one at zero."""
	dev = X.Device(0)
	rng = rng_for("query widths", hd, h, row_scales, seq, batch, window, spread)
	rows, width = seq * batch, h * hd
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)
	temp = ((0.5 + rng.random(h)) * spread).astype(np.float32)
	temp[0] = -temp[0]
	if h > 2:
		temp[2] = 0.0
	args = [t(i8_codes(rng, (rows, width)), X.INT8), t(i8_codes(rng, (rows, 2 * width)), X.INT8), t(i8_codes(rng, (h, hd)), X.INT8),
	        t(i8_codes(rng, (h, hd)), X.INT8), t(temp, X.F32)]
	tail = []
	if row_scales:
		kernel = recipes.attn_row_scaled_kernel(None, h, hd, X.BF16 if out_bf16 else X.INT8, False)
		qs, ks, vs = (0.125 * np.exp(0.5 * rng.standard_normal((h, rows))).astype(np.float32) for _ in range(3))
		tail = [t(a, X.F32) for a in (qs, ks, *recipes.attn_row_scale_operands(vs, X.BF16 if out_bf16 else X.INT8))]
	else:
		kernel = recipes.attn_kernel(None, h, hd, False)
	results = []
	for form in ("", "q16"):
		path = os.path.join(_ffi.kernel_cache_dir(), kernel.name, form)
		with open(os.path.join(path, "meta.json")) as f:
			meta = json.load(f)
		out, l = t(np.full((rows, width), 0x55, np.uint16 if out_bf16 else np.int8), X.BF16 if out_bf16 else X.INT8), t(np.full((h, rows), 7.0, np.float32), X.F32)
		dev.synchronize()
		_launch(shim, path, meta, (-(-seq // meta["Q_PER_BLOCK"]), h, batch), [seq, *args, out, l, window, *tail])
		results.append((np.ascontiguousarray(out.download()), l.download()))
	assert np.array_equal(results[0][1].view(np.uint32), results[1][1].view(np.uint32))
	assert np.array_equal(results[0][0].view(np.uint8), results[1][0].view(np.uint8))


@pytest.mark.parametrize("h,hd,row_scales", [(8, 64, True), (16, 128, False), (4, 32, False)])
def test_a_sequences_attention_does_not_depend_on_what_is_launched_with_it(h, hd, row_scales):
	"""One prompt alone, in a batch, and as the beginning of a longer sequence (causal: its tokens see the same keys): the same bytes,
	whichever code object the launches take."""
	dev = X.Device(0)
	rng = rng_for("launched with it", h, hd, row_scales)
	seq, window, many = 448, 128, 32
	width = h * hd
	q, kv = i8_codes(rng, (seq * many, width)), i8_codes(rng, (seq * many, 2 * width))
	sk, sv, temp = i8_codes(rng, (h, hd)), i8_codes(rng, (h, hd)), (0.5 + rng.random(h)).astype(np.float32)
	qs, ks, vw = (0.125 * (0.75 + 0.5 * rng.random((h, seq * many))).astype(np.float32) for _ in range(3))
	sw, osc = np.ones(h, np.float32), np.full(h, 0.125, np.float32)
	t = lambda a, dtype: X.Tensor.from_numpy(dev, np.ascontiguousarray(a), dtype)
	kernel = recipes.attn_row_scaled_kernel(dev, h, hd, X.BF16, False) if row_scales else recipes.attn_kernel(dev, h, hd, False)

	def launch(rows, batch):
		out, l = X.Tensor(dev, (rows, width), X.BF16 if row_scales else X.INT8), X.Tensor(dev, (h, rows), X.F32)
		args = (t(q[:rows], X.INT8), t(kv[:rows], X.INT8), t(sk, X.INT8), t(sv, X.INT8), t(temp, X.F32), out, l, window)
		if row_scales:
			kernel.launch_row_scaled(*args, *(t(a[:, :rows], X.F32) for a in (qs, ks, vw)), t(sw, X.F32), t(osc, X.F32), batch)
		else:
			kernel.launch(*args, batch)
		return np.ascontiguousarray(out.download()), l.download()
	alone = launch(seq, 1)
	widths = {kernel.queries_per_wavefront(seq, 1, window), kernel.queries_per_wavefront(seq, many, window), kernel.queries_per_wavefront(seq * many, 1, window)}
	assert widths == {16, 32}
	for rows, batch in ((seq * 3, 3), (seq * many, many), (seq * 2, 1), (seq * many, 1)):
		out, l = launch(rows, batch)
		assert np.array_equal(out[:seq].view(np.uint8), alone[0].view(np.uint8)), (rows, batch)
		assert np.array_equal(l[:, :seq].view(np.uint32), alone[1].view(np.uint32)), (rows, batch)
