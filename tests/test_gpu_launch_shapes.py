"""Launch geometries that the operator layer's own launchers do not use but the kernels accept, driven through the raw
shim: attention grids with groups of heads per workgroup (src/device/cuda/attn.rs:60-66, 413-415: grid.y counts groups of
128 / head_dim heads) give the bytes of the one-head-per-workgroup launch, forward and backward."""
import ctypes
import os

import numpy as np
import pytest

import x17ai_amd as X
from x17ai_amd import _ffi, recipes
from tests.gpu_common import i8_codes, rng_for
from tests.test_gpu_shim import P, SZ, _ok, _value, shim  # noqa: F401  (shim is a fixture)

pytestmark = pytest.mark.gpu


def _launch_groups(shim, kernel, grid, slots):
	"""One launch of a built kernel's code object with `grid`, on a stream of its own."""
	meta = kernel.metadata
	ctx = _value(shim, shim.x17ai_hip_open_context(0))
	stream = _value(shim, shim.x17ai_hip_open_stream(ctx))
	module = _value(shim, shim.x17ai_hip_load_module(ctx, os.path.join(_ffi.kernel_cache_dir(), kernel.name, "kernel.hsaco").encode()))
	function = _value(shim, shim.x17ai_hip_get_kernel(module, b"kernel", meta["SMEM_BYTES"]))
	values = [ctypes.c_uint64(s.device_ptr() if isinstance(s, X.Tensor) else s) for s in slots]
	args = (P * len(values))(*[ctypes.cast(ctypes.byref(v), P) for v in values])
	_ok(shim, shim.x17ai_hip_launch_kernel(stream, function, *grid, meta["THREADS_PER_BLOCK"], 1, 1, meta["SMEM_BYTES"], args))
	_ok(shim, shim.x17ai_hip_synchronize(stream))
	_ok(shim, shim.x17ai_hip_del_module(module))
	_ok(shim, shim.x17ai_hip_close_stream(stream))
	_ok(shim, shim.x17ai_hip_close_context(ctx))


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


@pytest.mark.parametrize("n,window,row_scales", [
	(8, 256, False), (8, 4096, True),                                        # at most one workgroup per compute unit: 256 / 1024 threads
	(9, 1040, False), (9, 1024, True), (32, 512, False), (32, 1024, False),    # more: 512 / 256 / 256 / 256 threads
	(33, 512, True), (33, 528, False), (33, 2048, False),                     # ... than four per compute unit: 128 / 256 / 512
])
def test_decode_workgroup_widths(n, window, row_scales):
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
		recipes.attn_decode_row_scaled_kernel(dev, h, hd, cap, X.BF16, True).launch_row_scaled(*args, *(t(a, X.F32) for a in (qs, ks, vw, sw, osc)))
	else:
		recipes.attn_decode_kernel(dev, h, hd, cap, True).launch(*args)
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
