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
