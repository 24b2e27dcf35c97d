"""What this framework is used for, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what a program has in hand before the call (inputs, weights,
caches, output tensors on the GPU), `run` is one pass through the public entry points (`Block.forward`,
`GemmKernel.launch*`, `AttnKernel.launch*`, `AttnDecodeKernel.launch*`), and its outputs are the tensors that pass
wrote, seen in place.  Kernel configurations (widths, heads, element types) are those the benchmark and the tests of
this repository use, so that their code objects are built; rows, sequences, lengths and windows are free.

The paths, with the sizes their ranges span:
  block      the quantized transformer block forward: one chunk of 256 tokens ... 32768 tokens in a batch
  reference  the same block exactly as the reference's own configuration runs it (strict math, no window, 64 heads of 32)
  ffn        the feed-forward pair alone: int8, int8 with run-time scales and bf16 results, e4m3; 256 ... 16384 tokens
  prefill    attention over whole sequences, fixed scale or one scale per (row, head): 128 ... 65536 tokens
  decode     one token per sequence against its int8 cache: 1 ... 64 sequences, up to 4096 cached positions
  train      attention forward and both backward kernels: 128 ... 32768 tokens
"""
from __future__ import annotations

import functools
import math

import torch

import x17ai_amd as X
from x17ai_amd import recipes
from x17ai_amd.block import Block, BlockConfig


# ---------------------------------------------------------------- the cases

def _block(name, batch, seq):
	return {"name": name, "kind": "block", "batch": batch, "seq": seq, "window": 512}


def _ffn(name, form, rows):
	return {"name": name, "kind": "ffn", "form": form, "rows": rows}


def _prefill(name, heads, head_dim, batch, seq, window, row_scales):
	return {"name": name, "kind": "prefill", "heads": heads, "head_dim": head_dim, "batch": batch, "seq": seq,
	        "window": window, "row_scales": row_scales}


def _decode(name, sequences, window, ragged, row_scales):
	return {"name": name, "kind": "decode", "sequences": sequences, "window": window, "ragged": ragged, "row_scales": row_scales}


def _train(name, heads, head_dim, batch, seq, window):
	return {"name": name, "kind": "train", "heads": heads, "head_dim": head_dim, "batch": batch, "seq": seq, "window": window}


def listed():
	return [
		# a full batch of prompts through one block: the benchmark's headline
		_block("block_4x8192", 4, 8192),
		# one short prompt, or one step of a continuous batch: the time to first token is made of such passes
		_block("block_1x256", 1, 256),
		# a few medium prompts whose length is no multiple of any tile
		_block("block_3x1088", 3, 1088),
		# a user who runs the reference's block.config.json as it stands, bit-exact build
		{"name": "reference_16384", "kind": "reference", "seq": 16384},
		# weights and activations quantised per channel and per token at run time, bf16 results: the int8 feed-forward
		# network as other frameworks' int8 checkpoints need it
		_ffn("ffn_dequant_8192", "dequant", 8192),
		# the e4m3 feed-forward network of a wide model, a large batch of tokens ...
		_ffn("ffn_e4m3_16384", "e4m3", 16384),
		# ... and the few tokens of one serving step, where the weights are read for 320 rows only
		_ffn("ffn_e4m3_320", "e4m3", 320),
		# the smallest attention call: one sequence of 1024, quantised per row, bf16 out
		_prefill("prefill_1024", 8, 64, 1, 1024, 256, True),
		# the long-context prompt
		_prefill("prefill_65536", 32, 128, 1, 65536, 4096, True),
		# decoding a full batch against full caches, the cache as the row-scaled prefill leaves it
		_decode("decode_64", 64, 4096, False, True),
		# decoding for a few users whose caches have different fills, fixed-scale cache
		_decode("decode_3_ragged", 3, 4096, True, False),
		# one attention layer of a training step: forward, dQ, dK and dV
		_train("train_4x8192", 16, 128, 4, 8192, 512),
	]


def _log_uniform(rng, low, high):
	return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _tokens(rng, low, high):
	"""A token count between low and high, spread over its logarithm, in the path's granularity of 64."""
	return min(high, max(low, 64 * round(_log_uniform(rng, low, high) / 64)))


def draw(rng):
	kind = rng.choice(["block", "block", "ffn", "ffn", "prefill", "prefill", "decode", "decode", "train", "reference"])
	if kind == "block":
		batch = rng.choice([1, 2, 3, 4])
		c = _block("", batch, _tokens(rng, 256, 32768 // batch // 64 * 64))
		c["window"] = 16 * _log_uniform(rng, 4, 128)
	elif kind == "reference":
		c = {"kind": "reference", "seq": _tokens(rng, 256, 16384)}
	elif kind == "ffn":
		form = rng.choice(["int8", "dequant", "e4m3"])
		c = _ffn("", form, _tokens(rng, 256, 16384))
	elif kind == "prefill":
		heads, head_dim = rng.choice([(8, 64), (2, 128), (32, 128), (32, 128)])
		row_scales = rng.random() < 0.5
		batch = rng.choice([1, 1, 2, 5])
		seq = _tokens(rng, 128, 65536 // batch // 64 * 64)
		# no window (the whole past) up to a length where its cost stays within the range
		window = 0 if seq <= 8192 and rng.random() < 0.25 else 16 * _log_uniform(rng, 4, 256)
		c = _prefill("", heads, head_dim, batch, seq, window, row_scales)
	elif kind == "decode":
		c = _decode("", _log_uniform(rng, 1, 64), rng.choice([4096, 16 * _log_uniform(rng, 8, 256)]), rng.random() < 0.7, rng.random() < 0.5)
	else:
		heads, head_dim = rng.choice([(16, 128), (16, 128), (4, 128), (8, 64)])
		batch = rng.choice([1, 2, 4])
		c = _train("", heads, head_dim, batch, _tokens(rng, 128, 8192), 16 * _log_uniform(rng, 4, 32))
	c.pop("name", None)
	return c


# ---------------------------------------------------------------- sizes of the kernel configurations

# the block of the benchmark, and the reference's own (block.config.json)
BLOCK = dict(model_dim=2048, n_heads=16, head_dim=128, f_width=8192)
REFERENCE = dict(model_dim=2048, n_heads=64, head_dim=32, f_width=2048)
# (model width, inner width) of the feed-forward pairs
FFN = {"int8": (2048, 8192), "dequant": (2048, 8192), "e4m3": (4096, 16384)}
# heads, head_dim and capacity of the decode cache
DECODE = (32, 128, 4096)


# ---------------------------------------------------------------- what a program keeps for its lifetime

@functools.lru_cache(maxsize=None)
def _device():
	return X.Device(0)


@functools.lru_cache(maxsize=None)
def _kernel(make, *args):
	return make(_device(), *args)


@functools.lru_cache(maxsize=None)
def _block_object(kind, batch, window):
	if kind == "block":
		return Block(_device(), BlockConfig(**BLOCK, window_size=window, batch=batch, rms_norm_input=X.BF16, strict_math=False, fused_qkv=True))
	return Block(_device(), BlockConfig(**REFERENCE))


# ---------------------------------------------------------------- inputs

_TYPES = {X.INT8: ("|i1", torch.int8), X.E4M3: ("|u1", torch.float8_e4m3fn), X.BF16: ("<u2", torch.bfloat16), X.F32: ("<f4", torch.float32)}


class _Memory:
	"""A framework tensor's device memory, offered to torch without a copy; keeps the tensor alive."""

	def __init__(self, t):
		self.owner = t
		self.__cuda_array_interface__ = {"shape": t.shape, "typestr": _TYPES[t.dtype][0], "data": (t.device_ptr(), False), "version": 2}


def _view(t):
	v = torch.as_tensor(_Memory(t), device="cuda")
	return v if v.dtype == _TYPES[t.dtype][1] else v.view(_TYPES[t.dtype][1])


def _empty(shape, dtype):
	return X.Tensor(_device(), shape, dtype)


class _Draws:
	"""Seeded inputs in the number formats of the path, made on the GPU, at most 2^27 values at a time."""

	def __init__(self, seed):
		self.g = torch.Generator(device="cuda").manual_seed(seed)

	def _fill(self, t, values):
		_device().synchronize()          # the tensor's allocation is ordered on the framework's stream
		flat = _view(t).reshape(-1)
		for at in range(0, flat.numel(), 1 << 27):
			part = flat[at:at + (1 << 27)]
			part.copy_(values(part.numel()))
		return t

	def _normal(self, n):
		return torch.randn(n, generator=self.g, device="cuda")

	def _uniform(self, n, low, high):
		return torch.rand(n, generator=self.g, device="cuda").mul_(high - low).add_(low)

	def codes(self, shape):
		"""FixedI8 codes of N(0, 1) reals: 8 x, rounded, within +-127."""
		return self._fill(_empty(shape, X.INT8), lambda n: self._normal(n).mul_(8).round_().clamp_(-127, 127).to(torch.int8))

	def e4m3(self, shape):
		"""e4m3 of N(0, 1) reals in the path's dialect: no subnormals, no negative zero."""
		def values(n):
			v = self._normal(n)
			return torch.where(v.abs() < 2.0 ** -6, 0.0, v).to(torch.float8_e4m3fn)
		return self._fill(_empty(shape, X.E4M3), values)

	def bf16(self, shape):
		return self._fill(_empty(shape, X.BF16), lambda n: self._normal(n).to(torch.bfloat16))

	def f32(self, shape, low, high):
		return self._fill(_empty(shape, X.F32), lambda n: self._uniform(n, low, high))

	def lengths(self, n, capacity, ragged):
		def values(k):
			v = torch.randint(capacity // 8, capacity + 1, (k,), generator=self.g, device="cuda") if ragged else torch.full((k,), capacity, device="cuda")
			return v.to(torch.int32).view(torch.float32)
		return self._fill(_empty((n,), X.F32), values)      # u32 values in a 4-byte tensor, as the decode kernel takes them

	def value_scales(self, v_scale, heads):
		"""The row-scaled attention's operands for value scales around 1/8 (recipes.attn_row_scale_operands, bf16 output)."""
		v = _view(v_scale)
		ref = v.amax(dim=1) if v.dim() == 2 else v.amax(dim=(0, 2))
		sink, out = _empty((heads,), X.F32), _empty((heads,), X.F32)
		_device().synchronize()
		v.div_(ref[:, None])
		_view(sink).copy_(0.125 / ref)
		_view(out).copy_(ref)
		return v_scale, sink, out


def _sinks(d, heads, head_dim):
	return d.codes((heads, head_dim)), d.codes((heads, head_dim)), d.f32((heads,), 0.5, 1.5)


def prepare(case, seed):
	d = _Draws(seed)
	state = globals()["_prepare_" + case["kind"]](case, d)
	state["views"] = {k: _view(t) for k, t in state["outputs"].items()}
	torch.cuda.synchronize()
	return state


def _prepare_block(case, d):
	batch = case.get("batch", 1)
	block = _block_object(case["kind"], batch, case.get("window", 0))
	c = block.config
	rows = batch * case["seq"]
	sink_k, sink_v, temperature = _sinks(d, c.n_heads, c.head_dim)
	w = {
		"attn_q_weights": d.codes((c.attn_width, c.model_dim)), "attn_kv_weights": d.codes((2 * c.attn_width, c.model_dim)),
		"attn_y_weights": d.codes((2 * c.model_dim, c.attn_width)), "ffn_f_weights": d.codes((2 * c.f_width, c.model_dim)),
		"ffn_y_weights": d.codes((2 * c.model_dim, c.f_width)), "sinks_k": sink_k, "sinks_v": sink_v, "attn_temperature": temperature,
	}
	x = d.codes((rows, c.model_dim)) if c.rms_norm_input is None else d.bf16((rows, c.model_dim))
	outputs = block.new_outputs(rows)
	return {"pass": lambda: block.forward(x, w, outputs), "outputs": outputs}


_prepare_reference = _prepare_block


def _prepare_ffn(case, d):
	m, form = case["rows"], case["form"]
	width, inner = FFN[form]
	if form == "dequant":
		first = _kernel(recipes.dequant_gemm_kernel, width, 2 * inner, X.INT8, X.INT8, True, False)
		second = _kernel(recipes.dequant_gemm_kernel, inner, width, X.INT8, X.INT8, False, False)
		# the activations between the two are quantised by the caller: the second product has codes of its own
		x, w1, f, w2 = d.codes((m, width)), d.codes((2 * inner, width)), d.codes((m, inner)), d.codes((width, inner))
		rows, cols1, cols2 = (d.f32((n,), 0.01, 0.02) for n in (m, 2 * inner, width))
		h, y = _empty((m, inner), X.BF16), _empty((m, width), X.BF16)

		def one():
			first.launch_dequant(x, w1, h, rows, cols1)
			second.launch_dequant(f, w2, y, rows, cols2)
		return {"pass": one, "outputs": {"h": h, "y": y}}
	if form == "int8":
		first = _kernel(recipes.ffn_f_kernel, width, 2 * inner, False, X.INT8)
		second = _kernel(recipes.ffn_y_kernel, width, inner, False, X.INT8, X.INT8)
		x, w1, w2, f = d.codes((m, width)), d.codes((2 * inner, width)), d.codes((2 * width, inner)), _empty((m, inner), X.INT8)
		residual = x
	else:
		first = _kernel(recipes.ffn_f_f8_kernel, width, 2 * inner, False)
		second = _kernel(recipes.ffn_y_kernel, width, inner, False, X.E4M3, X.E4M3)
		x, w1, w2, f = d.e4m3((m, width)), d.e4m3((2 * inner, width)), d.e4m3((2 * width, inner)), _empty((m, inner), X.E4M3)
		residual = d.codes((m, width))
	y = _empty((m, width), X.E4M3)

	def one():
		first.launch(x, w1, f)
		second.launch(f, w2, y, residual)
	return {"pass": one, "outputs": {"f": f, "y": y}}


def _prepare_prefill(case, d):
	h, hd, batch, window = case["heads"], case["head_dim"], case["batch"], case["window"]
	rows = batch * case["seq"]
	q, kv = d.codes((rows, h * hd)), d.codes((rows, 2 * h * hd))
	sink_k, sink_v, temperature = _sinks(d, h, hd)
	l = _empty((h, rows), X.F32)
	if case["row_scales"]:
		kernel = _kernel(recipes.attn_row_scaled_kernel, h, hd, X.BF16, False)
		scales = (d.f32((h, rows), 0.09375, 0.15625), d.f32((h, rows), 0.09375, 0.15625), *d.value_scales(d.f32((h, rows), 0.09375, 0.15625), h))
		out = _empty((rows, h * hd), X.BF16)
		one = lambda: kernel.launch_row_scaled(q, kv, sink_k, sink_v, temperature, out, l, window, *scales, batch)
	else:
		kernel = _kernel(recipes.attn_kernel, h, hd, False)
		out = _empty((rows, h * hd), X.INT8)
		one = lambda: kernel.launch(q, kv, sink_k, sink_v, temperature, out, l, window, batch)
	return {"pass": one, "outputs": {"out": out, "l": l}}


def _prepare_decode(case, d):
	h, hd, capacity = DECODE
	n, window = case["sequences"], case["window"]
	q, cache = d.codes((n, h * hd)), d.codes((n, capacity, 2 * h * hd))
	lengths = d.lengths(n, capacity, case["ragged"])
	sink_k, sink_v, temperature = _sinks(d, h, hd)
	l = _empty((n, h), X.F32)
	if case["row_scales"]:
		kernel = _kernel(recipes.attn_decode_row_scaled_kernel, h, hd, capacity, X.BF16, False)
		scales = (d.f32((n, h), 0.09375, 0.15625), d.f32((n, h, capacity), 0.09375, 0.15625), *d.value_scales(d.f32((n, h, capacity), 0.09375, 0.15625), h))
		out = _empty((n, h * hd), X.BF16)
		one = lambda: kernel.launch_row_scaled(q, cache, lengths, sink_k, sink_v, temperature, out, l, window, *scales)
	else:
		kernel = _kernel(recipes.attn_decode_kernel, h, hd, capacity, False)
		out = _empty((n, h * hd), X.INT8)
		one = lambda: kernel.launch(q, cache, lengths, sink_k, sink_v, temperature, out, l, window)
	return {"pass": one, "outputs": {"out": out, "l": l}}


def _prepare_train(case, d):
	h, hd, batch, window = case["heads"], case["head_dim"], case["batch"], case["window"]
	rows = batch * case["seq"]
	forward, d_q_kernel, d_kv_kernel = (_kernel(make, h, hd, False) for make in (recipes.attn_kernel, recipes.attn_d_q_kernel, recipes.attn_d_kv_kernel))
	q, kv, d_out = d.codes((rows, h * hd)), d.codes((rows, 2 * h * hd)), d.bf16((rows, h * hd))
	sink_k, sink_v, temperature = _sinks(d, h, hd)
	out, l, dd = _empty((rows, h * hd), X.INT8), _empty((h, rows), X.F32), _empty((h, rows), X.F32)
	d_q, d_kv = _empty((rows, h * hd), X.BF16), _empty((rows, 2 * h * hd), X.BF16)

	def one():
		forward.launch(q, kv, sink_k, sink_v, temperature, out, l, window, batch)
		d_q_kernel.launch_d_q(q, kv, sink_k, sink_v, temperature, out, d_out, d_q, l, dd, window, batch)
		d_kv_kernel.launch_d_kv(q, kv, temperature, d_out, l, dd, d_kv, window, batch)
	return {"pass": one, "outputs": {"out": out, "l": l, "d": dd, "d_q": d_q, "d_kv": d_kv}}


def run(state):
	state["pass"]()
	return state["views"]


# ---------------------------------------------------------------- the work of one pass

def _pairs(seq, window):
	"""Visible (query, key) pairs of one sequence: query i sees keys max(0, i - window) .. i - 1, without the sink."""
	w = min(window, seq) if window else seq
	return w * (w - 1) // 2 + (seq - w) * w


def work(case):
	kind = case["kind"]
	if kind in ("block", "reference"):
		c = BLOCK if kind == "block" else REFERENCE
		d, a, f = c["model_dim"], c["n_heads"] * c["head_dim"], c["f_width"]
		batch, seq = case.get("batch", 1), case["seq"]
		m = batch * seq
		weights = 3 * a * d + 2 * d * a + 2 * f * d + 2 * d * f
		# x (bf16 residual stream and the FixedI8 x it becomes, or the FixedI8 x), q, kv, rrms, attention and l, the two y, f
		tokens = (3 * d if kind == "block" else d) + 3 * a + 4 * c["n_heads"] + a + 4 * c["n_heads"] + 2 * d + f
		flops = 2 * m * weights + 4 * a * batch * _pairs(seq, case.get("window", 0))
		return {"bytes": weights + m * tokens, "flops": flops}
	if kind == "ffn":
		m = case["rows"]
		d, f = FFN[case["form"]]
		if case["form"] == "dequant":
			return {"bytes": 3 * f * d + m * (d + 2 * f + f + 2 * d) + 4 * (m + 2 * f + d), "flops": 2 * m * 3 * f * d}
		residual = d if case["form"] == "e4m3" else 0
		return {"bytes": 4 * f * d + m * (d + f + residual + d), "flops": 2 * m * 4 * f * d}
	h, hd = DECODE[:2] if kind == "decode" else (case["heads"], case["head_dim"])
	a = h * hd
	if kind == "decode":
		# the keys of the window; of the values only the rows whose 8-bit probability is not zero, about one in a hundred
		# for normal keys and queries, which is not counted.  Mean fill of a ragged batch: 9/16 of the capacity.
		n, capacity = case["sequences"], DECODE[2]
		seen = n * min(case["window"], capacity * 9 // 16 if case["ragged"] else capacity)
		return {"bytes": seen * a + (4 * seen * h if case["row_scales"] else 0) + n * (a + (2 if case["row_scales"] else 1) * a + 4 * h), "flops": 2 * seen * a}
	m = case["batch"] * case["seq"]
	pairs = case["batch"] * _pairs(case["seq"], case["window"])
	if kind == "prefill":
		row = a + 2 * a + 4 * h + ((2 * a + 12 * h) if case["row_scales"] else a)
		return {"bytes": m * row, "flops": 4 * a * pairs}
	# forward: q, kv in, out, l; backward: dO in, d, dQ, dKV out; 2 + 3 + 4 products of the pairs with head_dim
	return {"bytes": m * (3 * a + a + 4 * h + 2 * a + 4 * h + 2 * a + 4 * a), "flops": 18 * a * pairs}


# ---------------------------------------------------------------- how far another correct implementation may be off

def tolerance(case):
	"""About four times what the two builds of each kernel (deterministic and hardware transcendentals) differ by on the
	same inputs, measured over the listed cases and some smaller ones; less where a bound of the format is lower.
	One step of e4m3 is at most 1/8 of the value, one of bf16 1/128."""
	kind = case["kind"]
	if kind == "block":
		# attention flips 0.08 % of its int8 codes by one; through the next product that moves attn_y by 1.4e-2 (2-norm),
		# one e4m3 step at most
		return {"rel": 0.03, "max": 0.13, "differ": 0.0035}
	if kind == "reference":
		# every integer and every int8 product is defined bit for bit; ffn_y sums e4m3 products in float32, in any order
		return {"rel": 2.5e-3, "max": 0.13, "differ": 0.0}
	if kind == "ffn":
		if case["form"] == "dequant":
			return {"rel": 1e-4, "max": 0.016}
		return {"rel": 2.5e-3, "max": 0.13, "differ": 5e-6}      # 5.7e-4, one step, 2.2e-7 of the int8 codes
	if kind == "prefill":
		return {"rel": 4e-3, "max": 0.08} if case["row_scales"] else {"rel": 1e-5, "differ": 0.0035}      # 1.0e-3, 0.02; 8e-4 of the codes
	if kind == "decode":
		return {"rel": 1e-4, "max": 0.016} if case["row_scales"] else {"rel": 1e-5, "differ": 0.001}
	# the same flips of 0.08 % of the forward's codes enter D = rowsum(dO o) and with it every gradient: 9.7e-3 (2-norm),
	# 0.78 of the root mean square in the worst element
	return {"rel": 0.03, "max": 0.95, "differ": 0.0035}
