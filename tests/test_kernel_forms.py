"""The further forms of a kernel (small GEMM tiles, decode widths) live inside its cache directory; the scans of the built
code objects hold for them too: no hazard around the hand-written requests, no packed single-precision arithmetic, no
scratch memory, no spilled registers."""
import glob
import os
import shutil
import stat

import pytest

import x17ai_amd as X
from tests import test_code_objects as objects
from tests import test_kernel_hazards as scan
from x17ai_amd import recipes


@pytest.mark.skipif(not (os.path.exists(scan.BUNDLER) and os.path.exists(scan.OBJDUMP) and shutil.which("hipcc")), reason="needs the ROCm LLVM tools")
def test_forms_of_a_kernel_pass_the_code_object_scans(tmp_path):
	name = recipes.attn_q_kernel(None, 512, 384).name
	forms = [os.path.join(objects.KERNELS, name, form, "kernel.hsaco") for form in ("s64x4", "s128x4", "s128x2")]
	assert all(os.path.exists(f) for f in forms)
	for k in (1536, 2048, 2176):          # loops the compiler would unroll altogether, beyond a wavefront's 128 registers
		recipes.dequant_gemm_kernel(None, k, 256, X.E4M3, X.E4M3, False, True)
	names = {f: recipe().name for f, recipe in (("q16", lambda: recipes.attn_kernel(None, 2, 64, False)), ("s64x4", lambda: recipes.ffn_y_kernel(None, 128, 512, True, X.E4M3, X.INT8)))}
	scanned = glob.glob(os.path.join(objects.KERNELS, "*", "*", "kernel.hsaco"))
	assert all(os.path.join(objects.KERNELS, name, f, "kernel.hsaco") in scanned for f, name in names.items())      # 16 queries; weights widened once
	for path in scanned:
		ins = scan._instructions(path, str(tmp_path))
		assert scan._hazards(ins) == [] and scan._m0_hazards(ins) == [], path
		assert [line for line in ins if scan.PACKED_F32.match(line)] == [], path
		with open(path, "rb") as f:
			kernel, = objects.kernel_metadata(objects.device_elf(f.read()))
		assert kernel[".private_segment_fixed_size"] == 0 and kernel[".vgpr_spill_count"] == 0, path


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("make,picks", [
	# few tiles: the smallest form that covers the chip ...
	(lambda: recipes.attn_q_kernel(None, 2048, 2048), {256: "s64x4", 512: "s64x4", 4096: "s128x2", 32768: ""}),
	# (a tile more than a round of 256 x 256 begins another: 8192 rows fill one)
	(lambda: recipes.attn_q_kernel(None, 2048, 2048), {8192: "", 8320: "s128x2", 12288: ""}),
	(lambda: recipes.ffn_y_kernel(None, 2048, 8192, False), {256: "s64x4", 1024: "s128x2", 4096: "", 32768: ""}),
	(lambda: recipes.ffn_y_kernel(None, 4096, 16384, False, X.E4M3, X.E4M3), {320: "s128x4", 16384: ""}),
	# ... and with many of them the 256 x 256 kernel also where K is short: 131072 rows x 4096 columns, K = 512: 310 us and
	# 418 in the two-stage 128 x 128 form; 16384 x 4096 through the head-normalising writer, K = 256: 31 and 45
	(lambda: recipes.attn_q_kernel(None, 384, 1024), {256: "s128x2", 65536: "", 524288: ""}),
	(lambda: recipes.attn_kv_kernel(None, 256, 2048, 64), {256: "s64x4", 8192: "", 262144: ""}),
	# (short products of e4m3 operands in small tiles at any size: 16384 x 4096, K = 256, 46 us and 63 by the fitted code.  The GeGLU writer is
	# ahead of the fit: K = 384 40 us and 36)
	(lambda: recipes.ffn_f_f8_kernel(None, 384, 512, True), {256: "s128x2", 131072: "s128x2"}),
	# behind the first round of 256 x 256 tiles
	(lambda: recipes.ffn_f_f8_kernel(None, 4096, 32768, False), {320: "", 640: ""}),
	(lambda: recipes.ffn_f_kernel(None, 2048, 16384, False, X.E4M3), {1088: "", 2048: ""}),
	# there the writer decides (us of 256 x 256 / 128 x 128): GeGLU to eight bits, e4m3, K = 512, 16384 rows 73 / 86; plain dequantising,
	# e4m3, K = 768 63 / 41; int8, K = 128 47 / 35; residual, K = 1024 34 / 31; Scale, K = 256 22.8 / 20.3, K = 512 27 / 31
	(lambda: recipes.ffn_f_f8_kernel(None, 512, 8192, False), {16384: ""}),
	(lambda: recipes.dequant_gemm_kernel(None, 768, 2048, X.E4M3, X.E4M3, False, False), {16192: "s128x2"}),
	(lambda: recipes.dequant_gemm_kernel(None, 128, 8192, X.INT8, X.INT8, False, False), {4800: "s128x2"}),
	(lambda: recipes.attn_y_kernel(None, 1024, 1024, False), {9664: "s128x2"}),
	(lambda: recipes.attn_q_kernel(None, 256, 8192, False), {3968: "s128x2"}),
	(lambda: recipes.attn_q_kernel(None, 512, 8192, False), {4224: ""}),
	# (a band of the GeGLU writer's, too: 29 / 27 us)
	(lambda: recipes.ffn_f_kernel(None, 1024, 4096, False, X.E4M3), {4800: "s128x2"}),
], ids=["int8", "int8, past a round", "e4m3 x int8", "e4m3", "int8, short K", "L2 norm, short K", "e4m3, short K", "e4m3, second round", "int8, second round",
	"e4m3 GeGLU, K = 512", "e4m3 dequant, K = 768", "int8 dequant, K = 128", "int8 residual, K = 1024", "int8 scale, K = 256", "int8 scale, K = 512", "int8 GeGLU, K = 1024"])
def test_the_form_a_launch_takes(make, picks):
	kernel = make()
	assert {rows: kernel.form(rows) for rows in picks} == picks


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("k", [2048, 8192])
def test_widened_weights_pay_up_to_two_rounds_of_workgroups(k):
	kernel = recipes.ffn_y_kernel(None, 2048, k, k == 2048)
	assert {rows: kernel.form(rows) for rows in (256, 320, 512, 576)} == {256: "s64x4", 320: "s64x4", 512: "s64x4", 576: "s128x2"}


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("make,picks", [
	(lambda: recipes.attn_decode_kernel(None, 32, 128, 4096), {
		(1, 256): 256, (8, 256): 256, (8, 512): 512, (8, 4096): 1024,          # at most one workgroup per compute unit
		(9, 256): 256, (16, 1024): 512, (9, 0): 512,                           # up to two
		(32, 128): 256, (32, 1024): 256, (64, 128): 128, (48, 1024): 256, (64, 2048): 512, (64, 4096): 512}),
	# two wavefronts already stream at the memory's rate: 48 sequences 35 us, 37 on 256 threads
	(lambda: recipes.attn_decode_kernel(None, 2, 64, 4096), {(1, 4096): 1024, (384, 1024): 128, (384, 256): 256, (384, 4096): 512, (512, 4096): 128}),
], ids=["head_dim 128", "head_dim 64"])
def test_the_width_a_decode_launch_takes(make, picks):
	kernel = make()
	assert {key: kernel.threads(*key) for key in picks} == picks


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("make,picks", [
	# small launches: a head per workgroup fills the chip; large ones with short walks: the group saves its workgroup's start
	(lambda: recipes.attn_kernel(None, 8, 64, False), {(1024, 1, 256): 1, (4096, 8, 512): 1, (128, 128, 128): 2}),
	(lambda: recipes.attn_kernel(None, 64, 32), {(256, 1, 0): 1, (2048, 1, 0): 1, (128, 512, 128): 4}),
	(lambda: recipes.attn_d_q_kernel(None, 4, 32), {(1024, 1, 0): 1, (1024, 128, 64): 4}),
	# dK / dV, one workgroup per compute unit: 64 heads of 32, 16384 rows in sequences of 128 193 and 178 us
	(lambda: recipes.attn_d_kv_kernel(None, 4, 32), {(1024, 1, 0): 1, (128, 2048, 128): 4}),
	(lambda: recipes.attn_d_kv_kernel(None, 8, 64, False), {(1856, 2, 512): 1, (128, 512, 128): 2}),
	(lambda: recipes.attn_kernel(None, 16, 128, False), {(8192, 4, 512): 1}),
], ids=["forward 64", "forward 32", "dQ 32", "dK/dV 32", "dK/dV 64", "head_dim 128"])
def test_the_heads_a_workgroup_takes(make, picks):
	kernel = make()
	assert {key: kernel.heads_per_workgroup(*key) for key in picks} == picks


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("make,picks", [
	(lambda: recipes.attn_row_scaled_kernel(None, 8, 64, X.BF16, False), {(1024, 1, 256): 16, (2048, 1, 0): 16, (3072, 1, 256): 16, (3072, 1, 512): 32, (6144, 1, 128): 16, (6144, 1, 256): 32, (8192, 1, 64): 32}),
	(lambda: recipes.attn_kernel(None, 16, 128, False), {(256, 1, 512): 16, (1024, 1, 0): 16, (1536, 1, 64): 16, (1536, 1, 128): 32, (2048, 1, 64): 16, (8192, 4, 512): 32}),
	# the strict build has one order of operations; the backward kernels have no such form
	(lambda: recipes.attn_kernel(None, 2, 64, True), {(128, 1, 0): 32}),
	(lambda: recipes.attn_d_q_kernel(None, 4, 32), {(128, 1, 0): 32}),
], ids=["row scales 64", "head_dim 128", "strict", "dQ"])
def test_the_queries_a_wavefront_takes(make, picks):
	kernel = make()
	assert {key: kernel.queries_per_wavefront(*key) for key in picks} == picks


def _decode(): return recipes.attn_decode_kernel(None, 2, 64, 256)
def _gemm(): return recipes.attn_q_kernel(None, 512, 384)


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("make", [_gemm, _decode])
def test_the_forms_of_a_kernel_are_compiled_side_by_side(make, tmp_path, monkeypatch):
	"""A kernel is four compiler runs; a compiler that only notes when it starts and ends and sleeps in between."""
	script = tmp_path / "cc"
	script.write_text(f"#!/bin/bash\necho start >> {tmp_path}/log\nsleep 0.7\necho end >> {tmp_path}/log\n"
	                  "while [ $# -gt 0 ]; do [ \"$1\" = -o ] && touch \"$2\"; shift; done\n")
	script.chmod(script.stat().st_mode | stat.S_IXUSR)
	monkeypatch.setenv("X17AI_HIPCC", str(script))
	monkeypatch.setenv("X17AI_KERNEL_CACHE", str(tmp_path / "cache"))
	make()
	log = (tmp_path / "log").read_text().split()
	assert len(log) == 8 and log[:4] == ["start"] * 4, log


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
@pytest.mark.parametrize("make,source,marker,forms", [
	(_gemm, "gemm_b8_small.hip", '#include "common.h"', ("s64x4", "s128x4", "s128x2")),
	(_decode, "attn_decode_i8.hip", '#include "decode_tile.h"', ("t1024", "t512", "t256")),
])
def test_a_form_that_cannot_be_built_does_not_refuse_the_kernel(make, source, marker, forms, tmp_path, monkeypatch):
	"""Only the kernel itself has to compile: launches then take it at every size."""
	shutil.copytree(os.path.join(os.path.dirname(os.path.abspath(recipes.__file__)), "csrc", "kernels"), tmp_path / "kernels")
	path = tmp_path / "kernels" / source
	broken = "#if defined(X17_SMALL_TILE) || defined(X17_DECODE_THREADS) && X17_DECODE_THREADS > 128\n#error not this form\n#endif\n"
	path.write_text(path.read_text().replace(marker, marker + "\n" + broken, 1))
	monkeypatch.setenv("X17AI_KERNELS_DIR", str(tmp_path / "kernels"))
	monkeypatch.setenv("X17AI_KERNEL_CACHE", str(tmp_path / "cache"))
	kernel = make()
	assert all(f"form {f} is left out" in kernel.diagnostics for f in forms) and "not this form" in kernel.diagnostics
	assert kernel.form(256) == "" if make is _gemm else kernel.threads(1, 0) == 128
