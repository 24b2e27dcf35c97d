"""The further forms of a kernel (small GEMM tiles, decode widths) live inside its cache directory; the scans of the built
code objects hold for them too: no hazard around the hand-written requests, no packed single-precision arithmetic, no
scratch memory, no spilled registers."""
import glob
import os
import shutil

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
	for path in glob.glob(os.path.join(objects.KERNELS, "*", "*", "kernel.hsaco")):
		ins = scan._instructions(path, str(tmp_path))
		assert scan._hazards(ins) == [] and scan._m0_hazards(ins) == [], path
		assert [line for line in ins if scan.PACKED_F32.match(line)] == [], path
		with open(path, "rb") as f:
			kernel, = objects.kernel_metadata(objects.device_elf(f.read()))
		assert kernel[".private_segment_fixed_size"] == 0 and kernel[".vgpr_spill_count"] == 0, path
