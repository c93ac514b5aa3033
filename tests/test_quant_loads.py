"""The quantisation kernel's non-temporal variant is chosen by size for its loads; a compiler that turns those into ordinary ones
leaves two names for one kernel, and no result shows it (it did, while the choice was an argument of the load instead of a
template parameter).  Host-side: needs hipcc, no GPU."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "int8-flash-attention-fmha-quantization_amd", "csrc", "fmha_quant.hip")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_loads_bypass_the_cache_where_the_variant_says_so(tmp_path):
    out = tmp_path / "quant.s"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-mllvm", "-amdgpu-mfma-vgpr-form=1", "-S", "--cuda-device-only", "-o", str(out), SRC],
                   check=True, capture_output=True)
    kernels = re.split(r"\n(?=_ZN14fmha_i8_gfx950[^\n]*:\s)", out.read_text())[1:]
    seen = {"ELb1E": 0, "ELb0E": 0}  # the variant with and the one without
    for text in kernels:
        name = text.split(":")[0]
        wide = re.findall(r"\bglobal_load_dwordx4\b.*", text)
        for variant in seen:
            if "18quantize_i8_kernel" in name and variant in name:
                seen[variant] += 1
                assert wide and any(" nt" in load for load in wide) == (variant == "ELb1E"), name
    assert seen == {"ELb1E": 2, "ELb0E": 2}  # float and bfloat16
