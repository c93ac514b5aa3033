"""Calls of at most sixteen query rows per head (fmha_i8_few_kernel, alone and with shared-out key blocks): the bytes that the kernel of
256-row workgroups writes, nothing outside the output or the workspace, no access outside a tensor."""
import re
import shutil
import subprocess

import pytest

import routes
from test_gpu_split_kernel import CSRC

# (B, H, Sq, S, d): one round of four key blocks to many, rounds that are not full, both block sizes, ragged ends, 1 to 16 rows, mask
# rows of more than one classification pass; d128 in blocks of 128 keys is served with shared-out blocks alone
SHAPES = [
    (2, 3, 1, 129, 64), (1, 2, 16, 256, 64), (2, 2, 15, 1100, 64), (1, 3, 5, 8300, 64), (3, 2, 2, 65, 64), (2, 3, 16, 1000, 64), (40, 8, 3, 448, 64), (8, 16, 1, 2048, 64),
    (2, 3, 1, 65, 128), (1, 2, 16, 320, 128), (2, 2, 7, 1984, 128), (1, 3, 16, 8240, 128), (40, 8, 1, 700, 128),
    (2, 2, 1, 513, 128), (1, 3, 16, 2048, 128), (2, 1, 9, 8190, 128),
]


def build(pkg, dev, shape, pad, seed):
    import torch
    B, H, Sq, S, d = shape
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    t = [torch.randint(-127, 128, (B, H, n, d), generator=g, device=dev, dtype=torch.int8) for n in (Sq, S, S)]
    mask = (torch.rand((B, S), generator=g, device=dev) < (0.2 if pad == "scatter" else 0.0)).to(torch.int8)
    if pad == "dead":  # whole blocks without an unmasked key, at the end and inside; one batch entry with none at all
        mask[:, S - S // 3:] = 1
        mask[:, S // 8:S // 8 + 260] = 1
        mask[:, 0] = 0
        mask[1:2] = 1
    return t + [mask]


@pytest.mark.gpu
@pytest.mark.parametrize("full_range_p", [False, True], ids=["P_128_steps", "P_255_steps"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%d_H%d_Sq%d_S%d_d%d" % s)
def test_same_bytes_as_the_kernel_of_256_row_workgroups(pkg, dev, shape, full_range_p):
    import torch
    B, H, Sq, S, d = shape
    # scores read as floats; converted scores; an output scale that rules out the one-fma merge
    for n, (scale, o_amax, pad) in enumerate([(0.2, 1.0, "scatter"), (8.0, 1.0, "none"), (0.2, 0.02, "dead")]):
        t = build(pkg, dev, shape, pad, 31 * Sq + n)
        scales = (scale, 3.0, 3.0, o_amax)
        want = torch.empty_like(t[0])
        print(shape, full_range_p, pad, flush=True)
        routes.attend(pkg, routes.library(pkg), routes.ROUTES[256], t, scales, want, full_range_p)
        size = want.numel()
        for name in ("routed", "checked"):
            lib = routes.library(pkg, name)
            for route in (routes.FEW, routes.SHARED_OUT):
                o = torch.full((size + 256,), 77, dtype=torch.int8, device=dev)
                if routes.attend(pkg, lib, route, t, scales, o, full_range_p):
                    assert torch.equal(o[:size].view_as(want), want) and (o[size:] == 77).all(), (name, route, pad)
            for dtype in (torch.bfloat16, torch.float32):  # beside the de-quantised output
                o = torch.full((size + 256,), 77, dtype=torch.int8, device=dev)
                wide = torch.full((size + 256,), 3.0, dtype=dtype, device=dev)
                routes.attend(pkg, lib, routes.FEW, t, scales, o, full_range_p, wide)
                assert torch.equal(o[:size].view_as(want), want) and (o[size:] == 77).all(), (name, dtype, pad)
                assert torch.equal(wide[:size].view_as(want), pkg.dequantize_tensor(want, o_amax, dtype=dtype)) and (wide[size:] == 3).all(), (name, pad)
        assert lib.FMHAInferI8DebugOutOfBounds() == 0


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_no_read_of_an_asynchronously_loaded_register_before_its_wait(tmp_path):
    """The same check as for the other kernels (test_kernel_async_loads.py), on this one."""
    from test_kernel_async_loads import _check_function
    args = ["128, 64, true, true, false, false", "64, 64, false, false, true, false", "64, 128, false, true, false, false", "128, 128, true, true, true, true"]
    src = tmp_path / "few.hip"
    src.write_text("".join('#include "%s/fmha_i8_%skernel.hip"\n' % (CSRC, k) for k in ("", "split_", "few_")) + "namespace fmha_i8_gfx950 {\n" +
                   "".join("template __global__ void fmha_i8_few_kernel<%s>(SplitKernelArgs);\n" % a for a in args) + "}\n")
    out = tmp_path / "few.s"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-mllvm",
                    "-amdgpu-mfma-vgpr-form=1", "-S", "--cuda-device-only", "-o", str(out), str(src)], check=True, capture_output=True)
    funcs = re.split(r"\n(?=_ZN14fmha_i8_gfx950\d+fmha_i8_few_kernel[^\n]*:\s)", out.read_text())[1:]
    assert len(funcs) == len(args)
    for f in funcs:
        assert _check_function(f.split(":")[0], f) >= 4  # mask bytes (twice) and the Q rows
