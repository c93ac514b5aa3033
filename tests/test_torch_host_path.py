"""The host path of the torch entry points (csrc/fmha_torch.cpp) on two GPUs that are host memory (fake_hip.cpp): which
device and stream the work is queued on, and which exceptions leave it.  One GPU cannot show the former, and no test fills a
real GPU's memory.  Each case runs in a process of its own, whose torch calls the stand-in runtime."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_call.restype = ctypes.c_char_p
fake.fake_memory_limit.argtypes = [ctypes.c_size_t]
import torch
sys.path.insert(0, %r)
import __graft_entry__ as g
pkg = g.load_package()
torch.cuda.init()
assert torch._C._cuda_getDeviceCount() == 2

def calls():
    out = []
    for i in range(fake.fake_calls()):
        device, stream = ctypes.c_int(), ctypes.c_void_p()
        name = fake.fake_call(i, ctypes.byref(device), ctypes.byref(stream)).decode()
        out.append((name, device.value, stream.value or 0))
    fake.fake_forget_calls()
    return out

def attention(device, sq=128, s=128, dtype=torch.int8):
    q = torch.empty((1, 2, sq, 64), dtype=dtype, device=device)
    k, v = (torch.empty((1, 2, s, 64), dtype=dtype, device=device) for _ in range(2))
    return q, k, v, torch.empty((1, s), dtype=torch.int8, device=device)
""" % ROOT


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", "-o", out,
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return out


def run(fake, code):
    p = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), fake], stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-4000:]


def test_work_is_queued_on_the_device_of_the_tensors(fake):
    """Tensors on GPU 1 while GPU 0 is current: the null stream means GPU 1's, whoever names it, and GPU 0 stays current."""
    run(fake, """
    entries = {
        "attend": lambda s: pkg.fmha_infer_i8(*attention("cuda:1"), 1.0, 1.0, 1.0, stream=s),
        "full range": lambda s: pkg.fmha_infer_i8(*attention("cuda:1"), 1.0, 1.0, 1.0, stream=s, full_range_p=True),
        "decode": lambda s: pkg.fmha_infer_i8(*attention("cuda:1", 1, 8192), 1.0, 1.0, 1.0, stream=s),
        "cross": lambda s: pkg.fmha_infer_i8(*attention("cuda:1", 256, 128), 1.0, 1.0, 1.0, stream=s),
        "quantize": lambda s: pkg.quantize_tensor(torch.empty(999, device="cuda:1"), stream=s),
        "quantize by": lambda s: pkg.quantize_tensor(torch.empty(999, device="cuda:1"), 2.0, stream=s),
        "dequantize": lambda s: pkg.dequantize_tensor(torch.empty(999, dtype=torch.int8, device="cuda:1"), 1.0, stream=s),
    }
    floats = {
        "float": lambda s: pkg.fmha_infer_from_float(*attention("cuda:1", dtype=torch.float32)[:3], attention("cuda:1")[3], 1.0, stream=s),
        "float, large": lambda s: pkg.fmha_infer_from_float(*attention("cuda:1", 1 << 15, 128, torch.bfloat16)[:3], attention("cuda:1")[3], 1.0, stream=s),
        "float, decode": lambda s: pkg.fmha_infer_from_float(*attention("cuda:1", 1, 8192, torch.float32)[:3], attention("cuda:1", 1, 8192)[3], 1.0, stream=s),
        "float, decode over fewer keys": lambda s: pkg.fmha_infer_from_float(*attention("cuda:1", 1, 656, torch.float32)[:3], attention("cuda:1", 1, 656)[3], 1.0, stream=s),
        "float, decode as bfloat16": lambda s: pkg.fmha_infer_from_float(*attention("cuda:1", 1, 8192, torch.bfloat16)[:3], attention("cuda:1", 1, 8192)[3], 1.0, stream=s),
    }
    side, null = torch.cuda.Stream("cuda:1"), torch.cuda.default_stream(1)
    seen, of_entry = set(), {}
    for name, entry in {**entries, **floats}.items():
        for stream in (None, null, side) + ((0, side.cuda_stream) if name in entries else ()):
            entry(stream)
            got = calls()
            handle = stream if isinstance(stream, int) else stream.cuda_stream if stream is not None else 0
            assert got and all(c[1:] == (1, handle) for c in got), (name, stream, got)
            assert torch.cuda.current_device() == 0 and fake.fake_current_device() == 0, name
            assert torch.cuda.current_stream(0) == torch.cuda.default_stream(0) and torch.cuda.current_stream(1) == null
            seen |= {c[0] for c in got}
            of_entry[name] = [c[0] for c in got]
    assert {"FMHAInferI8Status", "FMHAInferI8CrossFullRangeP", "FMHAInferI8CrossWithWorkspace", "FMHAInferI8CrossToFloat",
            "FMHAInferI8Cross", "FMHAMeasureAndQuantizeI8", "FMHAQuantizeI8", "FMHADequantizeI8", "FMHADequantizeI8BF16"} <= seen, seen
    # the attention de-quantises its output itself wherever no key blocks are shared out, over few keys and in decoding too
    assert of_entry["float"] == of_entry["float, large"] == of_entry["float, decode over fewer keys"] == ["FMHAMeasureAndQuantizeI8", "FMHAInferI8CrossToFloat"], of_entry
    with torch.cuda.device(1), torch.cuda.stream(side):  # and the other way round, with a current stream of its own
        pkg.fmha_infer_i8(*attention("cuda:0"), 1.0, 1.0, 1.0)
        pkg.fmha_infer_i8(*attention("cuda:1"), 1.0, 1.0, 1.0)
        assert [c[1:] for c in calls()] == [(0, 0), (1, side.cuda_stream)]
    """)


def test_memory_that_runs_out_is_an_out_of_memory_error(fake):
    """A caller that catches torch.OutOfMemoryError and shrinks its batch sees that type, as from torch's own functions; where a
    call merely works faster with memory (decoding's workspace) it goes on without."""
    run(fake, """
    MB = 1 << 20
    big = dict(sq=32 * MB // 128, s=128)  # 32 MB of int8 output: more than the rest of a cached segment
    i8, f32 = attention("cuda:0", **big), attention("cuda:0", **big, dtype=torch.float32)
    decode = attention("cuda:0", 32, 65536)  # (a workspace of 8.7 MB)
    out = torch.empty_like(decode[0])
    x, x8 = torch.empty(32 * MB, device="cuda:0"), torch.empty(32 * MB, dtype=torch.int8, device="cuda:0")
    entries = [
        lambda: pkg.fmha_infer_i8(*i8, 1.0, 1.0, 1.0),
        lambda: pkg.fmha_infer_from_float(*f32[:3], i8[3], 1.0),
        lambda: pkg.quantize_tensor(x),
        lambda: pkg.quantize_tensor(x, 1.0),
        lambda: pkg.dequantize_tensor(x8, 1.0),
    ]
    torch.cuda.empty_cache()
    fake.fake_forget_calls()
    fake.fake_memory_limit(0)
    for n, entry in enumerate(entries):
        try:
            entry()
        except torch.OutOfMemoryError as e:
            assert "out of memory" in str(e)
        else:
            raise AssertionError(n)
        assert not calls()
    pkg.fmha_infer_i8(*decode, 1.0, 1.0, 1.0, out=out)
    assert calls() == [("FMHAInferI8Cross", 0, 0)]
    fake.fake_memory_limit(1 << 30)
    for entry in entries:
        entry()
    pkg.fmha_infer_i8(*decode, 1.0, 1.0, 1.0, out=out)
    assert calls()[-1] == ("FMHAInferI8CrossWithWorkspace", 0, 0)
    """)


def test_a_moved_package_uses_the_library_beside_it(tmp_path):
    """The built package works from any folder, with the kernels of that folder."""
    at = str(tmp_path / "elsewhere")
    shutil.copytree(os.path.join(ROOT, "int8-flash-attention-fmha-quantization_amd"), at, ignore=shutil.ignore_patterns("csrc", "__pycache__"))
    code = """
import importlib.util, sys
spec = importlib.util.spec_from_file_location("moved", sys.argv[1] + "/__init__.py")
pkg = importlib.util.module_from_spec(spec)
spec.loader.exec_module(pkg)
pkg._load_native()
used = {line.split()[-1] for line in open("/proc/self/maps") if "fmha" in line}
assert used == {sys.argv[1] + "/libfmha_i8.so", sys.argv[1] + "/_fmha_torch.so"}, used
"""
    p = subprocess.run([sys.executable, "-c", code, at], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-4000:]


def test_build_without_torch(tmp_path):
    """C and C++ callers build the library where torch is not installed; the rest of build() goes through, compilers stubbed."""
    code = """
import subprocess, sys
sys.modules["torch"] = None  # import torch raises ModuleNotFoundError
sys.path.insert(0, sys.argv[1])
import __graft_entry__ as g
commands = []
def run(cmd, **kw):
    commands.append(cmd)
    return subprocess.CompletedProcess(cmd, 0, stdout="")
subprocess.run = run
g.build()
assert any("fmha_i8_api.hip" in " ".join(c) for c in commands)
assert not any("fmha_torch.cpp" in " ".join(c) for c in commands)
"""
    p = subprocess.run([sys.executable, "-c", code, ROOT], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-4000:]
