"""FMHAMeasureAndQuantizeI8 in one launch that holds its tensors (quantize_held_kernel): at the edges of its forms, with a workgroup
that waits for nobody, and beside a graph, which keeps the two launches.  The oracle is the quantisation by a given maximum, which
test_gpu_quant.py holds to the CPU checker, with torch's maximum."""
import ctypes as C

import pytest

import routes

pytestmark = pytest.mark.gpu

UNIT = {"float32": 4, "bfloat16": 8}  # elements of 16 bytes
# units that 256 workgroups hold: 512 threads with 1, 2, 4, 8, 12, 16, 20 and 25 each, 1024 with 16, 20 and 25
EDGES = [256 * 512 * n for n in (1, 2, 4, 8, 12, 16, 20, 25, 32, 40, 50)]


class Tensor(C.Structure):
    _fields_ = [("x", C.c_void_p), ("out", C.c_void_p), ("n", C.c_longlong)]


def check(pkg, lib, xs, amaxes=None):
    import torch
    outs = [torch.full((x.numel() + 16,), 77, dtype=torch.int8, device=x.device) for x in xs]
    work = torch.full((1024,), 1e30, device=xs[0].device)
    amax = torch.full((len(xs),), -1.0, device=xs[0].device)
    items = (Tensor * len(xs))(*[Tensor(x.data_ptr(), o.data_ptr(), x.numel()) for x, o in zip(xs, outs)])
    st = lib.FMHAMeasureAndQuantizeI8(torch.cuda.current_stream().cuda_stream, C.addressof(items), len(xs), int(xs[0].dtype == torch.bfloat16),
                                      work.data_ptr(), amax.data_ptr(), None, 0)
    assert st == pkg.FMHA_I8_OK
    for i, (x, o) in enumerate(zip(xs, outs)):
        want = x.float().nan_to_num(nan=0.0, posinf=float("inf"), neginf=float("-inf")).abs().max().item()
        assert amax[i].item() == want
        assert torch.equal(o[:x.numel()], pkg.quantize_tensor(x, want)[0])
        assert (o[x.numel():] == 77).all()


@pytest.mark.parametrize("patience", [5000, 0], ids=["waits", "reads_the_others_shares"])
@pytest.mark.parametrize("dtype_name", ["float32", "bfloat16"])
def test_edges_of_the_forms(pkg, dev, dtype_name, patience):
    import torch
    lib = routes.library(pkg)
    lib.FMHAQuantDebugPatience.argtypes = [C.c_uint]
    lib.FMHAQuantDebugPatience(patience)
    try:
        per = UNIT[dtype_name]
        sizes = [32769, 32768 + per] + [per * e + more for e in EDGES for more in (-1, 0, 1)]
        if patience == 0:  # (every workgroup reads every share)
            sizes = [n for n in sizes if n <= 5 << 20]
        for n in sizes:
            x = torch.randn(n, device=dev).to(getattr(torch, dtype_name))
            x[n - 1] = -9.5  # the maximum is in the elements behind the last unit
            print(dtype_name, patience, n, flush=True)
            check(pkg, lib, [x])
    finally:
        lib.FMHAQuantDebugPatience(5000)


@pytest.mark.parametrize("dtype_name", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["nan", "many_nan", "inf", "minus_inf_and_nan", "zero", "denormal", "large", "most_negative"])
def test_special_values(pkg, dev, kind, dtype_name):
    import torch
    for n in (40003, 1000003, 27 << 20):  # the last: two launches
        x = torch.randn(n, device=dev) * {"denormal": 1e-39, "large": 5e37, "zero": 0.0}.get(kind, 1.0)
        if kind == "nan":
            x[n // 3], x[n // 3 + 1] = float("nan"), -9.0
        elif kind == "many_nan":
            x[::97], x[5] = float("nan"), -50.0
        elif kind == "inf":
            x[n // 2] = float("inf")
        elif kind == "minus_inf_and_nan":
            x[n // 2], x[7] = float("-inf"), float("nan")
        elif kind == "most_negative":
            x[n - 2] = -77.0
        print(kind, dtype_name, n, flush=True)
        check(pkg, pkg.load_library(), [x.to(getattr(torch, dtype_name))])


def test_several_tensors_share_the_workgroups(pkg, dev):
    import torch
    for sizes in [(40000, 4, 100001), (1 << 20, 5 << 20, 33), (8 << 20, 8 << 20, 8 << 20), (2000003, 7, 26 << 20)]:
        for dtype in (torch.float32, torch.bfloat16):
            print(sizes, dtype, flush=True)
            check(pkg, pkg.load_library(), [torch.randn(n, device=dev).to(dtype) for n in sizes])


def test_a_captured_call_measures_what_it_finds_on_every_replay(pkg, dev):
    import torch
    x = torch.randn(300001, device=dev)
    pkg.quantize_tensor(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        q, amax = pkg.quantize_tensor(x)
    for i in range(4):
        x.copy_(torch.randn(300001, device=dev) * (4 - i))  # smaller every time: a maximum left by the replay before would be larger
        eager_q, eager_amax = pkg.quantize_tensor(x)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert amax.item() == eager_amax.item() == x.abs().max().item()
        assert torch.equal(q, eager_q)


def test_calls_on_several_streams_at_once(pkg, dev):
    import torch
    xs = [torch.randn(n, device=dev) * (i + 1) for i, n in enumerate((8 << 20, 24 << 20, 300001, 16 << 20))]
    streams = [torch.cuda.Stream() for _ in xs]
    want = [pkg.quantize_tensor(x, x.abs().max().item())[0] for x in xs]
    torch.cuda.synchronize()
    got = []
    for _ in range(5):
        for x, s in zip(xs, streams):
            with torch.cuda.stream(s):
                got.append(pkg.quantize_tensor(x))
    torch.cuda.synchronize()
    for i, (q, amax) in enumerate(got):
        assert amax.item() == xs[i % 4].abs().max().item() and torch.equal(q, want[i % 4])
