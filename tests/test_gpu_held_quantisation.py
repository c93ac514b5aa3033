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
@pytest.mark.parametrize("kind", ["nan", "many_nan", "inf", "minus_inf_and_nan", "zero", "denormal", "large", "most_negative", "nan_but_one"])
def test_special_values(pkg, dev, kind, dtype_name):
    import torch
    for n in (40003, 1000003, (27 if dtype_name == "float32" else 53) << 20):  # the last: two launches
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
        elif kind == "nan_but_one":  # all shares but one have nothing else
            x.fill_(float("nan"))
            x[n // 2] = -3.0
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


@pytest.fixture
def patience(pkg):
    """Sets how long workgroups of the test build wait for each other, in ticks of 10 ns."""
    lib = routes.library(pkg)
    lib.FMHAQuantDebugPatience.argtypes = [C.c_uint]
    yield lib.FMHAQuantDebugPatience
    lib.FMHAQuantDebugPatience(1000)


@pytest.mark.parametrize("dtype_name", ["float32", "bfloat16"])
def test_whoever_measures_a_share_leaves_the_same_bits(pkg, dev, patience, dtype_name):
    """With little patience a share is measured by its own workgroup and by others, which all write the two words of its slot: were
    the maxima not the same bits, a reader could put halves of two together.  The largest value is in the last unit, which
    workgroups read again where their share ends before their threads do."""
    import torch
    lib, per = routes.library(pkg), UNIT[dtype_name]
    for e in EDGES:
        for n in (per * e - 1, per * (e - 7777)):
            x = torch.randn(n, device=dev).to(getattr(torch, dtype_name))
            x[n - per] = -9.517
            for ticks in (0, 60, 150, 400):
                patience(ticks)
                print(dtype_name, n, ticks, flush=True)
                check(pkg, lib, [x])


def call_us(pkg, lib, x, calls):
    import torch
    out = torch.empty(x.numel(), dtype=torch.int8, device=x.device)
    work, amax = torch.empty(1100, device=x.device), torch.empty(1, device=x.device)
    item = Tensor(x.data_ptr(), out.data_ptr(), x.numel())
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(calls):
        assert lib.FMHAMeasureAndQuantizeI8(torch.cuda.current_stream().cuda_stream, C.addressof(item), 1, 0, work.data_ptr(), amax.data_ptr(), None, 0) == 0
    e1.record()
    torch.cuda.synchronize()
    assert amax.item() == x.abs().max().item()
    return e0.elapsed_time(e1) * 1e3 / calls


def test_workgroups_without_patience_share_the_reading(pkg, dev, patience):
    """Where every workgroup finds most of the others missing, they read the input about once more between them (2.4 times the
    call's time), not once each (over a hundred times)."""
    import torch
    lib, x = routes.library(pkg), torch.randn(8 << 20, device=dev)
    patience(1000)
    waits = min(call_us(pkg, lib, x, 20) for _ in range(3))
    patience(0)
    reads = min(call_us(pkg, lib, x, 20) for _ in range(3))
    print(waits, reads, flush=True)
    assert reads <= 10 * waits, (waits, reads)


def test_beside_a_kernel_that_holds_half_of_the_compute_units(pkg, dev, patience):
    """A kernel of another stream on 128 compute units for half a millisecond: the call goes through beside it (66 us; 810 when every
    workgroup read the share of every one that was missing)."""
    import time

    import torch
    lib = routes.library(pkg)
    patience(1000)
    t = [torch.randint(-127, 128, (1, 128, rows, 128), device=dev, dtype=torch.int8) for rows in (256, 32768, 32768)]
    t += [torch.zeros((1, 32768), dtype=torch.int8, device=dev), torch.empty((1, 128, 256, 128), dtype=torch.int8, device=dev)]
    x, other = torch.randn(16 << 20, device=dev), torch.cuda.Stream()
    beside, alone = [], []
    lib.FMHAInferI8DebugRoute(routes.ROUTES[256])
    try:
        for _ in range(6):
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(other)
            assert lib.FMHAInferI8Cross(other.cuda_stream, pkg.FMHAParamI8(0.2, 3.0, 3.0, 1.0, 1.0), pkg.FMHACrossAttnDescriptor(1, 256, 32768, 128, 128),
                                        *[y.data_ptr() for y in t]) == 0
            e1.record(other)
            since = time.perf_counter()
            while time.perf_counter() - since < 60e-6:  # it has begun
                pass
            beside.append(call_us(pkg, lib, x, 1))
            alone.append(e0.elapsed_time(e1) * 1e3)
    finally:
        lib.FMHAInferI8DebugRoute(routes.OWN_CHOICE)
    print(beside, alone, flush=True)
    assert sorted(beside)[3] <= 250, (beside, alone)
