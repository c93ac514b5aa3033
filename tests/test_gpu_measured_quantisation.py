"""FMHAMeasureAndQuantizeI8 (abs-max and quantisation of up to three tensors in one call) against the CPU checker, bit for
bit, at the edges of its two forms: one workgroup per tensor up to 32768 elements, two kernels above."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Tensor(C.Structure):
    _fields_ = [("x", C.c_void_p), ("out", C.c_void_p), ("n", C.c_longlong)]


@pytest.mark.parametrize("dtype_name", ["float32", "bfloat16"])
@pytest.mark.parametrize("sizes", [(1,), (32767,), (32768,), (32769,), (0, 7, 32768), (5, 40000, 1), (600011, 1000003, 262144)])
def test_measured_quantisation_of_several_tensors(pkg, orc, dev, sizes, dtype_name):
    import torch
    dtype = getattr(torch, dtype_name)
    rng = np.random.default_rng(sum(sizes))
    xs = [torch.from_numpy((0.5 * (i + 1) * rng.standard_t(3, n)).astype(np.float32)).to(dev).to(dtype) for i, n in enumerate(sizes)]
    if sizes[-1] > 3:
        xs[-1][3] = float("nan")  # skipped by the maximum, quantised to 0
    outs = [torch.full((n + 16,), 77, dtype=torch.int8, device=dev) for n in sizes]
    work = torch.full((1024,), 1e30, dtype=torch.float32, device=dev)  # its contents do not matter
    amax = torch.full((len(sizes),), -1.0, dtype=torch.float32, device=dev)
    note = torch.zeros(len(sizes), dtype=torch.int64, pin_memory=True)
    items = (Tensor * len(sizes))(*[Tensor(x.data_ptr(), o.data_ptr(), x.numel()) for x, o in zip(xs, outs)])
    lib = pkg.load_library()
    st = lib.FMHAMeasureAndQuantizeI8(None, C.addressof(items), len(sizes), 0 if dtype_name == "float32" else 1,
                                      work.data_ptr(), amax.data_ptr(), note.data_ptr(), 4711)
    torch.cuda.synchronize()
    assert st == pkg.FMHA_I8_OK
    for i, (x, o, n) in enumerate(zip(xs, outs, sizes)):
        wide = x.float().cpu().numpy()
        want = np.float32(np.nanmax(np.abs(wide))) if n else np.float32(0)
        assert amax[i].item() == want
        word = int(note[i].item())
        assert word >> 32 == 4711 and np.uint32(word & 0xffffffff).view(np.float32) == want
        got = o.cpu().numpy()
        if n:
            assert np.array_equal(got[:n], np.where(np.isnan(wide), 0, orc.quantize_i8(np.nan_to_num(wide), want)))
        assert (got[n:] == 77).all()


@pytest.mark.parametrize("dtype_name,n", [("float32", (1 << 26) + 5), ("bfloat16", (1 << 27) + 9)])
def test_inputs_larger_than_the_last_level_cache(pkg, dev, dtype_name, n):
    """256 MiB and a few elements: another variant of both kernels, the bytes of pieces that the ordinary one quantises."""
    import torch
    x = torch.randn(n, device=dev).to(getattr(torch, dtype_name))
    amax = x.abs().max().item()
    measured, a = pkg.quantize_tensor(x)
    given, _ = pkg.quantize_tensor(x, amax)
    assert a.item() == amax
    for at in range(0, n, 1 << 24):
        piece = pkg.quantize_tensor(x[at:at + (1 << 24)], amax)[0]
        assert torch.equal(piece, measured[at:at + (1 << 24)]) and torch.equal(piece, given[at:at + (1 << 24)])


def test_measured_quantisation_checks_its_arguments(pkg, dev):
    import torch
    x = torch.zeros(64, device=dev)
    o = torch.zeros(64, dtype=torch.int8, device=dev)
    w = torch.zeros(1024, device=dev)
    lib = pkg.load_library()

    def status(count=1, xp=x.data_ptr(), work=w.data_ptr()):
        items = (Tensor * 3)(*[Tensor(xp, o.data_ptr(), 64)] * 3)
        return lib.FMHAMeasureAndQuantizeI8(None, C.addressof(items), count, 0, work, w.data_ptr(), None, 0)

    assert status(count=0) == pkg.FMHA_I8_ERR_NULL_POINTER
    assert status(count=4) == pkg.FMHA_I8_ERR_NULL_POINTER
    assert status(xp=None) == pkg.FMHA_I8_ERR_NULL_POINTER
    assert status(work=None) == pkg.FMHA_I8_ERR_NULL_POINTER
    assert status(xp=x.data_ptr() + 4) == pkg.FMHA_I8_ERR_ALIGNMENT


def test_mixed_types_through_the_float_flow(pkg, dev):
    """fmha_infer_from_float takes Q, K and V of different float types: each is measured and quantised by its own type."""
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    q, k, v = (torch.randn((1, 2, 200, 64), generator=g, device=dev) for _ in range(3))
    k = k.bfloat16()
    mask = torch.zeros((1, 200), dtype=torch.int8, device=dev)
    o, o8, amax = pkg.fmha_infer_from_float(q, k, v, mask, 1.0)
    (q8, qa), (k8, ka), (v8, va) = (pkg.quantize_tensor(t) for t in (q, k, v))
    assert amax == (qa.item(), ka.item(), va.item()) and o.dtype == torch.float32
    assert torch.equal(o8, pkg.fmha_infer_i8(q8, k8, v8, mask, *amax, 1.0))
    with pytest.raises(ValueError):
        pkg.fmha_infer_from_float(q, torch.zeros_like(q), v, mask, 1.0)


@pytest.mark.parametrize("as_handle", [False, True], ids=["stream", "handle"])
def test_workspace_of_a_call_on_another_stream_is_not_handed_out_early(pkg, dev, as_handle):
    """quantize_tensor on a stream that is still busy: tensors that the current stream allocates and fills in the meantime must
    not be the call's workspace (they would put their values among its partial maxima)."""
    import torch
    x = torch.randn(1 << 20, device=dev)
    stream = torch.cuda.Stream()
    pkg.quantize_tensor(x)  # the current stream's pool has a block of the workspace's size
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(20):
            y = torch.randn(4096, 4096, device=dev) @ torch.ones(4096, 4096, device=dev)  # some milliseconds
    q, amax = pkg.quantize_tensor(x, stream=stream.cuda_stream if as_handle else stream)
    for _ in range(200):  # between the two kernels of the call, whenever they run
        fills = [torch.full((1024,), 1e30, device=dev) for _ in range(64)]
    torch.cuda.synchronize()
    assert amax.item() == x.abs().max().item()
    assert torch.equal(q, pkg.quantize_tensor(x)[0])
    del y, fills


# one shape per attention kernel and head size: 256, 128, 64 and 32 query rows per workgroup, rows that do not fill the last group,
# key blocks shared out over workgroups (the last two)
@pytest.mark.parametrize("out_type", ["float32", "bfloat16"])
@pytest.mark.parametrize("B,H,Sq,S,d", [(4, 20, 900, 200, 128), (4, 20, 900, 200, 64), (1, 9, 100, 60, 64), (2, 24, 250, 600, 128), (2, 24, 250, 600, 64),
                                        (1, 32, 300, 1536, 128), (1, 12, 450, 1536, 64), (1, 3, 129, 777, 128), (1, 3, 129, 777, 64),
                                        (1, 2, 3, 4096, 128), (1, 2, 3, 4096, 64)])
def test_float_output_is_the_dequantised_int8_output(pkg, dev, B, H, Sq, S, d, out_type):
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(11)
    q, k, v = (torch.randn((B, H, rows, d), generator=g, device=dev) for rows in (Sq, S, S))
    mask = (torch.rand((B, S), generator=g, device=dev) < 0.2).to(torch.int8)
    dtype = getattr(torch, out_type)
    print((B, H, Sq, S, d, out_type), flush=True)
    o, o8, amax = pkg.fmha_infer_from_float(q, k, v, mask, 0.7, out_dtype=dtype)
    assert o.dtype == dtype and torch.equal(o, pkg.dequantize_tensor(o8, 0.7, dtype=dtype))
    (q8, _), (k8, _), (v8, _) = (pkg.quantize_tensor(t) for t in (q, k, v))
    assert torch.equal(o8, pkg.fmha_infer_i8(q8, k8, v8, mask, *amax, 0.7))
    lib = pkg.load_library()  # nothing behind the last row; what is not a pointer it can store to is refused
    desc, scales = pkg.FMHACrossAttnDescriptor(B, Sq, S, H, d), pkg.FMHAParamI8(*amax, 0.7, 1.0)
    wide = torch.full((o.numel() + 256,), 3.0, dtype=dtype, device=dev)
    again = torch.empty_like(o8)
    call = lambda p: lib.FMHAInferI8CrossToFloat(None, scales, desc, *(t.data_ptr() for t in (q8, k8, v8, mask, again)), 0, p, out_type == "bfloat16")
    torch.cuda.synchronize()
    assert call(wide.data_ptr()) == 0 and call(None) == pkg.FMHA_I8_ERR_NULL_POINTER and call(wide.data_ptr() + 8) == pkg.FMHA_I8_ERR_ALIGNMENT
    torch.cuda.synchronize()
    assert torch.equal(wide[:o.numel()].view_as(o), o) and (wide[o.numel():] == 3).all() and torch.equal(again, o8)
