"""De-quantised outputs stored by whole rows (store_wide_rows in csrc/fmha_i8_kernel.hip): the kernels of 256 and 128 rows with rows that do
not fill a wavefront or a workgroup, masked-out entries, both float types; nothing outside the output, the int8 bytes as without it."""
import pytest

import routes

pytestmark = pytest.mark.gpu

# (B, H, Sq, S, d): one key block to many, both block sizes, 1 to 33 rows in the last wavefront, whole wavefronts without a row
SHAPES = [(1, 2, 1, 320, 128), (2, 3, 31, 128, 64), (1, 3, 33, 64, 128), (2, 2, 257, 1000, 64), (1, 5, 300, 576, 128), (1, 3, 513, 777, 64), (2, 2, 128, 2048, 128)]


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%d_H%d_Sq%d_S%d_d%d" % s)
def test_float_rows_are_the_dequantised_int8_rows(pkg, dev, shape, dtype):
    import torch
    B, H, Sq, S, d = shape
    g = torch.Generator(device=dev)
    g.manual_seed(Sq + S)
    t = [torch.randint(-127, 128, (B, H, n, d), generator=g, device=dev, dtype=torch.int8) for n in (Sq, S, S)]
    mask = (torch.rand((B, S), generator=g, device=dev) < 0.2).to(torch.int8)
    mask[1:2] = 1  # nothing to attend to: zeros
    t.append(mask)
    kind = getattr(torch, dtype)
    for scale, full_range_p in ((0.5, False), (8.0, False), (0.5, True)):
        scales = (scale, 3.0, 3.0, 0.7)
        want = torch.empty_like(t[0])
        print(shape, dtype, scale, full_range_p, flush=True)
        routes.attend(pkg, routes.library(pkg), routes.ROUTES[256], t, scales, want, full_range_p)
        n = want.numel()
        for name in ("routed", "checked"):
            lib = routes.library(pkg, name)
            for rows in (256, 128):
                o = torch.full((n + 256,), 77, dtype=torch.int8, device=dev)
                wide = torch.full((n + 256,), 3.0, dtype=kind, device=dev)
                routes.attend(pkg, lib, routes.ROUTES[rows], t, scales, o, full_range_p, wide)
                assert torch.equal(o[:n].view_as(want), want) and (o[n:] == 77).all(), (name, rows)
                assert torch.equal(wide[:n].view_as(want), pkg.dequantize_tensor(want, 0.7, dtype=kind)) and (wide[n:] == 3).all(), (name, rows)
        assert lib.FMHAInferI8DebugOutOfBounds() == 0


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("shape", [(1, 2, 32768, 128, 64), (3, 5, 4099, 31, 128), (16, 16, 2048, 100, 64), (16, 16, 2049, 100, 64)], ids=lambda s: "B%d_H%d_Sq%d_S%d_d%d" % s)
def test_float_flow_over_few_keys(pkg, dev, shape, dtype):
    """Over at most 128 keys the last of these is the first output of more than 32 M elements, which a second launch de-quantises."""
    import torch
    B, H, Sq, S, d = shape
    kind = getattr(torch, dtype)
    q, k, v = (torch.randn((B, H, n, d), device=dev).to(kind) for n in (Sq, S, S))
    mask = (torch.rand((B, S), device=dev) < 0.2).to(torch.int8)
    print(shape, dtype, flush=True)
    wide, o, amax = pkg.fmha_infer_from_float(q, k, v, mask, 0.7)
    want = pkg.fmha_infer_i8(*(pkg.quantize_tensor(x, a)[0] for x, a in zip((q, k, v), amax)), mask, *amax, o_amax=0.7)
    assert torch.equal(o, want) and wide.dtype == kind and torch.equal(wide, pkg.dequantize_tensor(o, 0.7, dtype=kind))
