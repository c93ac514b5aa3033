"""Calls served by two launches (pieces_of in csrc/fmha_i8_api.hip): the heads, or the rows of every head, that make full waves of large
workgroups, and the rest in smaller ones.  The same bytes as the kernel of 256-row workgroups writes for the whole call, nothing outside
the output, and no access outside a tensor."""
import ctypes as C

import pytest

import routes

pytestmark = pytest.mark.gpu

# (B, H, Sq, S, d, by): heads shared out within a batch entry and across them, rows that do not fill the last workgroup, both block
# sizes, ragged ends, queries and keys that differ in number
SHAPES = [
    (1, 24, 3200, 3200, 128, "heads"), (3, 8, 2922, 2922, 128, "heads"), (7, 4, 2560, 2560, 64, "heads"), (8, 12, 704, 704, 64, "heads"),
    (2, 48, 700, 1000, 128, "heads"), (4, 16, 2108, 2108, 64, "rows"), (7, 16, 537, 1500, 64, "rows"), (3, 32, 1472, 1472, 128, "heads"),
    (4, 20, 790, 1100, 128, "rows"),
]
# (B, H, Sq, S, d): 1 to 16 rows are left over, for the kernel of sixteen rows (d = 64, and d = 128 in blocks of 64 keys), with ragged ends too
FEW_LEFT = [(4, 16, 2049, 2049, 64), (2, 32, 2064, 2048, 64), (8, 8, 2056, 2500, 64), (4, 16, 2049, 1984, 128), (4, 16, 1040, 2111, 128), (8, 16, 513, 1030, 128)]


def launches(pkg, lib, shape):
    B, H, Sq, S, d = shape[:5]
    heads, rows = C.c_int(), C.c_int()
    lib.FMHAInferI8DebugLaunches.argtypes = [pkg.FMHACrossAttnDescriptor, C.c_void_p, C.c_void_p]
    count = lib.FMHAInferI8DebugLaunches(pkg.FMHACrossAttnDescriptor(B, Sq, S, H, d), C.addressof(heads), C.addressof(rows))
    return count, heads.value, rows.value


@pytest.mark.parametrize("full_range_p", [False, True], ids=["P_128_steps", "P_255_steps"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B%d_H%d_Sq%d_S%d_d%d_by_%s" % s)
def test_two_launches_write_what_one_writes(pkg, dev, shape, full_range_p):
    B, H, Sq, S, d, by = shape
    count, heads, rows = launches(pkg, routes.library(pkg), shape)
    assert count == 2 and (heads < B * H, rows < Sq) == (by == "heads", by == "rows"), (count, heads, rows)
    check(pkg, dev, shape, full_range_p)


@pytest.mark.parametrize("full_range_p", [False, True], ids=["P_128_steps", "P_255_steps"])
@pytest.mark.parametrize("shape", FEW_LEFT, ids=lambda s: "B%d_H%d_Sq%d_S%d_d%d" % s)
def test_few_rows_left_over(pkg, dev, shape, full_range_p):
    B, H, Sq, S, d = shape
    lib = routes.library(pkg)
    lib.FMHAInferI8DebugSecondKernel.argtypes = [pkg.FMHACrossAttnDescriptor]
    count, heads, rows = launches(pkg, lib, shape)
    assert count == 2 and heads == B * H and 1 <= Sq - rows <= 16 and lib.FMHAInferI8DebugSecondKernel(pkg.FMHACrossAttnDescriptor(B, Sq, S, H, d)) == routes.FEW
    check(pkg, dev, shape, full_range_p)


def check(pkg, dev, shape, full_range_p):
    import torch
    B, H, Sq, S, d = shape[:5]
    lib = routes.library(pkg)
    g = torch.Generator(device=dev)
    g.manual_seed(Sq)
    t = [torch.randint(-127, 128, (B, H, n, d), generator=g, device=dev, dtype=torch.int8) for n in (Sq, S, S)]
    t.append((torch.rand((B, S), generator=g, device=dev) < 0.2).to(torch.int8))
    scales = (0.5, 3.0, 3.0, 1.0)
    print(shape, full_range_p, flush=True)
    want = torch.empty_like(t[0])
    routes.attend(pkg, lib, routes.ROUTES[256], t, scales, want, full_range_p)
    n = want.numel()
    for name in ("routed", "checked"):
        lib = routes.library(pkg, name)
        o = torch.full((n + 256,), 77, dtype=torch.int8, device=dev)
        wide = torch.full((n + 256,), 3.0, dtype=torch.bfloat16, device=dev)
        routes.attend(pkg, lib, routes.OWN_CHOICE, t, scales, o, full_range_p)
        assert torch.equal(o[:n].view_as(want), want) and (o[n:] == 77).all(), name
        o.fill_(77)
        routes.attend(pkg, lib, routes.OWN_CHOICE, t, scales, o, full_range_p, wide)
        assert torch.equal(o[:n].view_as(want), want) and (o[n:] == 77).all(), name
        assert torch.equal(wide[:n].view_as(want), pkg.dequantize_tensor(want, 1.0, dtype=torch.bfloat16)) and (wide[n:] == 3).all(), name
    assert lib.FMHAInferI8DebugOutOfBounds() == 0
