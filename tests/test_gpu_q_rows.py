"""Q rows that pass through LDS on their way to the operands of GEMM 1 (head_dim 128): eight rows to a load, 32 to a wavefront, loads of the
last rows repeated past the end.  Every row must come out as it does in a call of its own, on every kernel, at counts of rows around
those units, in blocks of 64 and of 128 keys and over a single block; no access outside a tensor."""
import pytest

import routes

pytestmark = pytest.mark.gpu


def check_every_row(pkg, dev, Sq, S, full_range_p, masked_of):
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(Sq + S)
    q, k, v = (torch.randint(-127, 128, (2, 2, n, 128), generator=g, device=dev, dtype=torch.int8) for n in (Sq, S, S))
    mask = masked_of(g)
    scales = (0.2, 3.0, 3.0, 1.0)
    alone = {}
    for row in sorted({0, 1, 6, 7, 8, 15, 16, 30, 31, 32, 63, 64, 127, 128, 255, 256, Sq - 1}):
        if row < Sq:
            one = torch.empty((2, 2, 1, 128), dtype=torch.int8, device=dev)
            routes.attend(pkg, routes.library(pkg), routes.OWN_CHOICE, [q[:, :, row:row + 1].contiguous(), k, v, mask], scales, one, full_range_p)
            alone[row] = one[:, :, 0]
    for name in ("routed", "checked"):
        lib = routes.library(pkg, name)
        for rows, route in routes.routes_of(q, k):
            out = torch.full(q.shape, 77, dtype=torch.int8, device=dev)
            print(Sq, S, full_range_p, name, rows, flush=True)
            if routes.attend(pkg, lib, route, [q, k, v, mask], scales, out, full_range_p):
                for row, want in alone.items():
                    assert torch.equal(out[:, :, row], want), (name, rows, row)
        if name == "checked":
            assert lib.FMHAInferI8DebugOutOfBounds() == 0


@pytest.mark.parametrize("full_range_p", [False, True], ids=["P_128_steps", "P_255_steps"])
@pytest.mark.parametrize("first,end", [(0, 64), (0, 128), (64, 128), (128, 256), (0, 256)])
@pytest.mark.parametrize("Sq,S", [(33, 320), (65, 1024), (129, 704), (257, 1000)])
def test_blocks_without_unmasked_keys_in_front(pkg, dev, Sq, S, first, end, full_range_p):
    """The first or second key blocks wholly masked: no GEMM 1 waits for the rows there, and what lies in their place next comes soonest.  (One entry of
    two; the other one has keys masked here and there.)"""
    import torch

    def masked(g):
        mask = (torch.rand((2, S), generator=g, device=dev) < 0.2).to(torch.int8)
        mask[0, first:end] = 1
        return mask
    check_every_row(pkg, dev, Sq, S, full_range_p, masked)


@pytest.mark.parametrize("full_range_p", [False, True], ids=["P_128_steps", "P_255_steps"])
@pytest.mark.parametrize("S", [100, 320, 1000, 1024])
@pytest.mark.parametrize("Sq", [7, 9, 31, 33, 65, 129, 257])
def test_every_row_as_in_a_call_of_its_own(pkg, dev, Sq, S, full_range_p):
    import torch
    check_every_row(pkg, dev, Sq, S, full_range_p, lambda g: (torch.rand((2, S), generator=g, device=dev) < 0.2).to(torch.int8))
