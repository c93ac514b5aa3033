"""Masked keys start GEMM 1 at a value that no score brings back (masked_start in csrc/fmha_i8_kernel.hip): one unmasked key per batch
entry, with a score below those of all masked ones, which have the largest there is.  The output is that key's V row, exactly, on
every kernel; a start value in the wrong place, or one that a score can lift, gives another row or a mixture."""
import pytest

import routes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("full_range_p", [False, True], ids=["P_128_steps", "P_255_steps"])
@pytest.mark.parametrize("scale", [0.05, 30.0], ids=["scores_as_floats", "scores_converted"])
@pytest.mark.parametrize("S,d", [(256, 128), (256, 64), (320, 128), (320, 64), (300, 128), (429, 64)])  # blocks of 128 and 64 keys, ragged ends
@pytest.mark.parametrize("Sq", [33, 16])  # (the kernel of sixteen rows serves no more)
def test_the_only_unmasked_key_is_the_output(pkg, dev, Sq, S, d, scale, full_range_p):
    import torch
    # edges of quads, of the 32-key tiles of a matrix instruction and of the blocks
    keys = sorted({k for k in (0, 3, 4, 7, 8, 31, 32, 36, 63, 64, 95, 96, 127, 128, 191, 192, 255, 256, 287, S - 32, S - 2, S - 1) if k < S})
    B, H = len(keys), 2
    g = torch.Generator(device=dev)
    g.manual_seed(S + d)
    q = torch.full((B, H, Sq, d), 127, dtype=torch.int8, device=dev)
    k = torch.full((B, H, S, d), 127, dtype=torch.int8, device=dev)
    v = torch.randint(-127, 128, (B, H, S, d), generator=g, device=dev, dtype=torch.int8)
    mask = torch.ones((B, S), dtype=torch.int8, device=dev)
    for b, key in enumerate(keys):
        k[b, :, key] = -1  # (a masked key enters the row maximum as the integer -1000000: this score is above it)
        mask[b, key] = 0
    want = torch.stack([v[b, :, key] for b, key in enumerate(keys)])[:, :, None, :].expand(B, H, Sq, d).contiguous()
    print(Sq, S, d, scale, full_range_p, flush=True)
    routes.check_every_route(pkg, (q, k, v, mask), (scale, 1.0, 1.0, 1.0), want, full_range_p)
