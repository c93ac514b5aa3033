"""The attention kernels compiled with FMHA_CHECK_BOUNDS (tests/bin/libfmha_i8_checked.so, built by the tests' Makefile):
every global access is checked against the tensor - for K and V the head - it belongs to, and an access that would
leave it is counted and redirected instead of performed.  An out-of-bounds READ changes no result and, inside the pool
of a caching allocator, raises no fault either, so no other test can see one; this one does, without ever faulting.
(A key sequence shorter than one block was once fetched whole at the later issue points of the key loop: 0 results
changed, the GPU faulted only when the tensors happened to lie at the end of mapped memory.)"""
import ctypes as C

import numpy as np
import pytest

import fmha_cases as fc
import routes


def test_the_shipped_library_has_no_debug_entry_point(pkg):
    lib = pkg.load_library()
    assert not hasattr(lib, "FMHAInferI8DebugOutOfBounds") and not hasattr(lib, "FMHAInferI8DebugRoute")


@pytest.fixture(scope="module")
def checked(pkg):
    lib = routes.library(pkg, "checked")
    lib.FMHAInferI8DebugOutOfBounds.argtypes = []
    lib.FMHAInferI8DebugOutOfBounds.restype = C.c_int
    return lib


@pytest.mark.gpu
def test_checked_build_counts_nothing_on_any_shape(pkg, orc, checked, dev):
    """Every kernel on every shape it can serve, shared-out key blocks and their merge among them."""
    import torch
    served = {name: 0 for name in ["rows %d" % r for r in [*routes.ROUTES, routes.FEW]] + ["shared out"]}
    assert checked.FMHAInferI8DebugOutOfBounds() == 0  # (also clears the counter)
    rng = np.random.default_rng(77)
    shapes = [(3, 3, 319, 3, 64), (1, 1, 1, 1, 128), (2, 2, 70, 70, 128), (2, 1, 300, 129, 64), (1, 2, 64, 64, 64),
              (1, 2, 1024, 1024, 128), (2, 2, 2048, 2048, 64), (1, 1, 100, 4095, 128), (1, 1, 4097, 65, 64),
              (2, 1, 40, 15, 64), (2, 1, 40, 16, 128), (2, 1, 40, 17, 64), (2, 1, 40, 31, 128), (1, 1, 40, 4100, 64),
              # few query rows, whose key blocks can be shared out: whole and partly filled blocks and rounds, one to 32 rows
              (1, 2, 1, 2048, 128), (2, 3, 5, 1030, 64), (1, 1, 8, 1089, 64), (3, 4, 2, 1027, 128), (1, 2, 32, 4096, 128),
              (1, 3, 17, 5000, 64), (1, 2, 3, 1100, 128), (1, 1, 31, 513, 128), (1, 4, 7, 8300, 64), (2, 2, 1, 640, 128), (1, 1, 1, 320, 64),
              # at most sixteen, on the kernel for those
              (2, 2, 16, 129, 64), (1, 3, 15, 256, 64), (2, 1, 1, 1000, 64), (1, 2, 16, 3000, 64), (2, 2, 1, 65, 128), (1, 2, 16, 577, 128), (1, 3, 9, 1984, 128)]
    for _ in range(40):
        S = int(rng.choice([rng.integers(1, 130), rng.integers(1, 700), rng.integers(500, 2600), 64 * rng.integers(1, 40)]))
        Sq = S if rng.random() < 0.4 else int(rng.choice([rng.integers(1, 70), rng.integers(1, 600), rng.integers(200, 1500)]))
        shapes.append((int(rng.integers(1, 4)), int(rng.integers(1, 4)), Sq, S, int(rng.choice([64, 128]))))
    for n, (B, H, Sq, S, d) in enumerate(shapes):
        c = fc.make_inputs(B, H, (S + 63) // 64 * 64, d, pad=str(rng.choice(["none", "scatter"])), seed=300 + n)
        mask = c["mask"][:, :S].copy()
        if n % 3 == 0:
            mask[:, S // 2 + 1:] = 1  # trailing padding: fewer blocks than the length has
        mask[:, 0] = 0
        k, v = (np.ascontiguousarray(c[x][:, :, :S]) for x in ("k", "v"))
        q = fc.make_inputs(B, H, Sq, d, seed=700 + n)["q"]
        scales = (c["q_amax"], c["k_amax"], c["v_amax"], 1.0)
        t = [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in (q, k, v, mask)]
        for full in (False, True):  # the reference's P on 128 steps, and P on 255 steps
            want = orc.fmha_i8_blockwise_cross(q, k, v, mask, *scales, full_range_p=full)
            first = None
            for name, route in routes.routes_of(t[0], t[1]):
                print("shape", B, H, Sq, S, d, full, name, flush=True)
                o = torch.full((q.size + 256,), 77, dtype=torch.int8, device=dev)
                if not routes.attend(pkg, checked, route, t, scales, o, full):
                    continue
                assert checked.FMHAInferI8DebugOutOfBounds() == 0, (B, H, Sq, S, d, full, name)
                served[name] += 1
                if first is None:
                    first = o
                    st = fc.parity_stats(o[:q.size].view(t[0].shape).cpu().numpy(), want)
                    assert st["within1"] >= 0.999 and st["max"] <= 2, ((B, H, Sq, S, d, full), st)
                assert torch.equal(o, first), name
                if route != routes.SHARED_OUT:  # the float output beside it
                    dtype = torch.bfloat16 if n % 2 else torch.float32
                    wide = torch.full((q.size + 256,), 55.0, dtype=dtype, device=dev)
                    routes.attend(pkg, checked, route, t, scales, o, full, wide)
                    assert checked.FMHAInferI8DebugOutOfBounds() == 0, (B, H, Sq, S, d, full, name, "float output")
                    # (float)o / 127 * o_amax, in that order (o_amax is 1 here); numpy divides, torch multiplies by a reciprocal
                    exact = torch.from_numpy(first[:q.size].cpu().numpy().astype(np.float32) / np.float32(127)).to(dtype)
                    assert torch.equal(wide[:q.size].cpu(), exact) and (wide[q.size:] == 55).all() and torch.equal(o, first), name
    assert min(served.values()) >= 20, served
