"""One problem on every kernel that can serve it.  The library chooses by size (row_groups_of in csrc/fmha_i8_api.hip), so the
small problems of the tests would leave the kernel of 256-row workgroups, the one behind the large calls, nearly unrun.
tests/bin/libfmha_i8_routed.so is the shipped library with FMHAInferI8DebugRoute, which makes that choice by hand."""
import ctypes as C
import os

HERE = os.path.dirname(os.path.abspath(__file__))
OWN_CHOICE, SHARED_OUT, ONE_LAUNCH = -1, -2, -3
ROUTES = {256: 0, 128: 4, 64: 2, 32: 1}  # query rows per workgroup -> FMHAInferI8DebugRoute
FEW = 16  # the kernel of sixteen rows: its rows, and its number there
_loaded = {}


def library(pkg, name="routed"):
    if name not in _loaded:
        path = os.path.join(HERE, "bin", "libfmha_i8_%s.so" % name)
        assert os.path.exists(path), "%s is not built; run `make -C tests`" % path
        lib = pkg.load_library(path)
        lib.FMHAInferI8DebugRoute.argtypes = [C.c_int]
        lib.FMHAInferI8DebugRoute.restype = None
        _loaded[name] = lib
    return _loaded[name]


def attend(pkg, lib, route, t, scales, o, full_range_p=False, wide=None):
    """One call with the tensors t = (q, k, v, mask) into o, on the kernel that `route` names; SHARED_OUT: False where the call
    cannot share its key blocks out.  wide: a float or bfloat16 output to write beside o."""
    import torch
    q, k = t[0], t[1]
    desc = pkg.FMHACrossAttnDescriptor(q.shape[0], q.shape[2], k.shape[2], q.shape[1], q.shape[3])
    args = [torch.cuda.current_stream(q.device).cuda_stream, pkg.FMHAParamI8(*scales, 1.0), desc] + [x.data_ptr() for x in t] + [o.data_ptr()]
    lib.FMHAInferI8DebugRoute(route)
    try:
        if wide is not None:
            st = lib.FMHAInferI8CrossToFloat(*args, full_range_p, wide.data_ptr(), wide.dtype == torch.bfloat16)
        elif route == SHARED_OUT:
            need = lib.FMHAInferI8CrossWorkspaceBytes(desc)
            if need == 0:
                return False
            work = torch.full((need + 256,), 0x7f, dtype=torch.int8, device=q.device)  # NaN as floats
            st = lib.FMHAInferI8CrossWithWorkspace(*args, full_range_p, work.data_ptr(), need)
            assert (work[need:] == 0x7f).all()
        else:
            st = (lib.FMHAInferI8CrossFullRangeP if full_range_p else lib.FMHAInferI8Cross)(*args)
    finally:
        lib.FMHAInferI8DebugRoute(OWN_CHOICE)
    assert st == pkg.FMHA_I8_OK, st
    return True


def routes_of(q, k):
    """Those that a call has: a single key block is the 256-row kernel's."""
    if k.shape[2] <= (128 if (k.shape[2] + 63) // 64 % 2 == 0 else 64):
        return [("rows 256", ROUTES[256])]
    return ([("rows %d" % rows, route) for rows, route in ROUTES.items()] + ([("rows 16", FEW)] if few_takes(q.shape[2], k.shape[2], k.shape[3]) else []) +
            ([("shared out", SHARED_OUT)] if q.shape[2] <= 32 else []))


def few_takes(rows, keys, d):
    """Whether fmha_i8_few_kernel serves such a call: not at d = 128 in blocks of 128 keys."""
    return rows <= FEW and not (d == 128 and (keys + 63) // 64 % 2 == 0)


def check_every_route(pkg, t, scales, want, full_range_p=False):
    """Every kernel writes the bytes that the shipped library wrote (`want`, on the GPU), and nothing behind them."""
    import torch
    lib = library(pkg)
    for name, route in routes_of(t[0], t[1]):
        o = torch.full((t[0].numel() + 256,), 77, dtype=torch.int8, device=t[0].device)
        if attend(pkg, lib, route, t, scales, o, full_range_p):
            got = o[:t[0].numel()].view(t[0].shape)
            assert (o[t[0].numel():] == 77).all() and torch.equal(got, want), (name, tuple(t[0].shape), t[1].shape[2], int((got != want).sum()))
