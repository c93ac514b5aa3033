#!/usr/bin/env python3
"""Times one build of the library on one benchmark configuration (a measurement tool, not a test).

    make -C tests variants
    python tests/variant_timing.py --lib tests/bin/libfmha_i8_ko_softmax.so --workload C3
    rocprofv3 --pmc SQ_INSTS_VALU SQ_INSTS_SALU SQ_INSTS_LDS SQ_WAIT_ANY ... -- python3 tests/variant_timing.py --lib ... --calls 50

The test builds (tests/Makefile, target `variants`) each remove or change one thing in the attention kernel - no softmax,
no MFMA phase, no LDS operand reads, no tile loads, no LDS swizzle - so that what every piece costs can be re-measured;
their results are garbage on purpose, and only the build called `few` (the shipped kernel with fewer instantiations) and
`no_swizzle` are checked against the shipped library here.  With a `trace_ticks` build the per-wavefront time stamps
of the barriers are read back and summarised: how long a wavefront works between two barriers and how long it waits.

    python tests/variant_timing.py --kernel-costs
    python tests/variant_timing.py --shapes "1,16,2048,2048,128 1,16,1,8192,64"

The first measures what the library's choice of kernels rests on, each kernel on half and on all of the CUs with one
workgroup each, the second times
(B, H, Sq, S, d) on every kernel that can serve it and on the library's own choice; both print tables and use the build
called `routed`.
"""
import argparse
import ctypes as C
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))


def events_us(torch, call, calls):
    """Best of five bursts, at the settled clock."""
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < 0.04:
        for _ in range(20):
            call()
        torch.cuda.synchronize()
    best = 1e30
    for _ in range(5):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(calls):
            call()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) * 1e3 / calls)
    return best


def time_route(pkg, lib, routes, route, shape, calls=100):
    """Microseconds per call, or None where the call does not have that route.  No masked key, uniform random bytes."""
    import torch
    B, H, Sq, S, d = shape
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    t = [torch.randint(-127, 128, (B, H, rows, d), generator=g, device="cuda", dtype=torch.int8) for rows in (Sq, S, S)]
    t.append(torch.zeros((B, S), dtype=torch.int8, device="cuda"))
    o = torch.empty_like(t[0])
    desc = pkg.FMHACrossAttnDescriptor(B, Sq, S, H, d)
    args = [torch.cuda.current_stream().cuda_stream, pkg.FMHAParamI8(0.2, 3.0, 3.0, 1.0, 1.0), desc] + [x.data_ptr() for x in t] + [o.data_ptr(), 0]
    lib.FMHAInferI8DebugRoute(route)
    need = lib.FMHAInferI8CrossWorkspaceBytes(desc)
    work = torch.empty(max(need, 16), dtype=torch.int8, device="cuda")
    if route == routes.SHARED_OUT and need == 0:
        return None
    args += [work.data_ptr(), need]

    def call():
        if lib.FMHAInferI8CrossWithWorkspace(*args) != 0:
            raise RuntimeError("call refused")

    us = events_us(torch, call, calls)
    lib.FMHAInferI8DebugRoute(routes.OWN_CHOICE)
    return us


def time_shapes(shapes):
    import torch  # noqa: F401
    import __graft_entry__ as g
    import routes
    pkg = g.load_package()
    lib = routes.library(pkg)
    names = list(routes.ROUTES) + [routes.FEW]
    print("| B, H, Sq, S, d | %s | key blocks shared out | the library's choice |" % " | ".join("%d rows" % r for r in names))
    print("|" + "---|" * (len(names) + 3))
    for shape in shapes:
        us = [time_route(pkg, lib, routes, routes.ROUTES.get(r, routes.FEW), shape) if r != routes.FEW or routes.few_takes(*shape[2:]) else None for r in names]
        us += [time_route(pkg, lib, routes, route, shape) for route in (routes.SHARED_OUT, routes.OWN_CHOICE)]
        print("| %s | %s |" % (", ".join(map(str, shape)), " | ".join("-" if u is None else "%.2f" % u for u in us)), flush=True)


def two_launches(count):
    """Random shapes that the library serves by two launches: one launch by the kernel it would choose then, and the two."""
    import ctypes as C
    import math
    import random

    import torch  # noqa: F401
    import __graft_entry__ as g
    import routes
    pkg = g.load_package()
    lib = routes.library(pkg)
    lib.FMHAInferI8DebugLaunches.argtypes = [pkg.FMHACrossAttnDescriptor, C.c_void_p, C.c_void_p]
    rng, ratios, looked_at = random.Random(7), [], 0
    print("| B, H, Sq, S, d | first launch | one launch | two launches | two / one |")
    print("|" + "---|" * 5)
    while len(ratios) < count:
        B, H, S, d = rng.randint(1, 8), rng.choice((4, 8, 12, 16, 20, 24, 32, 48)), int(2 ** rng.uniform(8, 12)), rng.choice((64, 128))
        Sq = S if rng.random() < 0.6 else int(2 ** rng.uniform(8, 12))
        if B * H * ((Sq + 255) // 256) < 100 or B * H * Sq * S * d > 1 << 36:
            continue
        looked_at += 1
        heads, rows = C.c_int(), C.c_int()
        if lib.FMHAInferI8DebugLaunches(pkg.FMHACrossAttnDescriptor(B, Sq, S, H, d), C.addressof(heads), C.addressof(rows)) != 2:
            continue
        one, two = (time_route(pkg, lib, routes, route, (B, H, Sq, S, d), calls=40) for route in (routes.ONE_LAUNCH, routes.OWN_CHOICE))
        ratios.append(two / one)
        first = "%d of %d heads" % (heads.value, B * H) if heads.value < B * H else "%d rows" % rows.value
        print("| %d, %d, %d, %d, %d | %s | %.2f | %.2f | %.3f |" % (B, H, Sq, S, d, first, one, two, two / one), flush=True)
    ratios.sort()
    mean = math.exp(sum(math.log(r) for r in ratios) / len(ratios))
    print("\n%d of %d shapes take two launches; two / one: geometric mean %.3f, least %.3f, median %.3f, most %.3f" %
          (len(ratios), looked_at, mean, ratios[0], ratios[len(ratios) // 2], ratios[-1]))


def kernel_costs():
    """Time of a call against its key blocks, with one workgroup on half of the CUs and on each (8 or 16 heads of 16 workgroups)."""
    import torch  # noqa: F401
    import __graft_entry__ as g
    import routes
    pkg = g.load_package()
    lib = routes.library(pkg)
    keys = {64: (448, 960, 1984, 4032), 128: (512, 1024, 2048, 4096)}
    print("| d | keys per block | query rows | workgroups | us at %s | start + step * rounds, us |" % " / ".join("%d or %d keys" % p for p in zip(keys[64], keys[128])))
    print("|" + "---|" * 6)
    for d in (64, 128):
        for block in (64, 128):
            for rows, route in list(routes.ROUTES.items()) + ([(routes.FEW, routes.FEW)] if routes.few_takes(1, block, d) else []):
                for heads in (8, 16):
                    # (sixteen workgroups per head, or with sixteen rows one workgroup per head)
                    shape = (1, 16 * heads, 1) if rows == routes.FEW else (1, heads, 16 * rows)
                    us = [time_route(pkg, lib, routes, route, (*shape, s, d)) for s in keys[block]]
                    rounds = [(s // block + 3) // 4 if rows <= 64 else s // block for s in keys[block]]
                    step = (us[3] - us[0]) / (rounds[3] - rounds[0])
                    print("| %d | %d | %d | %d | %s | %.2f + %.3f |" % (d, block, rows, 16 * heads, " / ".join("%.2f" % u for u in us),
                                                                       us[0] - step * rounds[0], step), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--lib", default=None, help="library to time (default: the shipped libfmha_i8.so)")
    ap.add_argument("--workload", default="C3", choices=["C1", "C2", "C3", "C4", "C5"])
    ap.add_argument("--calls", type=int, default=1000)
    ap.add_argument("--preheat-ms", type=float, default=100.0)
    ap.add_argument("--compare", action="store_true", help="compare the output bytes with the shipped library's")
    ap.add_argument("--kernel-costs", action="store_true", help="each kernel's time against the number of key blocks")
    ap.add_argument("--two-launches", type=int, default=0, help="this many random shapes that take two launches, against one launch")
    ap.add_argument("--shapes", default=None, help="\"B,H,Sq,S,d B,H,Sq,S,d ...\" on every kernel")
    args = ap.parse_args()
    if args.kernel_costs:
        return kernel_costs()
    if args.two_launches:
        return two_launches(args.two_launches)
    if args.shapes:
        return time_shapes([tuple(int(x) for x in shape.split(",")) for shape in args.shapes.split()])

    import numpy as np
    import torch
    import __graft_entry__ as g
    import fmha_cases as fc

    pkg = g.load_package()
    shipped = pkg.load_library()
    path = os.path.abspath(args.lib) if args.lib else None
    lib = C.CDLL(path) if path else shipped
    lib.FMHAInferI8Status.argtypes = [C.c_void_p, pkg.FMHAParamI8, pkg.AttnDataDescriptor] + [C.c_void_p] * 5 + [C.c_bool]
    lib.FMHAInferI8Status.restype = C.c_int
    dev = torch.device("cuda:0")
    c = fc.make_config(args.workload)
    B, H, S, d = c["q"].shape
    q, k, v, m = (torch.from_numpy(c[n]).to(dev) for n in ("q", "k", "v", "mask"))
    o = torch.zeros_like(q)
    P = pkg.FMHAParamI8(c["q_amax"], c["k_amax"], c["v_amax"], c["o_amax"], 1.0)
    A = pkg.AttnDataDescriptor(B, S, H, d)
    stream = torch.cuda.current_stream(dev)
    call = (stream.cuda_stream, P, A, q.data_ptr(), k.data_ptr(), v.data_ptr(), m.data_ptr(), o.data_ptr(), True)

    def step():
        st = lib.FMHAInferI8Status(*call)
        if st != 0:
            raise RuntimeError("status %d" % st)

    t0 = time.perf_counter()
    heat = 0
    while (time.perf_counter() - t0) * 1e3 < args.preheat_ms:
        for _ in range(200):
            step()
        torch.cuda.synchronize()
        heat += 200
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for _ in range(args.calls):
        step()
    e1.record(stream)
    torch.cuda.synchronize()
    us = e0.elapsed_time(e1) * 1e3 / args.calls
    out = {"lib": os.path.relpath(path, ROOT) if path else "shipped", "workload": args.workload, "calls": args.calls,
           "preheat_calls": heat, "us_per_call": round(us, 3),
           "pct_of_int8_peak": round(4.0 * B * H * S * S * d / (us * 1e-6) / 5033.2e12 * 100, 2)}
    if args.compare:
        got = o.cpu().numpy()
        ref = torch.zeros_like(q)
        rc = list(call)
        rc[7] = ref.data_ptr()
        assert shipped.FMHAInferI8Status(*rc) == 0
        torch.cuda.synchronize()
        out["bytes_differing_from_shipped"] = int((got != ref.cpu().numpy()).sum())
    if hasattr(lib, "FMHAInferI8DebugReadTrace"):
        nwg = min(4096, B * H * ((S + 255) // 256))
        buf = (C.c_uint * (nwg * 8 * 64))()
        lib.FMHAInferI8DebugReadTrace.argtypes = [C.c_void_p, C.c_int]
        assert lib.FMHAInferI8DebugReadTrace(buf, nwg * 8 * 64) == 0
        t = np.frombuffer(buf, dtype=np.uint32).reshape(nwg, 8, 64).astype(np.int64)
        work, wait = [[], []], [[], []]
        cycles = ticks = 0
        for wg in range(nwg):
            for w in range(8):
                x = t[wg, w, :62]
                n = int(np.argmax(x == 0)) if (x == 0).any() else 62
                if n >= 2 and n < 62:  # (a full stamp register has lost its last stamp)
                    cycles += int((x[n - 1] - x[0]) & 0xffffffff)
                    ticks += int((t[wg, w, 63] - t[wg, w, 62]) & 0xffffffff)
                dx = np.diff(x[:n]) & 0xffffffff  # start | (arrive, leave)* | end
                if len(dx) > 12:
                    wait[w // 4].append(dx[1::2][3:-3])
                    work[w // 4].append(dx[2::2][3:-3])
        for grp, name in ((0, "wavefronts 0-3"), (1, "wavefronts 4-7")):
            if not work[grp]:  # too few key blocks for a steady state
                continue
            wk, wt = np.concatenate(work[grp]), np.concatenate(wait[grp])
            out["ticks_" + name.replace(" ", "_")] = {
                "work_between_barriers_mean": round(float(wk.mean()), 1), "wait_at_barrier_mean": round(float(wt.mean()), 1),
                "work_even_ticks_mean": round(float(np.concatenate([a[0::2] for a in work[grp]]).mean()), 1),
                "work_odd_ticks_mean": round(float(np.concatenate([a[1::2] for a in work[grp]]).mean()), 1)}
        out["tick_unit"] = "s_memtime counts, steady-state ticks only (first and last three dropped)"
        if ticks:
            out["shader_mhz_inside_the_kernel"] = round(100.0 * cycles / ticks, 1)  # s_memtime counts per 10 ns
            out["wavefront_lifetime_cycles_mean"] = round(cycles / (nwg * 8.0), 1)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
