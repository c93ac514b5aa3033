"""The attention kernels load the mask bytes and the Q rows with inline-assembly loads whose results arrive
asynchronously, and retire them with explicit `s_waitcnt vmcnt(n)` that count the loads still allowed in flight.  The
compiler knows nothing of that protocol: were it to copy or read one of those registers between the load and its wait
(it did once, when the wait was written into two branches), it would read stale data without any error.  This test
compiles the kernels to assembly and checks, for every instantiation, that no instruction touches an asynchronously
loaded register before a wait that is strict enough to have retired the load.  Host-side: needs hipcc, no GPU."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "int8-flash-attention-fmha-quantization_amd", "csrc", "fmha_i8_api.hip")

WAIT = re.compile(r"\s+s_waitcnt\b.*vmcnt\((\d+)\)")


def _regs(line):
    used = set(int(x) for x in re.findall(r"\bv(\d+)\b", line))
    for a, b in re.findall(r"v\[(\d+):(\d+)\]", line):
        used |= set(range(int(a), int(b) + 1))
    return used


def _start_assembly(path, *extra):
    return subprocess.Popen(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                             "-packed-fp32-ops", "-mllvm", "-amdgpu-mfma-vgpr-form=1", "-S", "--cuda-device-only", *extra,
                             "-o", path, SRC], stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)


def _functions(path):
    funcs = re.split(r"\n(?=_ZN14fmha_i8_gfx950\d+fmha_i8_(?:fwd|split|pair)_kernel[^\n]*:\s)", open(path).read())[1:]
    # (head size, block size, two arithmetic variants, P range) for each kernel, and ragged ends (256 rows), row groups 1 and 2
    # (split); the shared-out form has one arithmetic variant less
    assert [sum(k in f.split(":")[0] for f in funcs) for k in ("fwd", "split", "pair")] == [64, 64 + 16, 32]
    return funcs


@pytest.fixture(scope="module")
def assembly_files(tmp_path_factory):
    """Every instantiation as shipped, and with contraction switched off on the command line."""
    at = tmp_path_factory.mktemp("asm")
    paths = str(at / "kernel.s"), str(at / "kernel_off.s")
    compilers = [_start_assembly(paths[0]), _start_assembly(paths[1], "-ffp-contract=off")]
    assert [c.wait() for c in compilers] == [0, 0]
    return paths


@pytest.fixture(scope="module")
def assembly(assembly_files):
    return [_functions(p) for p in assembly_files]


@pytest.fixture(scope="module")
def kernels(assembly):
    return assembly[0]


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_compiler_fuses_no_multiply_add_on_its_own(assembly):
    """The source pins floating-point contraction off and writes out every fma it wants, so the result bits do not
    depend on which products an optimiser fuses (hipcc's default is to fuse where it sees fit: two builds of the same
    arithmetic once differed in one output LSB of a few elements per thousand).  Compiled with contraction switched
    off on the command line, every kernel must come out the same instruction for instruction."""
    def stream(f):
        ops = []
        for line in f.split("\n")[1:]:
            t = line.split(";")[0].strip()
            if t.startswith("s_endpgm"):
                break
            if t and not t.startswith(".") and not t.endswith(":"):
                ops.append(re.sub(r"\.LBB\d+_\d+", "L", re.sub(r"_ZZN\w+", "SYM", t)))
        return ops
    for a, b in zip(*assembly):
        assert a.split(":")[0] == b.split(":")[0]
        assert stream(a) == stream(b), a.split(":")[0]


def _blocks(func_text):
    """Basic blocks of one function of the assembly: name -> (instructions, successors).  A block ends at a label or
    after a branch; `s_branch` has no fall-through, `s_endpgm` has no successor."""
    blocks, order, cur = {}, [], "entry"
    blocks[cur] = []
    order.append(cur)
    for line in func_text.split("\n")[1:]:
        t = line.split(";")[0].rstrip()
        m = re.match(r"^(\.LBB\d+_\d+):", t)
        if m:
            cur = m.group(1)
            blocks[cur] = []
            order.append(cur)
            continue
        t = t.strip()
        if not t or t.startswith(".") or t.endswith(":"):
            continue
        blocks[cur].append(t)
        if t.startswith("s_endpgm"):
            break
        if re.match(r"s_c?branch", t):  # a branch ends the block: what follows is an anonymous fall-through block
            nxt = "%s+%d" % (cur, len(blocks[cur]))
            blocks[nxt] = []
            order.append(nxt)
            cur = nxt
    succ = {}
    for i, name in enumerate(order):
        ins = blocks[name]
        out = []
        last = ins[-1] if ins else ""
        m = re.match(r"(s_c?branch\w*)\s+(\.LBB\d+_\d+)", last)
        if m:
            out.append(m.group(2))
        if not last.startswith("s_branch") and not last.startswith("s_endpgm") and i + 1 < len(order):
            out.append(order[i + 1])
        succ[name] = out
    return blocks, succ, order


VMEM = re.compile(r"(global|buffer|flat)_(load|store|atomic)\w*")
REG_LOAD = re.compile(r"global_load_(dword|dwordx2|dwordx3|dwordx4|ubyte|sbyte|ushort|sshort)\s+(v\[(\d+):(\d+)\]|v(\d+)),")


def _check_function(name, text):
    """For every load that returns into registers: on EVERY path from the load, its registers are not mentioned by any
    instruction until an `s_waitcnt vmcnt(n)` has been passed with n <= the number of vector memory instructions issued
    on that path since the load (memory reads return in issue order).  A forward data-flow over the basic blocks with
    the state "fewest memory instructions issued since the load on any path to here"; a wait that is strict enough
    ends the path."""
    blocks, succ, order = _blocks(text)
    checked = 0
    for bname in order:
        for idx, ins in enumerate(blocks[bname]):
            m = REG_LOAD.match(ins)
            if not m:
                continue
            regs = set(range(int(m.group(3)), int(m.group(4)) + 1)) if m.group(3) else {int(m.group(5))}
            # the compiler's own loads are followed by its own waits; the hand-written ones are those it knows nothing
            # about - both kinds must satisfy the property, so both are checked
            best = {}  # block -> fewest instructions issued since the load at block entry
            work = []

            def run(block, start, k):
                for j in range(start, len(blocks[block])):
                    t = blocks[block][j]
                    w = WAIT.match("\t" + t)
                    if w and int(w.group(1)) <= k:
                        return None  # retired on this path
                    if re.match(r"(v_|ds_|global_|buffer_|flat_|s_)", t) and (_regs(t) & regs) and not t.startswith("s_waitcnt"):
                        raise AssertionError("%s: `%s` touches v%s before the load `%s` has been waited for" % (
                            name, t, sorted(_regs(t) & regs), ins))
                    if VMEM.match(t):
                        k += 1
                return min(k, 64)

            k = run(bname, idx + 1, 0)
            if k is not None:
                work = [(s_, k) for s_ in succ[bname]]
            while work:
                b, k = work.pop()
                if b in best and best[b] <= k:
                    continue
                best[b] = k
                out = run(b, 0, k)
                if out is not None:
                    work.extend((s_, out) for s_ in succ[b])
            checked += 1
    return checked


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_no_read_of_an_asynchronously_loaded_register_before_its_wait(kernels):
    checked = 0
    for f in kernels:
        checked += _check_function(f.split(":")[0], f)
    # at least the two loads of mask bytes of every kernel and the Q rows of those that load them into registers
    assert checked >= 3 * len(kernels)


def test_the_checker_itself_finds_a_missing_wait():
    """A path on which the wait is too weak, and one on which a branch skips it."""
    ok = "f:\n\tglobal_load_dwordx4 v[2:5], v1, s[0:1]\n\tglobal_load_lds_dwordx4 v1, s[2:3]\n\ts_waitcnt vmcnt(1)\n\tv_mov_b32 v9, v2\n\ts_endpgm\n"
    assert _check_function("ok", ok) == 1
    weak = ok.replace("vmcnt(1)", "vmcnt(2)")
    with pytest.raises(AssertionError):
        _check_function("weak", weak)
    skipped = ("f:\n\tglobal_load_dwordx4 v[2:5], v1, s[0:1]\n\ts_cbranch_vccnz .LBB0_2\n\ts_waitcnt vmcnt(0)\n.LBB0_2:\n"
               "\tv_mov_b32 v9, v2\n\ts_endpgm\n")
    with pytest.raises(AssertionError):
        _check_function("skipped", skipped)


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_no_kernel_keeps_anything_in_scratch(assembly_files):
    """A launch bound that the register count does not meet is met by spilling, without a word: the reload of a spilled
    register in a key loop waits for every tile in flight (`s_waitcnt vmcnt(0)`), and the prefetch is gone."""
    scratch = dict(re.findall(r"\.amdhsa_kernel (\S+)\n(?:\s+\.amdhsa_(?!private)\S+ .*\n)*\s+\.amdhsa_private_segment_fixed_size (\d+)",
                              open(assembly_files[0]).read()))
    assert sum("_fwd_kernel" in name for name in scratch) == 64 and sum("_few_kernel" in name for name in scratch) > 0
    assert {name: size for name, size in scratch.items() if size != "0"} == {}


def _fmas_behind_operand_reads(func_text):
    """For every loop of a kernel: the fmas between four or more 128-bit LDS reads in a row and the matrix instruction behind
    them, where there are any."""
    at, ins, found = {}, [], []
    for line in func_text.split("\n")[1:]:
        label, t = re.match(r"^(\.LBB\d+_\d+):", line), line.split(";")[0].strip()
        if label:
            at[label.group(1)] = len(ins)
        elif t and not t.startswith(".") and not t.endswith(":"):
            ins.append(t)
            back = re.match(r"s_c?branch\w*\s+(\.LBB\d+_\d+)", t)
            if back and at.get(back.group(1), len(ins)) < len(ins) - 200:
                reads = fmas = most = 0
                for x in ins[at[back.group(1)]:]:
                    if "mfma" in x:
                        most, reads, fmas = max(most, fmas if reads >= 4 else 0), 0, 0
                    elif x.startswith("ds_read_b128"):
                        reads, fmas = reads + 1, 0
                    elif x.startswith("v_fma"):
                        fmas += 1
                found.append(most)
    return found


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_last_merge_covers_the_first_operand_reads_of_the_next_block(kernels):
    """Steady-state loops of the 256-row kernel without masked keys: the first K operands are asked for in front of the sixteen fmas of the last
    output tile.  Where the compiler chose by itself, what changed elsewhere in the kernel could put them behind twelve of those.  (At d = 128
    blocks of 64 keys leave it to the compiler.)"""
    for f in kernels:
        name = f.split(":")[0]
        d, block, full = re.search(r"fwd_kernelILi(\d+)ELi(\d+)ELb.ELb.ELb.ELb(.)E", name).groups() if "fwd_kernel" in name else (0,) * 3
        if d == "64" or block == "128":
            # both halves of the workgroup; with 255 steps (the last template argument) the column sums stand there in the second
            loops = [n for n in _fmas_behind_operand_reads(f) if n >= 16]
            assert len(loops) >= (1 if full == "1" else 2), (name, _fmas_behind_operand_reads(f))


def _jumps_behind_the_end(func_text):
    """Blocks behind the last `s_endpgm` of a kernel that do nothing but jump back."""
    tail, alone = func_text.split("s_endpgm")[-1].split(".section")[0], []
    for block in re.split(r"\n(?=\.LBB\d+_\d+:)", tail)[1:]:
        ins = [t for t in (line.split(";")[0].strip() for line in block.split("\n")[1:]) if t and not t.startswith(".")]
        if len(ins) == 1 and ins[0].startswith("s_branch"):
            alone.append(block.split(":")[0])
    return alone


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_first_block_without_masked_keys_is_not_reached_by_way_of_the_end(kernels):
    """GEMM 1 of the first key block has two forms; the usual one, without masked keys, is reached without a jump to the end of the kernel and
    back, whose instruction fetch the smallest calls wait for (whole blocks)."""
    found = {f.split(":")[0]: _jumps_behind_the_end(f) for f in kernels if re.search(r"fwd_kernelILi\d+ELi\d+ELb.ELb.ELb0E", f.split(":")[0])}
    assert len(found) == 32 and {name: jumps for name, jumps in found.items() if jumps} == {}


def _runs_of_moves(func_text):
    """Lengths of the runs of eight and more register moves (of a register or 0) in a kernel, address arithmetic between them not counted."""
    runs, n = [], 0
    for line in func_text.split("\n")[1:]:
        t = line.split(";")[0].strip()
        if re.match(r"v_mov_b(32|64)(_e32)? v(\d+|\[\d+:\d+\]), (v(\d+|\[\d+:\d+\])|0)$", t):
            n += 1
        elif t and not t.startswith(".p2align") and not re.match(r"s_(?!c?branch|barrier)|v_or_b32", t):
            runs += [n] if n >= 8 else []
            n = 0
    return runs


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_general_loop_carries_no_p_of_blocks_that_have_none(kernels):
    """P of a key block without an unmasked key is never used; where the general loop does not say so, the compiler starts it at zero, 14 to 24
    moves in front of the loop that every call takes for its last key block.  The last run of moves is then that one, and not the start of O (some
    32 registers or more).  Not at d = 128 with partly filled ends, or with 255 steps and blocks of 64 keys."""
    late = {}
    for f in kernels:
        name = f.split(":")[0]
        d, block, ragged, full = re.search(r"fwd_kernelILi(\d+)ELi(\d+)ELb.ELb.ELb(.)ELb(.)E", name).groups() if "fwd_kernel" in name else (0,) * 4
        if d == "64" or (d == "128" and ragged == "0" and (block, full) != ("64", "1")):
            late[name] = _runs_of_moves(f)
    assert len(late) == 32 + 12 and {name: runs for name, runs in late.items() if runs[-1] < 30} == {}


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_tile_of_a_short_sequence_asks_for_no_lane(kernels):
    """A key sequence shorter than one block is all prologue: the loads of its tile take their row from the address they are given, and the kernels for
    partly filled ends ask for the lane as often as those without (eight times more often cost such a call 0.1 us)."""
    asked = {re.search(r"fwd_kernelI(\S+?EL)b(.)(ELb.E)EEvNS", f.split(":")[0]).groups(): f.count("v_mbcnt_lo") for f in kernels if "fwd_kernel" in f.split(":")[0]}
    assert len(asked) == 64 and {k: n for k, n in asked.items() if n > asked[k[0], "0", k[2]]} == {}


def _maxima_behind_operand_reads(func_text):
    """Float maxima between the transposing reads of V (and what stands between those) and the next matrix instruction, for each run of them."""
    found, reads, maxima = [], 0, 0
    for line in func_text.split("s_endpgm")[0].split("\n")[1:]:
        t = line.strip()
        if t.startswith("ds_read_b64_tr"):
            reads, maxima = reads + 1, 0
        elif t.startswith("v_mfma"):
            found += [maxima] if reads else []
            reads = 0
        elif t.startswith("v_max_f32"):
            maxima += 1
    return found


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_the_first_product_of_a_merge_does_not_wait_for_the_weights(kernels):
    """Split kernel: the weights of a round's key blocks, a chain of maxima and exponentials, are computed behind the first product, which needs none of
    them - but where the operands of all blocks are asked for together (one row group, blocks of 64 keys, 128 steps), over whose latency they are."""
    late = {}
    for f in kernels:
        m = re.search(r"split_kernelILi\d+ELi(\d+)ELb.ELb.ELb(.)ELi(\d)ELb0E", f.split(":")[0])
        if m:
            all_held = m.groups() == ("64", "0", "1")
            late[f.split(":")[0]] = (_maxima_behind_operand_reads(f)[0] > 0) == all_held
    assert len(late) == 64 and [name for name, as_meant in late.items() if not as_meant] == []


def _whole_function(func_text):
    """Basic blocks and successors as in _blocks, those behind the first `s_endpgm` with them; comments stay."""
    blocks, order, cur = {"entry": []}, ["entry"], "entry"
    for line in func_text.split(".Lfunc_end")[0].split("\n")[1:]:
        m, t = re.match(r"^(\.LBB\d+_\d+):", line), line.strip()
        if m:
            cur = m.group(1)
            blocks[cur] = []
            order.append(cur)
        elif t and (t.startswith("; Q from LDS") or not re.match(r"[.;]|[^;]*:$", t)):
            blocks[cur].append(t)
            if re.match(r"s_c?branch|s_endpgm", t):
                cur = "%s+%d" % (cur, len(blocks[cur]))
                blocks[cur] = []
                order.append(cur)
    succ = {}
    for i, name in enumerate(order):
        last = blocks[name][-1] if blocks[name] else ""
        to = re.match(r"s_c?branch\w*\s+(\.LBB\d+_\d+)", last)
        falls = not re.match(r"s_branch|s_endpgm", last) and i + 1 < len(order)
        succ[name] = ([to.group(1)] if to else []) + ([order[i + 1]] if falls else [])
    return blocks, succ


def _paths(blocks, succ, block, start, state, step):
    """Runs step(state, instruction) along every path from there; a state is a tuple of numbers, step returns None where a path is done with."""
    seen, work = set(), [(block, start, state)]
    while work:
        b, i, s = work.pop()
        for t in blocks[b][i:]:
            s = step(s, t)
            if s is None:
                break
        else:
            work += [x for x in ((to, 0, s) for to in succ[b]) if x not in seen]
            seen.update((to, 0, s) for to in succ[b])


def _check_q_through_lds(func_text, waits=True):
    """How many loads ask for Q rows through LDS.  On every path (a) from such a load the place where the rows are read again (the reads cannot be
    moved in front of it) stands behind the wait that retires the load, and, where other wavefronts fetch some of the rows, behind a barrier after that
    wait; (b) from there, where the rows' place is written again later, no 128-bit LDS read is in flight at the next barrier."""
    blocks, succ = _whole_function(func_text)

    def landed(shared):
        def step(s, t):
            issued, waited = s
            w = WAIT.match("\t" + t)
            waited |= bool(w and int(w.group(1)) <= issued)
            if waited and (not shared or t.startswith("s_barrier")):
                return None
            assert not t.startswith("; Q from LDS"), "read too early"
            return min(issued + bool(VMEM.match(t)), 63), waited
        return step

    def arrived(s, t):
        behind, = s  # LDS and scalar memory instructions behind the last 128-bit read; -1: none in flight
        w = re.match(r"s_waitcnt\b.*lgkmcnt\((\d+)\)", t)
        if w and int(w.group(1)) <= behind:
            behind = -1
        if t.startswith("s_barrier"):
            assert behind < 0, "read in flight at a barrier"
            return None
        if t.startswith("ds_read_b128"):
            return 0,
        return min(behind + (behind >= 0 and bool(re.match(r"ds_|s_load", t))), 15),

    loads = 0
    for b in blocks:
        for i, t in enumerate(blocks[b]):
            m = re.search(r"global_load_lds_dwordx4.*; Q, shared (\d)", t)
            loads += bool(m)
            if m and waits:
                _paths(blocks, succ, b, i + 1, (0, False), landed(m.group(1) == "1"))
            if t == "; Q from LDS, place reused":
                _paths(blocks, succ, b, i + 1, (-1,), arrived)
    return loads


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_q_rows_through_lds_are_waited_for(kernels):
    """The kernels of head size 128 whose Q rows pass through LDS: all but the split kernel's forms of one row group and blocks of 64 keys.  (No counting of
    waits in the pair kernel and for partly filled ends in the 256-row one: two branches on one condition there, whose paths this would mix.)"""
    counted = lambda name: not re.search(r"pair_kernel|fwd_kernelILi128ELi\d+ELb.ELb.ELb1E", name)
    through = {f.split(":")[0]: _check_q_through_lds(f, counted(f.split(":")[0])) for f in kernels}
    for name, loads in through.items():
        kind, d, block = re.search(r"(fwd|split|pair)_kernelILi(\d+)ELi(\d+)", name).groups()
        own_k = re.search(r"split_kernelILi\d+ELi64ELb.ELb.ELb.ELi1E", name)
        assert (loads > 0) == (d == "128" and not own_k), (name, loads)


def test_the_q_checker_itself_finds_what_it_looks_for():
    ok = ("f:\n\tglobal_load_lds_dwordx4 v1, s[2:3] ; Q, shared 1\n\ts_waitcnt vmcnt(0)\n\ts_barrier\n\t; Q from LDS, place reused\n\tds_read_b128 v[2:5], v1\n\ts_waitcnt lgkmcnt(0)\n"
          "\ts_barrier\n\ts_endpgm\n.Lfunc_end0:\n")
    assert _check_q_through_lds(ok) == 1
    late = ok.replace("\ts_waitcnt lgkmcnt(0)\n\ts_barrier", "\ts_cbranch_scc1 .LBB0_9\n\ts_waitcnt lgkmcnt(0)\n.LBB0_9:\n\ts_barrier")
    for wrong in (ok.replace("vmcnt(0)", "vmcnt(1)"), ok.replace("vmcnt(0)\n\ts_barrier", "vmcnt(0)"), ok.replace("lgkmcnt(0)", "lgkmcnt(1)"), late):
        with pytest.raises(AssertionError):
            _check_q_through_lds(wrong)
