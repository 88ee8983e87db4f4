"""The attention kernels issue some loads as asm that the compiler does not count (the Q
operands; the token ids): their destination registers are valid only behind a hand-placed
vmcnt wait.  To the compiler those registers hold their values from the moment the asm
statement ends, so nothing stops it from copying or spilling them while the load is still in
flight.  This test compiles the three attention translation units to assembly (no GPU needed)
and checks that between every such load and the first wait that covers it no other instruction
names its destination registers.

The HBM -> LDS copies set m0 inside their asm statement without telling the compiler (naming a
reserved register as clobbered only draws a warning).  That is sound as long as the compiler
itself never uses m0 in these kernels: the second check asserts that no instruction outside an
asm statement names m0 in any translation unit that issues such copies.

The tile loop of the attention kernels waits for its copies with hand-counted vmcnt values: that
holds only while the compiler puts no vector-memory instruction of its own into the loop.  The
third check finds the tile loop of every instantiation (one inner loop, closed by a branch back to
its header) and asserts that it holds no scratch access (a spill) and no s_waitcnt vmcnt outside
the asm statements (the compiler waiting for a load of its own).  The same holds for the walk of the votes kernel,
from its first copy to the wait for the last one.

The asm statements take base addresses in scalar registers.  A vector-memory instruction may read a scalar register that the
vector ALU wrote (readfirstlane, readlane) five wait states later; the compiler keeps that distance for its own instructions
and does not look into asm, so the listing is checked for it, along every path.

A copy into LDS may read m0 one wait state behind a scalar write of it; the compiler puts it there behind its own writes only.

The row maxima read accumulators of matrix multiplies in asm.  The vector ALU may read or write what a multiply writes only some
wait states later (twelve behind a 32x32x16, eight behind a 16x16x32); the compiler keeps that distance for its own instructions
and does not look into asm, so the listing is checked for it, along every path.

The votes kernel lists rows in LDS as 16-bit numbers and reads several entries at a time.  A read through another scalar
type would be free to move ahead of the stores (type-based aliasing); the last check looks at the types of its LDS
loads and stores before any optimisation."""
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

import pytest

from fgattn_tk_cuda_amd import build

CSRC = Path(build.__file__).resolve().parent / "csrc"
UNITS = ["attn_inst_blocks.hip", "attn_inst_tokens.hip", "attn_inst_dense.hip"]
VOTES_UNIT = "votes_kernels.hip"
M0_UNITS = UNITS + ["mask_kernels.hip", VOTES_UNIT]
TOPK_UNIT = "topk_kernels.hip"   # asm and matrix multiplies, no copies into LDS


def _regs(text):
    out = set()
    for m in re.finditer(r"\b([va])\[(\d+):(\d+)\]", text):
        out.update(m.group(1) + str(i) for i in range(int(m.group(2)), int(m.group(3)) + 1))
    for m in re.finditer(r"\b([va])(\d+)\b", text):
        out.add(m.group(1) + m.group(2))
    return out


def _is_vmem(op):
    return op.startswith(("global_load", "global_store", "scratch_load", "scratch_store", "buffer_", "flat_"))


def inflight_accesses(listing):
    """[(line of the access, line of the load)] for a straight-line scan of an assembly listing."""
    lines = listing.split("\n")
    found = []
    for n, raw in enumerate(lines):
        t = raw.strip().split(";")[0].strip()
        if not t.startswith("global_load_dword") or t.startswith("global_load_lds"):
            continue
        dst = _regs(t.split(None, 1)[1].split(",")[0])
        younger = 0
        for j in range(n + 1, min(n + 6000, len(lines))):
            t2 = lines[j].strip().split(";")[0].strip()
            if not t2 or t2.startswith("."):
                continue
            if re.match(r"^_Z\w+:", lines[j]):
                break
            op = t2.split()[0]
            if op == "s_endpgm":
                break
            if op == "s_waitcnt":
                m = re.search(r"vmcnt\((\d+)\)", t2)
                if m and int(m.group(1)) <= younger:
                    break          # every load up to ours has landed
                continue
            if " " in t2 and _regs(t2.split(None, 1)[1]) & dst:
                found.append((j + 1, n + 1, t2, t))
                break
            if _is_vmem(op):
                younger += 1
    return found


def m0_uses_outside_asm(listing):
    """Lines outside ASMSTART/ASMEND blocks whose instruction names m0."""
    found, inside = [], False
    for n, raw in enumerate(listing.split("\n")):
        if "#ASMSTART" in raw:
            inside = True
            continue
        if "#ASMEND" in raw:
            inside = False
            continue
        t = raw.split(";")[0].strip()
        if not inside and t and not t.startswith(".") and re.search(r"\bm0\b", t):
            found.append((n + 1, t))
    return found


class Flow:
    """The instructions of one kernel, [(operation, operands, inside an asm statement)], and what may follow each."""

    def __init__(self, body):
        self.ins, labels, inside = [], {}, False
        for raw in body.split("\n"):
            inside = "#ASMSTART" in raw or (inside and "#ASMEND" not in raw)
            t = raw.split(";")[0].strip()
            label = re.match(r"(\.?\w+):", t)
            if label:
                labels[label.group(1)] = len(self.ins)
            elif t and not t.startswith("."):
                op, _, args = t.partition(" ")
                self.ins.append((op, args.strip(), inside))
        self.after = []
        for i, (op, args, _) in enumerate(self.ins):
            follow = [] if op in ("s_branch", "s_endpgm", "s_setpc_b64") or i + 1 == len(self.ins) else [i + 1]
            self.after.append(follow + ([labels[args]] if op == "s_branch" or op.startswith("s_cbranch") else []))

    def within(self, i, states):
        """{instruction: fewest wait states between it and instruction i} of those that less than `states` lie ahead of."""
        near, todo = {}, [(j, 0) for j in self.after[i]]
        while todo:
            j, passed = todo.pop()
            if passed >= states or near.get(j, states) <= passed:
                continue
            near[j] = passed
            op, args, _ = self.ins[j]
            todo += [(n, passed + 1 + (int(args, 0) if op == "s_nop" else 0)) for n in self.after[j]]
        return near


def kernel_flows(listing):
    for m in re.finditer(r"^(_Z\w+):(.*?)^\.Lfunc_end", listing, re.S | re.M):
        yield m.group(1), Flow(m.group(2))


def scalar_bases_too_close(listing, states=5):
    """[(vector-ALU write, vector-memory instruction, wait states between them)] where an instruction reads a scalar register
    fewer than `states` wait states after the vector ALU wrote it, along any path."""
    def sregs(text):
        out = {"s" + m for m in re.findall(r"\bs(\d+)\b", text)} | set(re.findall(r"\bvcc\b", text))
        for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
            out.update("s%d" % r for r in range(int(lo), int(hi) + 1))
        return out

    found = []
    for _, flow in kernel_flows(listing):
        for i, (op, args, _) in enumerate(flow.ins):
            # the result, or the carry that add, sub and div_scale write beside it
            written = sregs(",".join(args.split(",")[:2 if "_co_" in op or "div_scale" in op else 1])) if op.startswith("v_") else None
            for j, passed in flow.within(i, states).items() if written else ():
                op2, args2, _ = flow.ins[j]
                if _is_vmem(op2) and written & sregs(args2):
                    found.append((op + " " + args, op2 + " " + args2, passed))
    return found


def multiplies_too_close(listing):
    """[(kernel, multiply, asm instruction, wait states between them)] where a vector-ALU or memory instruction of an asm
    statement names a register that a matrix multiply writes before it may."""
    found = []
    for kernel, flow in kernel_flows(listing):
        for i, (op, args, _) in enumerate(flow.ins):
            if not op.startswith("v_mfma"):
                continue
            dst = _regs(args.split(",")[0])
            for j, passed in flow.within(i, 12 if "32x32x16" in op else 8 if "16x16x32" in op else 20).items():
                op2, args2, asm = flow.ins[j]
                if asm and (op2.startswith("v_") or _is_vmem(op2)) and _regs(args2) & dst:
                    found.append((kernel, op + " " + args, op2 + " " + args2, passed))
    return found


def m0_too_close(listing):
    """[(kernel, scalar write of m0, copy)] where a copy into LDS follows a scalar write of m0, which it reads, without a wait
    state between them, along any path."""
    found = []
    for kernel, flow in kernel_flows(listing):
        for i, (op, args, _) in enumerate(flow.ins):
            if op.startswith("s_") and args.split(",")[0] == "m0":
                found += [(kernel, op + " " + args, " ".join(flow.ins[j][:2])) for j in flow.within(i, 1) if "_lds_" in flow.ins[j][0]]
    return found


def tile_loop_findings(listing):
    """{kernel: (scratch accesses, compiler vmcnt waits)} inside the tile loop of every attn_fwd_kernel
    instantiation of a listing; a kernel whose loop is not found maps to None."""
    out, name, cur = {}, None, []
    for line in listing.split("\n"):
        m = re.match(r"^(_ZN6spattn15attn_fwd_kernel\w+):", line)
        if m:
            name, cur = m.group(1), []
        if name is None:
            continue
        cur.append(line)
        if not line.startswith(".Lfunc_end"):
            continue
        hdr = next(((i, l.split(":")[0]) for i, l in enumerate(cur) if l.startswith(".LBB") and "Loop Header" in l), None)
        last = None
        if hdr is not None:
            back = re.compile(r"s_c?branch\w*\s+" + re.escape(hdr[1]) + r"\b")
            last = max((i for i in range(hdr[0], len(cur)) if back.match(cur[i].strip())), default=None)
        if hdr is None or last is None:
            out[name] = None
        else:
            scratch = waits = 0
            inside = False
            for l in cur[hdr[0]:last + 1]:
                if "#ASMSTART" in l:
                    inside = True
                elif "#ASMEND" in l:
                    inside = False
                t = l.split(";")[0].strip()
                scratch += t.startswith("scratch_")
                waits += (not inside) and t.startswith("s_waitcnt") and "vmcnt" in t
            out[name] = (scratch, waits)
        name = None
    return out


def walk_findings(listing, kernel="blockmax_votes_kernel"):
    """{kernel: (scratch accesses, compiler vmcnt waits)} between the first copy and the last hand-written wait for all
    copies, of every instantiation; None where no such wait follows the last copy."""
    out = {}
    for m in re.finditer(r"^(_ZN6spattn\d+" + kernel + r"\w+):(.*?)^\.Lfunc_end", listing, re.S | re.M):
        inside, lines = False, []   # (instruction, is inside an asm statement)
        for l in m.group(2).split("\n"):
            inside = "#ASMSTART" in l or (inside and "#ASMEND" not in l)
            lines.append((l.split(";")[0].strip(), inside))
        copies = [i for i, (t, _) in enumerate(lines) if t.startswith("global_load_lds")]
        done = [i for i, (t, asm) in enumerate(lines) if asm and t == "s_waitcnt vmcnt(0)"]
        if not copies or not done or done[-1] < copies[-1]:
            out[m.group(1)] = None
            continue
        walk = lines[copies[0]:done[-1]]
        out[m.group(1)] = (sum(t.startswith("scratch_") for t, _ in walk),
                           sum(not asm and t.startswith("s_waitcnt") and "vmcnt" in t for t, asm in walk))
    return out


def test_walk_checker():
    asm = "\t;;#ASMSTART\n\t%s\n\t;;#ASMEND\n"
    name = "_ZN6spattn21blockmax_votes_kernelILi64EEEvNS_11VotesParamsE"
    body = (name + ":\n\ts_waitcnt vmcnt(0)\n" + asm % "global_load_lds_dwordx4 v1, s[0:1]" + "%s" + asm % "s_waitcnt vmcnt(8) lgkmcnt(0)" +
            asm % "global_load_lds_dwordx4 v1, s[0:1]" + asm % "s_waitcnt vmcnt(0)" + "\ts_waitcnt vmcnt(0)\n\ts_endpgm\n.Lfunc_end0:\n")
    assert walk_findings(body % "") == {name: (0, 0)}
    assert walk_findings(body % "\tscratch_load_dword v1, off, off\n\ts_waitcnt vmcnt(0)\n") == {name: (1, 1)}
    assert walk_findings((body % "").replace(asm % "s_waitcnt vmcnt(0)", "")) == {name: None}
    assert walk_findings("") == {}


def test_tile_loop_checker():
    body = ("_ZN6spattn15attn_fwd_kernelILi64EEEvNS_10AttnParamsE:\n\ts_nop 0\n.LBB0_3:   ; =>This Inner Loop Header: Depth=1\n"
            "\t;;#ASMSTART\n\ts_waitcnt vmcnt(4)\n\t;;#ASMEND\n%s\ts_cbranch_scc1 .LBB0_3\n\ts_endpgm\n.Lfunc_end0:\n")
    assert tile_loop_findings(body % "") == {"_ZN6spattn15attn_fwd_kernelILi64EEEvNS_10AttnParamsE": (0, 0)}
    assert list(tile_loop_findings(body % "\tscratch_load_dword v1, off, off\n\ts_waitcnt vmcnt(0)\n").values()) == [(1, 1)]
    assert list(tile_loop_findings(body.replace("s_cbranch_scc1 .LBB0_3", "s_nop 1") % "").values()) == [None]


def test_scalar_base_checker():
    def found(*lines):
        body = "_ZN6spattn1kE:\n" + "".join("\t" * (not l.endswith(":")) + l + "\n" for l in lines) + "\ts_endpgm\n.Lfunc_end0:\n"
        return sorted(f[2] for f in scalar_bases_too_close(body))

    write = ("v_readfirstlane_b32 s21, v9", "v_readfirstlane_b32 s20, v8")
    copy = ("s_mov_b32 m0, s3", "global_load_lds_dwordx4 v7, s[20:21]")
    assert found(*write, *copy) == [1, 2] and found(*write, "s_nop 2", *copy) == [4] and found(*write, "s_nop 3", *copy) == []
    assert found(*write, copy[0], "global_load_lds_dwordx4 v7, s[22:23]") == []
    assert found(".LBB0_1:", *copy, write[1], "s_cbranch_scc1 .LBB0_1") == [2]                         # around a loop
    assert found(write[1], "s_cbranch_scc1 .LBB0_2", "s_nop 15", ".LBB0_2:", *copy) == [2]            # past the wait
    assert found(write[1], "s_branch .LBB0_2", *copy, ".LBB0_2:") == []                               # not on a path
    assert found("v_add_co_u32_e32 v1, vcc, v2, v3", "global_load_lds_dwordx4 v7, vcc") == [0]
    assert found("v_cmp_gt_i32_e64 s[20:21], v1, v2", copy[1]) == [0] and found("v_add_u32_e32 v1, s20, v2", copy[1]) == []


def test_multiply_checker():
    asm = "\t;;#ASMSTART\n\tv_max3_f32 v1, v%d, v1, v2\n\t;;#ASMEND\n"
    multiply = "\tv_mfma_f32_32x32x16_bf16 v[64:79], v[4:7], v[8:11], 0\n"

    def states(*lines):
        body = "_ZN6spattn15attn_fwd_kernelILi64EEEvNS_10AttnParamsE:\n" + "".join(lines) + "\ts_endpgm\n.Lfunc_end0:\n"
        return [f[3] for f in multiplies_too_close(body)]

    branch, target = "\ts_cbranch_scc1 .LBB0_2\n", ".LBB0_2:\n"
    assert states(multiply, asm % 79) == [0] and states(multiply, asm % 80) == []
    assert states(multiply, "\ts_nop 10\n", asm % 79) == [11] and states(multiply, "\ts_nop 11\n", asm % 79) == []
    assert states(multiply, branch, "\ts_nop 15\n", target, asm % 64) == [1]                # the way past the wait
    assert states(target, asm % 64, multiply, branch) == [1]                               # around a loop
    assert states(target, asm % 64, multiply, "\ts_nop 15\n", branch) == []
    assert states(multiply, "\ts_branch .LBB0_2\n", asm % 64, "\ts_nop 15\n", target) == []  # not on a path
    small = multiply.replace("32x32x16", "16x16x32").replace("v[64:79]", "v[64:67]")
    assert states(small, "\ts_nop 6\n", asm % 64) == [7] and states(small, "\ts_nop 7\n", asm % 64) == []


def test_m0_distance_checker():
    def found(*lines):
        return len(m0_too_close("_ZN6spattn1kE:\n.LBB0_1:\n\t" + "\n\t".join(lines) + "\n\ts_endpgm\n.Lfunc_end0:\n"))

    copy, write = "global_load_lds_dwordx4 v1, s[0:1]", "s_mov_b32 m0, s3"
    assert found(write, copy) == 1 and found(write, "s_nop 0", copy) == 0 and found(write, "v_mov_b32_e32 v2, v3", copy) == 0
    assert found(copy, write, "s_cbranch_scc1 .LBB0_1") == 0 and found("global_load_dwordx4 v[0:3], v[4:5], off", write) == 0


def test_m0_checker_sees_a_compiler_use():
    ok = "\t;;#ASMSTART\n\ts_mov_b32 m0, s3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 v1, s[0:1]\n\t;;#ASMEND\n\tv_mov_b32_e32 v2, v3\n"
    bad = ok + "\ts_mov_b32 m0, -1\n"
    assert m0_uses_outside_asm(ok) == []
    assert len(m0_uses_outside_asm(bad)) == 1


def test_checker_sees_an_access_to_a_register_in_flight():
    bad = "\tglobal_load_dwordx4 v[4:7], v[2:3], off\n\tglobal_load_lds_dwordx4 v9, s[0:1]\n\tv_mov_b32_e32 v20, v5\n\ts_waitcnt vmcnt(0)\n"
    good = "\tglobal_load_dwordx4 v[4:7], v[2:3], off\n\tglobal_load_lds_dwordx4 v9, s[0:1]\n\ts_waitcnt vmcnt(1)\n\tv_mov_b32_e32 v20, v5\n"
    assert len(inflight_accesses(bad)) == 1
    assert inflight_accesses(good) == []


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(), reason="hipcc not found")
def test_no_instruction_touches_a_register_with_a_load_in_flight(tmp_path):
    hipcc = build._hipcc()

    def listing(unit):
        out = tmp_path / (unit + ".s")
        subprocess.run([hipcc, *build.HIPCC_FLAGS, "-S", "--cuda-device-only", "-o", str(out), str(CSRC / unit)],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        return out.read_text()

    with ThreadPoolExecutor(max_workers=4) as ex:
        texts = list(ex.map(listing, M0_UNITS + [TOPK_UNIT]))
    for unit, text in zip(M0_UNITS + [TOPK_UNIT], texts):
        near = multiplies_too_close(text)
        assert not near, "%s: %d asm instructions name a multiply's result too early, e.g. %s" % (unit, len(near), near[0])
    for unit, text in zip(M0_UNITS, texts):
        assert "global_load_lds_dwordx4" in text, unit
        uses = m0_uses_outside_asm(text)
        assert not uses, "%s: the compiler uses m0 next to hand-written copies: %s" % (unit, uses[:3])
        early = m0_too_close(text)
        assert not early, "%s: %d copies too close behind their m0, e.g. %s" % (unit, len(early), early[0])
        close = scalar_bases_too_close(text)
        assert not close, "%s: %d bases written too late, e.g. %s" % (unit, len(close), close[0])
        if unit == VOTES_UNIT:
            walks = walk_findings(text)
            assert len(walks) == 4 and all(f == (0, 0) for f in walks.values()), "%s: %s" % (unit, walks)
        if unit not in UNITS:
            continue
        assert "global_load_dword" in text, unit
        found = inflight_accesses(text)
        assert not found, "%s: %s" % (unit, found[:3])
        loops = tile_loop_findings(text)
        assert len(loops) >= 4, "%s: %d attention kernels found" % (unit, len(loops))
        for kernel, f in loops.items():
            assert f == (0, 0), "%s %s: tile loop not found, or scratch accesses / compiler vmcnt waits inside it: %s" % (unit, kernel, f)


def scalar_lds_types(ir):
    """({types loaded}, {types stored}) by scalar integer accesses to LDS in an LLVM listing; vector types alias everything."""
    found = [set(re.findall(op + r" (?:volatile )?(%s)" % ty, "\n".join(l for l in ir.split("\n") if "ptr addrspace(3) " in l)))
             for op, ty in (("load", r"i\d+(?=, ptr addrspace)"), ("store", r"i\d+(?= [%\w.-]+, ptr addrspace)"))]
    return tuple(found)


def test_scalar_lds_type_checker():
    ir = ("  store i16 %a, ptr addrspace(3) %p, align 2, !tbaa !1\n  %b = load i32, ptr addrspace(3) %p, align 4\n"
          "  %c = load <2 x i16>, ptr addrspace(3) %p, align 4\n  store i16 4096, ptr addrspace(3) %p\n  store i32 %x, ptr %y\n")
    assert scalar_lds_types(ir) == ({"i32"}, {"i16"})


@pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(), reason="hipcc not found")
def test_row_lists_are_read_as_they_were_written(tmp_path):
    out = tmp_path / "votes.ll"
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "-S", "-emit-llvm", "-Xclang", "-disable-llvm-passes", "--cuda-device-only", "-o",
                    str(out), str(CSRC / VOTES_UNIT)], check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    loaded, stored = scalar_lds_types(out.read_text())
    assert "i16" in stored and loaded <= stored, (loaded, stored)
