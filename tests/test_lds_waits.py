"""Barriers of the built kernels and the LDS reads before them, on the CPU, from the disassembly of the
library built here. Where a barrier frees a piece of LDS for another wave to overwrite (loads straight into LDS
above all, which no LDS queue orders), every read of it must have returned before the barrier."""
import os
import re
import shutil
import subprocess

import pytest

import flint_attn as fa

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
ADDR = re.compile(r"// ([0-9A-F]+):")
TARGET = re.compile(r"<(\S+?)(?:\+0x([0-9a-f]+))?>\s*$")
MAX_COUNT = 40  # operations followed per path: more than lgkmcnt can count (15)


def _kernels(text):
    """{kernel: (first address, [(address, instruction, branch target address or None)])}"""
    out, code = {}, None
    for line in text.splitlines():
        head = re.match(r"^([0-9a-f]+) <(\S+)>:", line)
        if head:
            start, code = int(head[1], 16), []
            out[head[2]] = (start, code)
        elif code is not None and (a := ADDR.search(line)):
            op = line.split("//")[0].strip()
            t = TARGET.search(line) if "branch" in op else None
            code.append((int(a[1], 16), op, start + int(t[2] or "0", 16) if t else None))
    return out


def reads_at_barriers(code):
    """The addresses of the barriers that some path reaches with LDS reads not yet waited for. A state is the operations under lgkmcnt since they were last all waited for, oldest first (True: an
    LDS read); lgkmcnt(n) leaves the newest n."""
    at = {a: i for i, (a, _, _) in enumerate(code)}
    state, bad, work = [None] * len(code), set(), [(0, ())]
    while work:
        i, s = work.pop()
        while i < len(code):
            if state[i] is not None:  # joins: the longer list, a read where either path has one
                n = max(len(s), len(state[i]))
                s = tuple(x or y for x, y in zip((False,) * (n - len(s)) + s, (False,) * (n - len(state[i])) + state[i]))
                if s == state[i]:
                    break
            state[i] = s
            addr, op, target = code[i]
            name = op.split()[0]
            if name.startswith("ds_"):
                s = (s + (True,))[-MAX_COUNT:]
            elif name.startswith(("s_load", "s_buffer_load")):
                s = (s + (False,))[-MAX_COUNT:]
            elif name == "s_waitcnt" and (m := re.search(r"lgkmcnt\((\d+)\)", op)):
                s = s[len(s) - int(m[1]):] if int(m[1]) < len(s) else s
            elif name == "s_barrier" and any(s):
                bad.add(addr)
            if name == "s_branch":
                i = at[target]
                continue
            if name.startswith("s_cbranch"):
                work.append((at[target], s))
            assert not name.startswith(("s_setpc", "s_swappc")), "a call: not followed"
            if name == "s_endpgm":
                break
            i += 1
    return sorted(bad)


def test_reads_at_barriers_follows_waits_and_branches():
    """The check itself, on a loop written out here: a read that is waited for in one branch only."""
    loop = [(0, "ds_read_b128 v[0:3], v9", None), (8, "s_cbranch_scc0 1", 16), (12, "s_waitcnt lgkmcnt(0)", None),
            (16, "s_barrier", None), (20, "s_cbranch_scc1 65531", 0), (24, "s_endpgm", None)]
    assert reads_at_barriers(loop) == [16]
    loop[1] = (8, "s_nop 0", None)
    assert reads_at_barriers(loop) == []
    loop[2] = (12, "s_waitcnt vmcnt(3) lgkmcnt(1)", None)
    assert reads_at_barriers(loop) == [16]


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    so = shutil.copy(fa.LIB_PATH, d)  # the code objects are written beside it
    subprocess.run([OBJDUMP, "--offloading", so], check=True, capture_output=True)
    out = {}
    for f in sorted(d.glob("*gfx950")):
        r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True, capture_output=True, text=True)
        out.update(_kernels(r.stdout))
    assert sum("gemm_int_kernel" in k for k in out) == 8
    return out


def test_no_lds_read_outstanding_at_a_barrier(kernels):
    """Every barrier of every kernel. gemm_int_kernel's stages are overwritten by loads straight into LDS after
    its barrier; the reads that feed FMAs (scales, token sums, mins) once crossed it unwaited for."""
    bad = {k: b for k, (_, code) in kernels.items() if (b := reads_at_barriers(code))}
    assert not bad
