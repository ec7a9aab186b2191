"""Loads that go straight from global memory into LDS hold no register, so nothing but a counted wait
(s_waitcnt vmcnt) keeps a wave from passing the barrier that publishes a block whose load is still in
flight.  The compiler orders the other loads around them: this test walks every control-flow path of
the kernels in the built library and checks that each such load is waited for before the next
barrier.  Vector memory operations retire in issue order, so vmcnt(N) covers a load once at least N
were issued after it.  No GPU needed."""

import os
import re
import shutil
import subprocess

import pytest

import libcc_amd

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
VMEM = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")
VMCNT = re.compile(r"vmcnt\((\d+)\)")
TARGET = re.compile(r"<[^>]*\+0x([0-9a-f]+)>")


def listing(tmp):
    """{kernel: [(offset, instruction, branch target offset or None)]} of the gfx950 code in the library"""
    lib = shutil.copy(libcc_amd.LIB_PATH, os.path.join(tmp, "lib.so"))   # objdump writes beside its input
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    out = {}
    for name in sorted(os.listdir(tmp)):
        if "amdgcn" not in name:
            continue
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(tmp, name)], check=True,
                              capture_output=True, text=True).stdout
        code, base = None, 0
        for line in text.splitlines():
            m = re.match(r"([0-9a-f]+) <(\S+)>:", line)
            if m:
                base, code = int(m.group(1), 16), out.setdefault(m.group(2), [])
            elif code is not None and "//" in line:
                ins, tail = line.split("//", 1)
                t = TARGET.search(tail)
                code.append((int(tail.split(":")[0], 16) - base, ins.strip(), int(t.group(1), 16) if t else None))
    return out


def unwaited(code):
    """(direct loads, those that reach a barrier without a wait that covers them)"""
    at = {off: i for i, (off, _, _) in enumerate(code)}
    direct = [i for i, (_, t, _) in enumerate(code) if t.startswith("global_load_lds") or re.search(r"^buffer_load.* lds$", t)]
    bad = []
    for d in direct:
        todo, seen = [(d + 1, 0)], set()
        while todo:
            i, later = todo.pop()
            if (i, later) in seen or i >= len(code):
                continue
            seen.add((i, later))
            _, t, target = code[i]
            op = t.split(None, 1)[0]
            if VMEM.match(op):
                later = min(later + 1, 63)
            elif op == "s_waitcnt":
                m = VMCNT.search(t)
                if m and later >= int(m.group(1)):
                    continue
            elif op == "s_barrier":
                bad.append(code[d])
                break
            elif op == "s_endpgm":
                continue
            if op == "s_branch":
                todo.append((at[target], later))
                continue
            if op.startswith("s_cbranch"):
                todo.append((at[target], later))
            todo.append((i + 1, later))
    return len(direct), bad


def test_walk_finds_an_uncovered_load():
    """The walk itself, on a loop whose wait leaves two later loads in flight: covered when two follow
    the direct load, not when one does, nor on the path that skips them."""
    def code(*ins):
        return [(4 * i, t, target) for i, (t, target) in enumerate(ins)]

    dma, load = ("buffer_load_dwordx4 v0, s[0:3], 0 offen lds", None), ("global_load_dwordx4 v[2:5], v[0:1], off", None)
    wait, bar, end = ("s_waitcnt vmcnt(2)", None), ("s_barrier", None), ("s_endpgm", None)
    assert unwaited(code(dma, load, load, wait, bar, ("s_branch 1", 0))) == (1, [])
    assert len(unwaited(code(load, dma, load, wait, bar, ("s_branch 1", 0)))[1]) == 1
    assert len(unwaited(code(dma, ("s_cbranch_vccnz 1", 16), load, load, wait, bar, end))[1]) == 1


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="llvm-objdump is not installed")
def test_every_direct_load_is_waited_for(tmp_path):
    found = {}
    for name, code in listing(str(tmp_path)).items():
        n, bad = unwaited(code)
        if n:
            found[name] = n
        assert not bad, (name, bad[:3])
    # the FP32 and split forms of both item kernels, and the gBX back-contraction
    for part in ("triples_kernelIfLi1E", "triples_kernelIfLi2E", "triples_kernelIfLi3E", "triples_kernelIfLi4E",
                 "adj_item_kernelILi1E", "adj_item_kernelILi2E", "gbx_kernel"):
        assert any(part in name for name in found), (part, sorted(found))
