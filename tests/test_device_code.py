"""Properties of the built gfx950 code that no run can be relied on to show.

The library's own kernels are disassembled (llvm-objdump) and walked over
every path; no GPU is needed.
"""
import collections
import glob
import os
import re
import shutil
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
INSN = re.compile(r"^\t(\S+)\s*(.*?)\s*//\s*([0-9A-F]+):")
TARGET = re.compile(r"<[^>]*\+0x([0-9a-f]+)>\s*$")


def disassemble(tk, tmp_path, kernel):
    """[(address from the kernel's start, mnemonic, operands, branch target)]
    of the one kernel of the built library whose mangled name holds `kernel`."""
    tk.lib()
    src = os.path.join(os.path.dirname(tk.__file__), "libtnr_hip.so")
    shutil.copy(src, tmp_path / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    found = []
    for obj in glob.glob(str(tmp_path / "*gfx950")):
        syms = subprocess.run([OBJDUMP, "-t", obj], check=True, capture_output=True, text=True).stdout
        found += [(obj, s.split()[-1]) for s in syms.splitlines() if " F .text" in s and kernel in s]
    assert len(found) == 1, found
    obj, name = found[0]
    text = subprocess.run([OBJDUMP, "-d", "--disassemble-symbols=" + name, obj], check=True,
                          capture_output=True, text=True).stdout
    code, base = [], None
    for line in text.splitlines():
        m = INSN.match(line)
        if not m:
            continue
        at = int(m.group(3), 16)
        base = at if base is None else base
        t = TARGET.search(line) if m.group(1).startswith(("s_branch", "s_cbranch")) else None
        code.append((at - base, m.group(1), m.group(2), int(t.group(1), 16) if t else None))
    assert len(code) > 100
    return code


def reads_in_flight_at_barriers(code, read):
    """Addresses of the barriers that some path reaches with a `read` of this
    wave issued and not known to be complete.  A wave's LDS accesses complete
    in order, so s_waitcnt lgkmcnt(n) completes a read that n or more LDS
    accesses have followed."""
    index = {a: i for i, (a, *_) in enumerate(code)}
    # per instruction: the fewest LDS accesses since the last such read, on
    # any path to it (absent: no path, None: no such read in flight)
    state, todo, bad = {0: None}, collections.deque([0]), set()
    while todo:
        i = todo.popleft()
        at, op, args, target = code[i]
        s = state[i]
        if op == "s_barrier" and s is not None:
            bad.add(at)
        if op == read:
            s = 0
        elif op.startswith("ds_"):
            s = None if s is None else min(s + 1, 15)
        elif op == "s_waitcnt":
            m = re.search(r"lgkmcnt\((\d+)\)", args)
            if m and s is not None and s >= int(m.group(1)):
                s = None
        nxt = []
        if op == "s_endpgm":
            pass
        elif op == "s_branch":
            nxt = [index[target]]
        else:
            assert not op.startswith(("s_setpc", "s_swappc", "s_call")), op
            nxt = [i + 1] + ([index[target]] if op.startswith("s_cbranch") else [])
        for j in nxt:
            if j not in state or (s is not None and (state[j] is None or s < state[j])):
                state[j] = s
                todo.append(j)
    return sorted(bad)


def test_the_walk_sees_reads_in_flight():
    ok = [(0, "ds_read_b128", "", None), (4, "ds_read_b64", "", None), (8, "s_waitcnt", "lgkmcnt(1)", None),
          (12, "s_barrier", "", None), (16, "s_endpgm", "", None)]
    assert reads_in_flight_at_barriers(ok, "ds_read_b128") == []
    late = ok[:2] + [(8, "s_barrier", "", None), (12, "s_waitcnt", "lgkmcnt(0)", None), ok[4]]
    assert reads_in_flight_at_barriers(late, "ds_read_b128") == [8]
    # the read of a loop's turn is in flight at the barrier of the next
    loop = [(0, "s_barrier", "", None), (4, "ds_read_b128", "", None), (8, "s_cbranch_scc1", "", 0),
            (12, "s_endpgm", "", None)]
    assert reads_in_flight_at_barriers(loop, "ds_read_b128") == [0]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_jacobi_rotations_are_read_before_the_barrier_that_frees_them(tk, tmp_path):
    """k_jacobi's Q wave reads the rotations of a round (double2, the kernel's
    only 16-byte LDS reads) from one of two buffers; the rotation wave writes
    that buffer again behind the next barrier, which must therefore find the
    reads complete, on every path and at every size."""
    code = disassemble(tk, tmp_path, "k_jacobi")
    assert sum(op == "ds_read_b128" for _, op, *_ in code) >= 8
    assert reads_in_flight_at_barriers(code, "ds_read_b128") == []
