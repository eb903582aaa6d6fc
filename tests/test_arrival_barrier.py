"""The arrival counters of the launches whose last workgroup writes a
sequence's seq_len / sealed / generation: a workgroup counts as arrived only
once all of its waves have read them.  Each wave reads for itself, so every
path from a kernel's entry to its arrival (the returning atomic add of thread
0) has to cross a workgroup barrier; without one a late wave reads counters
that another workgroup has already advanced, and takes another number of
barriers than the rest of its workgroup.  Such a race shows too seldom to be
tested by running: the compiled kernels' control flow is walked instead."""
import os
import re
import shutil
import subprocess

import pytest

import solidattention_amd as sa

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
HEADER = re.compile(r"^([0-9a-f]+) <(.+)>:$")
INSTR = re.compile(r"^\s+(\S+)(.*?)// ([0-9A-F]+):")
TARGET = re.compile(r"<[^>]+?(?:\+0x([0-9a-f]+))?>\s*$")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel name: [(address, mnemonic, operands, branch target or None)]} of the gfx950 code of libsa_hip.so."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    where = tmp_path_factory.mktemp("code")
    sa.lib()  # built
    shutil.copy(os.path.join(os.path.dirname(sa.__file__), "..", "libsa_hip.so"), where / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=where, check=True, capture_output=True)
    found = {}
    for f in sorted(os.listdir(where)):
        if "gfx950" not in f or os.path.getsize(where / f) == 0:
            continue
        text = subprocess.run([OBJDUMP, "-d", f], cwd=where, check=True, capture_output=True, text=True).stdout
        code, base = None, 0
        for line in text.splitlines():
            head = HEADER.match(line)
            if head:
                base = int(head.group(1), 16)
                wanted = "decode_kernel" in head.group(2) or "append_seal_online_kernel" in head.group(2)
                code = found.setdefault(head.group(2), []) if wanted else None
                continue
            ins = INSTR.match(line) if code is not None else None
            if ins:
                target = None
                if ins.group(1).startswith(("s_cbranch", "s_branch")):
                    target = base + int(TARGET.search(line).group(1) or "0", 16)
                code.append((int(ins.group(3), 16), ins.group(1), ins.group(2), target))
    assert found
    return found


def is_arrival(mnemonic, operands):
    return mnemonic.startswith(("global_atomic_add", "flat_atomic_add")) and " sc0" in operands


def reached_without_barrier(code):
    """The addresses of arrivals that some path from the entry reaches without an s_barrier."""
    at = {ins[0]: i for i, ins in enumerate(code)}
    seen, todo, bad = set(), [0], []
    while todo:
        i = todo.pop()
        while i < len(code) and i not in seen:
            seen.add(i)
            address, mnemonic, operands, target = code[i]
            assert not mnemonic.startswith(("s_setpc", "s_swappc", "s_call")), "a call: not followed"
            if is_arrival(mnemonic, operands):
                bad.append(hex(address))
            if mnemonic in ("s_barrier", "s_endpgm") or is_arrival(mnemonic, operands):
                break
            if target is not None:
                todo.append(at[target])
                if mnemonic == "s_branch":
                    break
            i += 1
    return bad


@pytest.mark.parametrize("family", ["append_seal_online_kernel", "decode_kernel"])
def test_arrival_behind_a_barrier(kernels, family):
    members = {n: c for n, c in kernels.items() if family in n and any(is_arrival(i[1], i[2]) for i in c)}
    assert members, family
    bad = {n: b for n, b in ((n, reached_without_barrier(c)) for n, c in members.items()) if b}
    assert not bad, f"arrivals reached without a barrier: {bad}"


def masked_barriers(code):
    """The addresses of barriers behind a narrowing of the lane mask that is not undone before them."""
    bad, narrowed = [], False
    for address, mnemonic, operands, _ in code:
        if "_saveexec_" in mnemonic:
            narrowed = True
        elif operands.strip().startswith("exec,") or mnemonic == "s_branch":  # undone, or another path's code follows
            narrowed = False
        elif mnemonic == "s_barrier" and narrowed:
            bad.append(hex(address))
    return bad


def test_every_lane_reaches_the_same_barriers(kernels):
    """A workgroup barrier stands in code that all of the workgroup's waves
    run, not in the branch of some of its lanes (two halves of a workgroup at
    two barriers only pair up for as long as the compiler keeps each branch's
    skip)."""
    bad = {n: b for n, b in ((n, masked_barriers(c)) for n, c in kernels.items()) if b}
    assert not bad, f"barriers under a lane mask: {bad}"
