"""CPU: in the gfx950 assembly of every persistent kernel, each load from the
ring is waited for before its slot is released.

A ring slot's tile is counted as loaded at the places that carry the comment
"ring slot released"; another group may store to the slot from then on.  The
loads from the ring are the buffer loads with sc1 and without nt.  Vector memory
operations complete in the order in which they were issued, so a load with k of
them behind it has arrived after `s_waitcnt vmcnt(n)`, n <= k.  A forward pass
over the control flow takes the smallest k of any path to each place.
"""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "numrs_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["-O3", "--offload-arch=gfx950", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "--cuda-device-only", "-S"]
SOURCES = ["fused_f32.hip", "fused_f64.hip", "queue_api.hip"]
MARK = "ring slot released"
NONE = 1 << 20  # no load from the ring is outstanding
VMEM = re.compile(r"(buffer|global|flat|scratch)_(load|store|atomic)")


def kernels(asm):
    """{name: [(label, [instructions])]} of the persistent kernels."""
    out, name, blocks = {}, None, None
    for line in asm.splitlines():
        m = re.match(r"(_ZN5nrfft(?:8k_fused4|7k_queue)\w+):", line)
        if m:
            name, blocks = m.group(1), [("entry", [])]
            continue
        if name is None:
            continue
        if line.startswith(".Lfunc_end"):
            out[name], name = blocks, None
            continue
        m = re.match(r"(\.LBB\w+):", line)
        if m:
            blocks.append((m.group(1), []))
            continue
        t = line.strip()
        if MARK in t:
            blocks[-1][1].append(MARK)
        elif t and not t.startswith((".", ";")):
            t = t.split(";")[0].strip()
            blocks[-1][1].append(t)
            if t.startswith(("s_cbranch", "s_branch", "s_endpgm")):  # code behind a branch: a block of its own
                blocks.append((f"after{len(blocks)}", []))
    return out


def step(k, ins):
    if ins.startswith("s_waitcnt"):
        m = re.search(r"vmcnt\((\d+)\)", ins)
        return NONE if m and int(m.group(1)) <= k else k
    if VMEM.match(ins):
        if ins.startswith("buffer_load") and re.search(r"\bsc1\b", ins) and not re.search(r"\bnt\b", ins):
            return 0
        return min(k + 1, NONE) if k < NONE else NONE
    return k


def unreleased(blocks):
    """(places marked, those with loads from the ring outstanding, loads from the ring)"""
    index = {label: i for i, (label, _) in enumerate(blocks)}
    at = [None] * len(blocks)
    at[0] = NONE
    work = [0]
    while work:
        i = work.pop()
        k, ins = at[i], blocks[i][1]
        for x in ins:
            k = step(k, x)
        nxt = []
        last = ins[-1] if ins else ""
        if last.startswith(("s_branch", "s_cbranch")):
            nxt.append(index[last.split()[-1]])
        if not last.startswith(("s_branch", "s_endpgm")) and i + 1 < len(blocks):
            nxt.append(i + 1)
        for j in nxt:
            if at[j] is None or k < at[j]:
                at[j] = k
                work.append(j)
    marks = loads = 0
    bad = []
    for (label, ins), k in zip(blocks, at):
        if k is None:
            continue
        for x in ins:
            if x == MARK:
                marks += 1
                if k < NONE:
                    bad.append((label, k))
            k = step(k, x)
            loads += k == 0
    return marks, bad, loads


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_ring_loads_arrive_before_the_release(tmp_path):
    def compile_one(src):
        out = str(tmp_path / (src + ".s"))
        subprocess.run([HIPCC, *FLAGS, os.path.join(CSRC, src), "-o", out], check=True, capture_output=True)
        with open(out) as f:
            return kernels(f.read())

    with ThreadPoolExecutor(len(SOURCES)) as pool:
        found = {}
        for part in pool.map(compile_one, SOURCES):
            found.update(part)
    assert sum("8k_fused4" in n for n in found) >= 60 and sum("7k_queue" in n for n in found) == 4
    for name, blocks in found.items():
        marks, bad, loads = unreleased(blocks)
        assert marks >= 1 and loads >= 8, (name, marks, loads)
        assert not bad, (name, bad)


def test_the_check_itself():
    load, add = "buffer_load_dwordx2 v[0:1], v9, s[0:3], 0 offen sc1", "global_atomic_add v[0:1], v2, off sc1"
    wait = "s_waitcnt vmcnt(1)"

    def run(*ins):
        return len(unreleased([("entry", list(ins))])[1])

    assert run(load, MARK, add) == 1
    assert run(load, wait, MARK) == 1                  # the load may be the one outstanding
    assert run(load, add, wait, MARK) == 0
    assert run(load, load, add, wait, MARK) == 0
    assert run(load, "s_waitcnt lgkmcnt(0)", MARK) == 1
    assert run(load.replace("sc1", "nt"), MARK) == 0   # not from the ring
    # one of two ways waits
    blocks = [("entry", [load, "s_cbranch_scc0 .LBB0_2"]), ("after1", ["s_waitcnt vmcnt(0)"]), (".LBB0_2", [MARK])]
    assert len(unreleased(blocks)[1]) == 1
