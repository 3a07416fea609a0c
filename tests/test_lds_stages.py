"""Kernels that copy operands straight into LDS stages while other waves still read (raw barriers, which wait for nothing by
themselves). Such a kernel refills, behind a barrier, the stage that was read before the barrier before that one; so in the
compiled code no wave may pass a barrier with reads of LDS on their way that it began before the barrier before. Found by
walking the kernel's instructions along every branch; a wave's LDS reads finish in their order."""
import os
import re
import shutil
import subprocess

import pytest

from return_amd.kernels import build

MANY = 64


def _compiled(source, tmp_path):
    out = str(tmp_path / "kernel.s")
    subprocess.run([build._hipcc(), *build.FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, source), "-o", out],
                   check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    with open(out) as f:
        return f.read()


def _kernels(text):
    """name -> blocks in their order, each (label, instructions)."""
    found, name, blocks = {}, None, []
    for line in text.splitlines():
        line = line.split(";")[0].strip()
        label = re.match(r"([\w.$]+):$", line)
        if label and label.group(1).startswith("_Z"):
            name, blocks = label.group(1), [("", [])]
        elif line.startswith(".Lfunc_end"):
            if name:
                found[name] = blocks
            name = None
        elif name and label:
            blocks.append((label.group(1), []))
        elif name and line and not line.startswith("."):
            blocks[-1][1].append(line)
    return found


def unfinished_reads(blocks, behind_same=False):
    """(copies into LDS, those behind a barrier that a wave may have passed with old reads unfinished: (block, instruction,
    reads)). State along a path: reads a wave may have on their way, those of them that it began before the last barrier,
    those that it had begun before the barrier before when it passed the last one. behind_same: for a kernel that refills a
    stage behind the very barrier in front of which it was read: no read at all may be on its way at that barrier."""
    at = {label: i for i, (label, _) in enumerate(blocks)}
    state = {0: (0, 0, 0)}
    todo, bad, copies = [0], {}, set()
    while todo:
        i = todo.pop()
        reads, old, passed = state[i]
        ends, far = False, None

        def on(j):
            was = state.get(j, (0, 0, 0))
            new = tuple(max(p) for p in zip((reads, old, passed), was))
            if j not in state or new != was:
                state[j] = new
                todo.append(j)

        for ins in blocks[i][1]:
            op = ins.split()[0]
            if op.startswith("ds_read"):
                reads = min(reads + 1, MANY)
            elif op == "s_waitcnt":
                left = re.search(r"lgkmcnt\((\d+)\)", ins)
                if left:                                   # the oldest finish first
                    now = min(reads, int(left.group(1)))
                    old, reads = max(0, old - (reads - now)), now
            elif op == "s_barrier":
                passed, old = reads if behind_same else old, reads
            elif op.startswith("buffer_load") and re.search(r"\blds\b", ins):
                copies.add((i, ins))
                if passed:
                    bad[blocks[i][0], ins] = passed
            elif op.startswith("s_cbranch"):
                on(at[ins.split()[1]])
            elif op in ("s_add_u32", "s_add_i32") and ".LBB" in ins:      # the address of a branch that goes far
                far = re.search(r"\.LBB\w+", ins).group()
            elif op in ("s_branch", "s_setpc_b64"):
                on(at[ins.split()[1] if op == "s_branch" else far])
                ends = True
                break
            elif op == "s_endpgm":
                ends = True
                break
        if not ends and i + 1 < len(blocks):
            on(i + 1)
    return len(copies), sorted((*k, n) for k, n in bad.items())


def test_the_walk_finds_what_it_is_for():
    """Stages in turn: a step's reads finished before the barrier behind the next step's, and only behind that one."""
    def loop(wait):
        return [("", []), ("top", ["s_barrier", "buffer_load_dwordx4 v1, s[0:3], s9 offen lds", "ds_read_b128 v[2:5], v6",
                                   "ds_read_b128 v[7:10], v6 offset:1024", *wait, "s_cbranch_scc1 top"]),
                ("end", ["s_waitcnt lgkmcnt(0)", "s_endpgm"])]
    for wait, good in (([], False), (["s_waitcnt lgkmcnt(3)"], False), (["s_waitcnt vmcnt(4) lgkmcnt(2)"], True),
                       (["s_waitcnt vmcnt(0)"], False), (["s_waitcnt lgkmcnt(0)"], True)):
        copies, bad = unfinished_reads(loop(wait))
        assert copies == 1 and (not bad) == good, (wait, bad)


@pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")), reason="no hipcc")
@pytest.mark.parametrize("source", ["moe_tile.hip", "gemm_tile.hip", "gemm_rows.hip"])
def test_no_stage_is_refilled_before_it_is_read(source, tmp_path):
    kernels = {n: b for n, b in _kernels(_compiled(source, tmp_path)).items() if any(" lds" in i for _, c in b for i in c)}
    assert kernels
    for name, blocks in kernels.items():
        copies, bad = unfinished_reads(blocks)
        assert copies > 0
        assert not bad, (name, bad[:8], len(bad))


@pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")), reason="no hipcc")
@pytest.mark.parametrize("source", ["moe_tile.hip", "gemm_rows.hip"])
def test_stages_refilled_behind_the_barrier_they_are_read_before(source, tmp_path):
    kernels = {n: b for n, b in _kernels(_compiled(source, tmp_path)).items() if any(" lds" in i for _, c in b for i in c)}
    for name, blocks in kernels.items():
        copies, bad = unfinished_reads(blocks, behind_same=True)
        assert copies > 0 and not bad, (name, bad[:8], len(bad))
