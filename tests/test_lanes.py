"""Values that a kernel's lanes hold for their whole wavefront are read where the whole wavefront runs.

v_readlane reads the register of a lane whether that lane takes part or not, but a copy or a spill that the compiler makes
where only some lanes do leaves the others' behind: a read after it gives what the register held before, without any error.
The intermediate code of every kernel says where that can be: the compiler's own analysis marks the branches on which the
lanes of a wavefront part, and between such a branch and the block where all its ways meet only some of them run. A value
that is made there may be read there, one from before the branch may not."""
import re
import shutil
import subprocess

import pytest

from trips_amd import build

OPT = "/opt/rocm/llvm/bin/opt"


def _kernels(source, tmp_path):
    """{kernel: {block: (values read with readlane, values made, whether the lanes part at its end, successors)}}"""
    ll = tmp_path / "code.ll"
    subprocess.check_call([build.hipcc()] + [f for f in build.FLAGS if f != "-fPIC"] +
                          ["-Wno-unused-command-line-argument", "--cuda-device-only", "-emit-llvm", "-S", f"{build.CSRC}/{source}", "-o", str(ll)])
    text = subprocess.run([OPT, "-mtriple=amdgcn-amd-amdhsa", "-mcpu=gfx950", "-passes=print<uniformity>", "-disable-output", str(ll)],
                          check=True, capture_output=True, text=True).stderr
    out = {}
    for part in text.split("UniformityInfo for function '")[1:]:
        blocks = {}
        for name, body in re.findall(r"^BLOCK (\S+)\n(.*?)^END BLOCK", part, re.M | re.S):
            end = body[body.index("TERMINATORS"):]
            blocks[name] = (re.findall(r"llvm\.amdgcn\.readlane[^(]*\(\w+ %([\w.\-]+)", body), re.findall(r"%([\w.\-]+) =", body),
                            "DIVERGENT:" in end, re.findall(r"label %([\w.\-]+)", end))
        out[part[:part.index("'")]] = blocks
    return out


def _meeting_blocks(blocks):
    """The first block that every way out of a block leads through, per block (None: the kernel's end)."""
    order, seen = [], set()
    for root in blocks:
        stack = [(root, iter(blocks[root][3]))] if root not in seen else []
        seen.add(root)
        while stack:
            node, it = stack[-1]
            nxt = next((s for s in it if s not in seen), None)
            if nxt is None:
                order.append(node)
                stack.pop()
            else:
                seen.add(nxt)
                stack.append((nxt, iter(blocks[nxt][3])))
    every = set(blocks) | {None}
    after = {b: every for b in blocks}
    after[None] = {None}
    changed = True
    while changed:  # the blocks that all ways to the end lead through
        changed = False
        for b in order:
            new = set.intersection(*(after[s] for s in (blocks[b][3] or [None]))) | {b}
            if new != after[b]:
                after[b], changed = new, True
    return {b: next(m for m in after[b] - {b} if after[m] == after[b] - {b}) for b in blocks}


def _read_where_lanes_part(blocks):
    """The blocks that read values of the whole wavefront where only some of its lanes run."""
    meet, bad = _meeting_blocks(blocks), set()
    for b, (_, _, parts, succ) in blocks.items():
        if not parts:
            continue
        between, todo = set(), list(succ)
        while todo:
            at = todo.pop()
            if at not in between and at != meet[b]:
                between.add(at)
                todo += blocks[at][3]
        made = {value for at in between for value in blocks[at][1]}
        bad |= {at for at in between if any(value not in made for value in blocks[at][0])}
    return bad


def test_the_analysis_finds_reads_behind_a_branch_and_in_a_loop_that_lanes_leave():
    branch = {"0": (["v"], ["v"], True, ["1", "2"]), "1": (["v"], [], False, ["2"]), "2": (["v"], [], False, [])}
    assert _read_where_lanes_part(branch) == {"1"}
    own = dict(branch, **{"1": (["w"], ["w"], False, ["2"])})
    assert not _read_where_lanes_part(own)
    left = {"0": ([], ["v"], False, ["1"]), "1": (["v"], [], False, ["2"]), "2": ([], [], True, ["1", "3"]), "3": (["v"], [], False, [])}
    assert _read_where_lanes_part(left) == {"1"}
    uniform = {"0": ([], ["v"], False, ["1"]), "1": (["v"], [], False, ["1", "2"]), "2": (["v"], [], False, [])}
    assert not _read_where_lanes_part(uniform)


@pytest.mark.skipif(not shutil.which(OPT), reason="needs LLVM's opt")
@pytest.mark.parametrize("source", ["splat_forward.hip", "splat_backward.hip"])
def test_lanes_are_read_where_the_whole_wavefront_runs(source, tmp_path):
    kernels = _kernels(source, tmp_path)
    reading = [k for k, blocks in kernels.items() if any(b[0] for b in blocks.values())]
    assert reading, "no kernel with a readlane was found"
    bad = {k: found for k in reading if (found := _read_where_lanes_part(kernels[k]))}
    assert not bad
