"""The grouped GEMM's pipeline waits for a chunk's staged activations with a
counted `s_waitcnt vmcnt(N)`, N being the loads issued after that chunk's
LDS-DMA.  That count is only right if every chunk's DMAs are issued before
its weight loads; a scheduler that hoisted weight loads above the DMAs made
the wait return early (stale LDS read as activations).  This test compiles
gw_prefill.hip for gfx950 to assembly (the library's own flags) and checks,
for every instantiation of prefill_gemm_kernel, that the vector-memory loads
of each issue group come as DMAs first, then the four 16-byte weight loads.
CPU only: it needs hipcc, not a GPU."""
import os
import re
import subprocess

import pytest

from godwit_amd import build as gwbuild

SRC = os.path.join(gwbuild.CSRC, "gw_prefill.hip")


def _compile(tmp_path_factory, src):
    if not os.path.exists(gwbuild.HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("asm") / "kernel.s")
    flags = [f for f in gwbuild.FLAGS if f not in ("-shared", "-fvisibility=hidden")]
    cmd = [gwbuild.HIPCC, *flags, "-I", os.path.join(gwbuild.HERE, "..", "include"),
           "--cuda-device-only", "-S", src, "-o", out]
    subprocess.run(cmd, check=True, capture_output=True, timeout=600)
    with open(out) as f:
        return f.read()


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    return _compile(tmp_path_factory, SRC)


@pytest.fixture(scope="module")
def wide_assembly(tmp_path_factory):
    return _compile(tmp_path_factory, os.path.join(gwbuild.CSRC, "gw_prefill_wide.hip"))


def _issue_sequence(asm, name):
    body = asm[asm.index(name + ":"):]
    body = body[:body.index(".Lfunc_end")]
    seq = []
    for line in body.split("\n"):
        op = line.strip()
        if op.startswith("buffer_load") and " lds" in op:
            seq.append("X")                       # activation / scale / bias LDS-DMA
        elif op.startswith("global_load_dwordx4"):
            seq.append("W")                       # weight ring
    return "".join(seq)


def check_issue_order(asm, name):
    """First group: the scale and bias copies, then chunk 0's 2*planes DMAs,
    then its 4 weight loads; every later group: >= 2*planes DMAs, 4 loads."""
    planes = int(re.match(r"_ZN2gw19prefill_gemm_kernelILi(\d)E", name).group(1))
    seq = _issue_sequence(asm, name)
    groups = re.findall(r"X+W+", seq)
    assert groups and "".join(groups) == seq.rstrip("X"), (name, seq[:80])
    assert groups[0].count("X") >= 2 + 2 * planes, (name, seq[:40])
    for g in groups:
        assert g.count("W") == 4 and g.count("X") >= 2 * planes, (name, g)


def test_every_gemm_issues_dma_before_weights(assembly):
    names = re.findall(r"^(_ZN2gw19prefill_gemm_kernel\w+):", assembly, re.M)
    assert len(names) >= 11, names            # 8x4 / 12x4 / 8x2 shapes, planes, combine flag
    for name in names:
        check_issue_order(assembly, name)


# The wide kernel's rings (WideRing): weight chunks and input steps, by column groups.
WIDE_RINGS = {1: (3, 6), 2: (3, 3), 3: (2, 3)}


def _wide_loops(asm, name):
    """The K loops of one wide kernel, each as four steps (wait, loads): `wait` is the vmcnt
    ahead of the step's barrier, `loads` the step's memory loads in order, an LDS-DMA as its
    resource register and any other load as "G"."""
    body = asm[asm.index(name + ":"):]
    body = body[:body.index(".Lfunc_end")]
    loops = []
    for label, block in re.findall(r"^(\.LBB\w+):(.*?)(?=^\.LBB)", body, re.M | re.S):
        if not re.search(r"s_cbranch\w+ " + label + r"\b", block) or "v_mfma" not in block:
            continue
        steps, wait = [], None
        for line in block.split("\n"):
            op = line.strip()
            if op.startswith("s_waitcnt") and "vmcnt" in op:
                wait = int(re.search(r"vmcnt\((\d+)\)", op).group(1))
            elif op.startswith("s_barrier"):
                steps.append((wait, []))
            elif op.startswith("buffer_load") and " lds" in op:
                steps[-1][1].append(re.search(r"s\[(\d+):", op).group(1))
            elif op.startswith(("global_load", "flat_load", "buffer_load")):
                steps[-1][1].append("G")
        loops.append(steps)
    return loops


def _most_in_flight(groups, i):
    """Loads that may be in flight at the wait of a step (i = 0: a chunk's first), with the
    step's inputs and, at a chunk's first step, its weights landed: what was issued after
    them, when step u issues the inputs of step u + DB - 1 and, if odd, then the weights
    of chunk u // 2 + DW."""
    dw, db = WIDE_RINGS[groups]
    u = 40 + i
    issued = []
    for t in range(u):
        issued += [("X", t + db - 1)] * groups
        if t % 2:
            issued += [("W", t // 2 + dw)] * 4
    needed = [k for k, load in enumerate(issued)
              if load == ("X", u) or (i == 0 and load == ("W", u // 2))]
    assert needed
    return len(issued) - 1 - max(needed)


def test_wide_gemm_issue_order_and_waits(wide_assembly):
    """The wide kernel's K loops, as compiled: every step issues its input DMAs, a chunk's
    second step then its four weight DMAs, the scale loads ahead of both (they are not
    counted), and the vmcnt ahead of each barrier leaves no load in flight that the step
    reads."""
    names = re.findall(r"^(_ZN2gw19prefill_wide_kernel\w+):", wide_assembly, re.M)
    assert len(names) == 3, names
    for name in names:
        loops = _wide_loops(wide_assembly, name)
        # one loop for each number of column groups, and the general body's
        assert sorted(len(s[0][1]) - s[0][1].count("G") for s in loops) == [1, 1, 2, 3], name
        for steps in loops:
            assert len(steps) == 4, (name, steps)
            groups = len(steps[0][1]) - steps[0][1].count("G")
            x = steps[0][1][-1]
            for k, (wait, loads) in enumerate(steps):
                dma = [r for r in loads if r != "G"]
                assert loads == ["G"] * (loads.count("G")) + dma, (name, loads)
                assert dma[:groups] == [x] * groups, (name, loads)
                assert len(set(dma[groups:]) | {x}) == (2 if k % 2 else 1), (name, loads)
                assert len(dma) == groups + (4 if k % 2 else 0), (name, loads)
                assert wait <= _most_in_flight(groups, k % 2), (name, groups, k, wait)
