"""The matrix products' counted waits (models_amd/csrc/jma_qgemm.hip) against the code the compiler
emits. A step's barrier waits until at most N of the wave's loads are in flight, N counted by hand
from the source: if the compiler merged, dropped or moved a load, N could let the barrier pass before
the next step's activations are in LDS, silently. Here every kernel instance is compiled to gfx950
assembly with the library's own flags, and the emitted loads and waits of the prologue and of three
rounds of its main loop are played through the hardware's in-order load counter."""

import os
import re
import subprocess

import pytest

from models_amd import build as B

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INSTANCES = 16  # qgemm_kernel and qkgemm_kernel: 5 formats x 3 tiles; q6gemm_kernel


def emitted(text):
    """Per kernel instance: (label, [ops]) with ops 'a' (16-byte load to LDS), 's' (4-byte load to LDS),
    'l' (any other vector-memory access), ('w', n) (wait for n in flight), 'b' (barrier), 'j' (branch),
    '#' (label)."""
    kernels, ops = {}, None
    for line in text.splitlines():
        start = re.match(r"(_ZN3jma\d+q\w*gemm_kernel\w*):", line)
        if start:
            ops = kernels.setdefault(start.group(1), [])
            continue
        if ops is None:
            continue
        code = line.split(";")[0].strip()
        if code.startswith("s_endpgm"):
            ops = None
        elif re.match(r"\.LBB\w+:", code):
            ops.append("#")
        elif code.startswith(("s_cbranch", "s_branch")):
            ops.append("j")
        elif code.startswith("s_barrier"):
            ops.append("b")
        elif re.match(r"(buffer|global|flat|scratch)_", code):
            to_lds = re.search(r"\blds\b", code)
            ops.append("l" if not to_lds else "a" if "dwordx4" in code else "s")
        elif code.startswith("s_waitcnt"):
            n = re.search(r"vmcnt\((\d+)\)", code)
            if n:
                ops.append(("w", int(n.group(1))))
    return kernels


def loop_segments(ops, steps):
    """The prologue and the main loop's steps, each up to and with its barrier."""
    cuts = [i for i, op in enumerate(ops) if op == "b"]
    assert len(cuts) == steps + 1, f"{len(cuts)} barriers, not a prologue's and {steps} steps'"
    prologue, loop = ops[:cuts[0] + 1], ops[cuts[0] + 1:cuts[-1] + 1]
    assert loop.count("#") == 1 and "j" not in loop[loop.index("#"):], "the loop is not straight-line code"
    tail = ops[cuts[-1] + 1:]
    assert not set("asl") & set(tail[:tail.index("j")]), "a load after the loop's last barrier"
    loop = loop[loop.index("#") + 1:]
    segments, at = [prologue], 0
    for _ in range(steps):
        end = loop.index("b", at) + 1
        segments.append(loop[at:end])
        at = end
    return segments


def check(ops, steps, pieces, scale_step, scale_read, scales_before):
    """pieces: 16-byte loads of one step's activations a wave makes; scale_step: the step whose 4-byte
    loads bring the activation scales that step scale_read (counted on from it) reads, or None;
    scales_before: whether the prologue has loaded the first ones."""
    segments = loop_segments(ops, steps)
    queue, arrived, issued, want_scales = [], 0, 0, []
    scales_issued = scales_arrived = 0
    for i in range(1 + 3 * steps):
        step = i - 1  # the prologue counts as step -1: its barrier opens step 0
        for op in segments[0] if i == 0 else segments[1 + step % steps]:
            if op in ("a", "s", "l"):
                queue.append(op)
                issued += op == "a"
                scales_issued += op == "s"
            elif isinstance(op, tuple):
                while len(queue) > op[1]:
                    done = queue.pop(0)
                    arrived += done == "a"
                    scales_arrived += done == "s"
        if scale_step is not None:
            if i == 0 and scales_before:
                want_scales.append((-1, scales_issued))
            elif i and step % steps == scale_step:
                want_scales.append((step - scale_step + scale_read - 1, scales_issued))
            for at, count in want_scales:
                assert at != step or scales_arrived >= count, f"step {step + 1} reads activation scales in flight"
        assert issued == pieces * (step + 4), f"step {step}: {issued} activation loads issued"
        assert arrived >= pieces * (step + 2), f"step {step + 1}'s activations are in flight at its barrier"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("isa") / "qgemm.s"
    flags = [f for f in B.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    run = subprocess.run([B.hipcc(), *flags, "-I", os.path.join(ROOT, "include"), "--cuda-device-only", "-S",
                          os.path.join(ROOT, "models_amd", "csrc", "jma_qgemm.hip"), "-o", str(out)],
                         capture_output=True, text=True)
    assert run.returncode == 0, run.stderr
    return emitted(out.read_text())


def test_every_step_waits_for_its_activations(kernels):
    assert len(kernels) == INSTANCES, sorted(kernels)
    for name, ops in kernels.items():
        try:
            if "q6gemm" in name:
                check(ops, 8, 1, 5, 8, True)
                continue
            fmt, bt, _, nb, nw = (int(x) for x in re.findall(r"Li(\d+)E", name))
            waves, per_step = nb * nw, bt * nb * 2  # 1 KB pieces of 32 x bt x nb activation rows
            pieces = -(-per_step // waves)
            if fmt in (2, 4):
                check(ops, 8, pieces, 4, 7, False)
            else:
                check(ops, 4, pieces, None, None, False)
        except AssertionError as e:
            raise AssertionError(f"{name}: {e}") from None


def test_a_merged_load_is_noticed(kernels):
    """The walk fails where one register load of a step is missing (planted in the parsed listing)."""
    name = next(n for n in kernels if "qgemm_kernelILi0ELi1ELi1ELi2ELi2E" in n)
    ops = list(kernels[name])
    bars = [i for i, op in enumerate(ops) if op == "b"]
    for lo, hi in zip(bars, bars[1:]):  # every step loses one, as a merge in the source's load() would
        at = next(i for i in range(lo, hi) if ops[i] == "l")
        ops[at] = "-"
    with pytest.raises(AssertionError, match="in flight at its barrier"):
        check([op for op in ops if not isinstance(op, tuple) or op[1] == 8], 4, 1, None, None, False)
