"""What the compiler put into the K loops of csrc/dual_gemm.hip.  A loop that keeps a ring of loads in flight waits for
memory once per K step, at the counted wait in front of the barrier; a wait of the compiler's own (for a register that a
load from before the loop may still write) or a register spilled to scratch drains the ring or adds a memory round trip to
every pass, which no test of results shows."""
import os
import re
import subprocess
import sys

import pytest

from conftest import PKG_ROOT

CSRC = os.path.join(PKG_ROOT, "csrc")
sys.path.insert(0, CSRC)
import build as csrc_build  # noqa: E402


def compile_to_assembly(source, out):
    flags = [f for f in csrc_build.FLAGS if f != "-fPIC"]
    subprocess.run([csrc_build._hipcc()] + flags + ["--cuda-device-only", "-S", source, "-o", out], check=True, capture_output=True)
    with open(out) as f:
        return f.read()


def k_loops(text):
    """(kernel, instructions) of every innermost loop with MFMAs, from the block of its first MFMA to its last MFMA or
    barrier: what lies before and behind runs where a tile ends, not in every pass."""
    for kernel, body in re.findall(r"^(_ZN\S+):[^\n]*\n(.*?)^\.Lfunc_end", text, re.M | re.S):
        lines = [line.split(";")[0].strip() for line in body.split("\n")]
        labels = {line[:-1]: i for i, line in enumerate(lines) if line.startswith(".LBB") and line.endswith(":")}
        loops = set()
        for i, line in enumerate(lines):
            m = re.match(r"s_c?branch\S* (\.LBB\S+)", line)
            if m and labels.get(m.group(1), i) < i and sum("v_mfma" in x for x in lines[labels[m.group(1)]:i]) >= 8:
                loops.add((labels[m.group(1)], i))
        for a, b in sorted(loops):
            if any(a <= c and d <= b and (c, d) != (a, b) for c, d in loops):
                continue
            first = next(i for i in range(a, b) if "v_mfma" in lines[i])
            start = max(i for i in range(a, first) if lines[i].startswith(".LBB"))
            stop = max(i for i in range(a, b) if "v_mfma" in lines[i] or lines[i].startswith("s_barrier"))
            yield kernel, [line for line in lines[start:stop + 1] if line and not line.startswith(".")]


def stray_waits(loop):
    """Waits for memory in a loop with barriers that are not the counted wait in front of one."""
    stray, waiting = [], None
    for line in loop:
        if "s_waitcnt" in line and "vmcnt" in line:
            if waiting is not None:
                stray.append(waiting)
            waiting = line
        elif line.startswith("s_barrier"):
            waiting = None
        elif waiting is not None and line.startswith(("v_mfma", "ds_", "buffer_", "global_")):
            stray.append(waiting)
            waiting = None
    return stray + ([waiting] if waiting is not None else [])


@pytest.fixture(scope="module")
def loops(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("asm") / "dual_gemm.s")
    return list(k_loops(compile_to_assembly(os.path.join(CSRC, "dual_gemm.hip"), out)))


def test_the_k_loops_are_found(loops):
    names = {k for k, _ in loops}
    for part in ("dual_gemm_kernel", "down_split_kernel", "dual_gemm_few_rows_kernel", "ffn_fused_kernel", "ffn_few_rows_norm_kernel"):
        assert any(part in n for n in names), part
    assert sum(any("lds" in x for x in body) for _, body in loops) >= 18  # loops that fill a ring


def test_a_ring_is_never_drained_in_its_k_loop(loops):
    bad = [(k, stray_waits(body)) for k, body in loops if any(x.startswith("s_barrier") for x in body) and stray_waits(body)]
    assert not bad, bad


def test_no_k_loop_spills(loops):
    bad = [(k, [x for x in body if x.startswith("scratch_")]) for k, body in loops if any(x.startswith("scratch_") for x in body)]
    assert not bad, bad


@pytest.mark.parametrize("kernel", ["dual_gemm_kernel", "down_split_kernel", "dual_gemm_few_rows_kernel", "ffn_few_rows_norm_kernel", "ffn_fused_kernel"])
def test_the_build_warns_of_a_spill_in_any_gemm_kernel(kernel, capsys):
    remark = "f.hip:1:1: remark: Function Name: _ZN2wx{}E [-Rpass]\nf.hip:1:1: remark:     ScratchSize [bytes/lane]: {} [-Rpass]\n"
    csrc_build._check_resources("dual_gemm.hip", remark.format(kernel, 96))
    assert not capsys.readouterr().err
    csrc_build._check_resources("dual_gemm.hip", remark.format(kernel, 100))
    assert kernel in capsys.readouterr().err
