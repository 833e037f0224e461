"""The pipelined GEMM kernels wait for a chunk of x by the number of younger requests in flight, so
the requests of their first chunks must be issued chunk by chunk: read from the assembly the build's
own flags give."""
import re
import shutil
import subprocess

import pytest

from if_i_could_turn_back_time_amd import build_lib as B

KERNELS = {"fourbit_gemm.hip": (r"gemm_kernel", 23), "fourbit_grad.hip": (r"grad_gemm_kernel", 8)}


def _prologues(text, pattern):
    """name -> (groups of requests before the first barrier, its vmcnt): 'x' a load into LDS, 'w' a
    load of weights, one string per run between two marks of the source (empty asm blocks)."""
    out, name, groups = {}, None, None
    for line in text.splitlines():
        line = line.strip()
        m = re.match(rf"(_Z\w*\d{pattern}I\w+):", line)
        if m:
            name, groups, allowed = m.group(1), [""], None
        elif name is None:
            continue
        elif line.startswith(";;#ASMSTART"):
            groups.append("")
        elif re.match(r"(buffer|global)_load", line):
            groups[-1] += "x" if line.endswith(" lds") else "w"
        elif m := re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)", line):
            allowed = int(m.group(1))
        elif line.startswith("s_barrier"):
            out[name] = [g for g in groups if g], allowed
            name = None
    return out


@pytest.mark.skipif(not (shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")),
                    reason="no hipcc")
@pytest.mark.parametrize("source", KERNELS)
def test_first_chunks_are_requested_in_order(source, tmp_path):
    pattern, count = KERNELS[source]
    asm = tmp_path / "k.s"
    subprocess.run([B._hipcc(), *(f for f in B.HIP_FLAGS if f != "-fPIC"), f"-I{B.INCLUDE}",
                    "--cuda-device-only", "-S", str(B.CSRC / source), "-o", str(asm)], check=True)
    found = _prologues(asm.read_text(), pattern)
    assert len(found) == count
    for name, (groups, allowed) in found.items():
        rt, ct = map(int, re.findall(r"Li(\d+)", name)[-2:])
        xs = [g.count("x") for g in groups]
        assert xs == [ct] * len(xs), (name, groups)  # one chunk's x pieces (XD = CT) per group
        # what the barrier leaves in flight is younger than the first chunk
        assert allowed <= sum(map(len, groups[1:])), (name, groups, allowed)
