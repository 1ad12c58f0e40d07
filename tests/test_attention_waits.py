"""Waits of the fused attention kernels, checked on the assembly the compiler makes of attention.hip: the
barriers are written as assembly, so the compiler adds no wait in front of them, and a wavefront
whose LDS reads are still in flight at a barrier reads what another one transfers to that place
behind it.  No device needed."""
import os
import re
import subprocess

import pytest

from adrastea_amd import build


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc here")
    out = tmp_path_factory.mktemp("asm") / "attention.s"
    flags = [f for f in build.CXXFLAGS if f != "-fPIC"]
    subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-S", os.path.join(build.CSRC, "attention.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    return out.read_text()


def instructions(assembly, kernel):
    """The instructions of the one kernel whose mangled name contains `kernel`, in program order."""
    names = set(re.findall(rf"^(_Z\w*{kernel}\w*):", assembly, re.M))
    assert len(names) == 1, names
    body = assembly.split(names.pop() + ":", 1)[1].split("s_endpgm", 1)[0]
    return [line.split(";")[0].strip() for line in body.splitlines()]


def reads_in_flight_at_first_barrier(lines):
    flying = reads = 0
    for line in lines:
        if line.startswith("ds_read"):
            flying += 1
            reads += 1
        elif line.startswith("s_waitcnt"):
            left = re.search(r"lgkmcnt\((\d+)\)", line)
            if left or line.split()[1:] == ["0"]:
                flying = min(flying, int(left.group(1)) if left else 0)
        elif line == "s_barrier":
            return reads, flying
    raise AssertionError("no barrier")


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("groups", [1, 2])
def test_query_rows_are_read_before_their_place_is_overwritten(assembly, d, groups):
    """The query rows pass through the buffers of the V tiles; behind the first barrier any wavefront may
    transfer the first V tile there, one without rows of its own at once."""
    reads, flying = reads_in_flight_at_first_barrier(
        instructions(assembly, f"attention_fwd_kernelILi{d}ELi{groups}ELb0E"))
    assert reads == d // 16  # (the fragments of Q: nothing else is read up to there)
    assert flying == 0
