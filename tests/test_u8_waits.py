"""Requests and waits of the tiled u8 kernels, read from the device code of the built library's gemm_mfma object.  A slice of K
ends with one counted wait and a barrier; the count has to match what the compiler left of the slice's requests, where it
put them and in which order, or a transfer to LDS is read before it has landed (count too high) or awaited a slice early
(too low).  No device needed."""
import os
import re
import subprocess

import pytest

from adrastea_amd import build

OBJECT = os.path.join(build.LIBDIR, "gemm_mfma.o")
TOOLS = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin")


@pytest.fixture(scope="module")
def device_code(tmp_path_factory):
    if not (os.path.exists(OBJECT) and os.path.exists(os.path.join(TOOLS, "llvm-objdump"))):
        pytest.skip("the library's objects or the LLVM tools are not here")
    tmp = tmp_path_factory.mktemp("device_code")
    bundle, code = str(tmp / "bundle"), str(tmp / "code.o")
    for cmd in (["llvm-objcopy", "--dump-section", ".hip_fatbin=" + bundle, OBJECT, os.devnull],
                ["clang-offload-bundler", "--unbundle", "--type=o", "--input=" + bundle,
                 "--targets=hipv4-amdgcn-amd-amdhsa--" + build.ARCH, "--output=" + code]):
        subprocess.run([os.path.join(TOOLS, cmd[0]), *cmd[1:]], check=True, capture_output=True)
    r = subprocess.run([os.path.join(TOOLS, "llvm-objdump"), "-d", code], check=True, capture_output=True, text=True)
    return r.stdout


def slices(device_code, kernel):
    """Per slice of the one kernel whose mangled name contains `kernel`, wherever it lies: its requests in order (A:
    a transfer to LDS, W: weights or scales) and the count of its last wait."""
    names = set(re.findall(rf"^[0-9a-f]+ <(_Z\w*{kernel}\w*)>:", device_code, re.M))
    assert len(names) == 1, names
    body = device_code.split(f"<{names.pop()}>:", 1)[1].split("s_endpgm", 1)[0]
    found, requests, count = [], "", None
    for line in body.splitlines():
        line = line.split("//")[0].strip()
        assert not line.startswith("scratch"), line   # (a spilled register would be a request as well)
        if line.startswith("buffer_load"):
            requests += "A" if line.endswith(" lds") else "W"
        elif line.startswith("s_waitcnt"):
            left = re.search(r"vmcnt\((\d+)\)", line)
            count = int(left.group(1)) if left else count
        elif line == "s_barrier":
            found.append((requests, count))
            requests, count = "", None
    prologue = found.pop(0)
    return prologue, [s for s in found if "A" in s[0]]


# (rows, columns, wavefronts along them, groups)
@pytest.mark.parametrize("tile", [(256, 192, 4, 2, 1), (256, 128, 4, 2, 1), (128, 128, 4, 2, 1), (128, 64, 2, 2, 1),
                                  (64, 64, 2, 2, 1), (128, 64, 2, 2, 2), (64, 64, 2, 2, 4),
                                  (192, 192, 2, 4, 1), (192, 128, 2, 4, 1), (96, 96, 3, 2, 1)],
                         ids=lambda t: "%dx%d_%dx%d_k%d" % t)
def test_a_slice_waits_for_the_transfers_of_the_slice_before(device_code, tile):
    rows, columns, wm, wn, groups = tile
    transfers = rows * 8 // (wm * wn * 64)           # 16-byte chunks of a slice of 64 per lane
    weights = 2 * (columns * 8 // (wm * wn * 64))    # eight weights and their scale per chunk
    prologue, loop = slices(device_code, f"gemm_nt_u8_kernelILi{rows}ELi{columns}ELi{wm}ELi{wn}ELb1ELi64ELi{groups}E")
    # two slices' transfers and three's weights; the youngest requests are the second slice's transfers, and the wait
    # leaves nothing but them
    assert sorted(prologue[0]) == sorted("A" * 2 * transfers + "W" * 3 * weights)
    assert prologue[0].endswith("A" * transfers) and prologue[1] == transfers
    # Six slices in the loop and five behind it, the last two of which request no weights (no slice uses them).  All
    # requests of weights come behind the transfers of their slice: what is younger than the transfers of the slice before
    # is at least one slice's weights and one slice's transfers, the count of the wait.
    live, dead = "A" * transfers + "W" * weights, "A" * transfers
    assert [requests for requests, _ in loop].count(live) == 9, loop
    assert [requests for requests, _ in loop].count(dead) == 2 and len(loop) == 11, loop
    assert {count for _, count in loop} == {transfers + weights}
