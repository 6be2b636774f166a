"""Vector registers of kernels that lose waves when their bound is passed, as
the built library's own metadata states them: a change that keeps more
values alive shows here before it shows in a frame's time."""
import os
import re
import subprocess

import pytest

import ctamd

BIN = "/opt/rocm/llvm/bin"
TOOLS = [os.path.join(BIN, t) for t in ("llvm-objcopy", "clang-offload-bundler", "llvm-readelf")]

# (kernel, bound): 512 / bound waves a SIMD.  k_pt_end's third template value
# is the pass (2 finish, 3 request), its fourth the hybrid shift.
BOUNDS = [
    (r"k_pt_endILi2ELb0E", 128),
    (r"k_pt_endILi2ELb1E", 168),
    (r"k_pt_endILi1ELb0E", 128),
    (r"k_pt_endILi3ELb1E", 64),
    (r"k_risE", 96),
    (r"k_trace_any_framesILi2ELb0E", 72),
    (r"k_trace_segmentsILi2ELb0E", 72),
    (r"k_adj_forwardILi2E", 128),
    (r"k_path_traceILi2E", 128),
]


@pytest.fixture(scope="module")
def registers(tmp_path_factory):
    """Mangled kernel name -> VGPR count."""
    if not os.path.exists(ctamd.LIB_PATH):
        pytest.skip("libctamd.so is not built")
    if not all(map(os.path.exists, TOOLS)):
        pytest.skip("no LLVM binary tools")
    tmp = tmp_path_factory.mktemp("co")
    fat = str(tmp / "fat")
    subprocess.run([TOOLS[0], "--dump-section", f".hip_fatbin={fat}", ctamd.LIB_PATH, str(tmp / "copy.so")], check=True)
    data, out = open(fat, "rb").read(), {}
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)]
    for k, at in enumerate(starts):  # one bundle per source file
        part, co = str(tmp / f"b{k}"), str(tmp / f"c{k}")
        with open(part, "wb") as fh:
            fh.write(data[at:starts[k + 1] if k + 1 < len(starts) else len(data)])
        subprocess.run([TOOLS[1], "--unbundle", "--type=o", f"--input={part}", f"--output={co}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        notes = subprocess.run([TOOLS[2], "--notes", co], capture_output=True, text=True, check=True).stdout
        for block in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", block)
            count = re.search(r"\.vgpr_count:\s+(\d+)", block)
            if name and count:
                out[name.group(1)] = int(count.group(1))
    return out


@pytest.mark.parametrize("kernel,bound", BOUNDS)
def test_registers(registers, kernel, bound):
    found = {n: v for n, v in registers.items() if re.search(kernel, n)}
    assert found, kernel
    assert max(found.values()) <= bound, found
