"""What the compiler made of kernels whose comments count on it, read from the built library's metadata."""
import os
import re
import shutil
import subprocess

import pytest

LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def kernel_notes(tmp_path):
    """kernel name -> its block of the code object's notes, over all code objects of the library"""
    from glide_amd import capi
    fat = tmp_path / "fatbin"
    subprocess.run([LLVM + "/llvm-objcopy", "--dump-section", ".hip_fatbin=%s" % fat, capi.LIB_PATH, str(tmp_path / "rest")], check=True)
    blob, notes = fat.read_bytes(), {}
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", blob)] + [len(blob)]
    for first, last in zip(starts, starts[1:]):
        (tmp_path / "bundle").write_bytes(blob[first:last])
        subprocess.run([LLVM + "/clang-offload-bundler", "--unbundle", "--type=o", "--input=%s" % (tmp_path / "bundle"),
                        "--output=%s" % (tmp_path / "code"), "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        text = subprocess.run([LLVM + "/llvm-readelf", "--notes", str(tmp_path / "code")], check=True, capture_output=True, text=True).stdout
        for block in text.split("\n  - .agpr_count")[1:]:
            notes[re.search(r"\.name:\s+(\S+)", block).group(1)] = block
    return notes


@pytest.mark.skipif(shutil.which(LLVM + "/clang-offload-bundler") is None, reason="no ROCm compiler tools")
def test_kmeans_kernels_use_no_private_memory(tmp_path):
    """Masked row loads are loads: a zero row kept in private memory makes them flat ones, which wait for each other."""
    kernels = {n: b for n, b in kernel_notes(tmp_path).items() if re.search(r"glide\d+kmeans", n)}
    assert len(kernels) >= 10
    for name, block in kernels.items():
        assert int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", block).group(1)) == 0, name
