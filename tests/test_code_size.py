"""Host: what a kernel is compiled with is what its launches can reach, as far as its code's length shows it."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "x-attention_amd", "csrc")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def _kernel_sizes(lib, tmp):
    """Bytes of code of every kernel of the built library, by mangled name."""
    fat = os.path.join(tmp, "fat")
    subprocess.run(["objcopy", "-O", "binary", "--only-section=.hip_fatbin", lib, fat], check=True)
    data, sizes = open(fat, "rb").read(), {}
    for i, at in enumerate(m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):      # one per source file
        part, code = os.path.join(tmp, f"part{i}"), os.path.join(tmp, f"code{i}")
        open(part, "wb").write(data[at:])
        subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--type=o", "--unbundle", "--input=" + part, "--output=" + code,
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True, capture_output=True)
        out = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "-sW", code], check=True, capture_output=True, text=True).stdout
        for line in out.splitlines():
            f = line.split()
            if len(f) >= 8 and f[3] == "FUNC":
                sizes[f[7]] = int(f[2], 0)
    return sizes


def test_the_selection_of_a_few_candidates_is_compiled_for_them(tmp_path):
    """The estimate of short prompts selects among at most 16 blocks in the same kernel.  With the ways of longer rows in it too, of which
    none can be reached, it had 55 KB of code; the estimate alone has 6, and a sort of 16 lanes and a list are a few more."""
    lib = os.path.join(CSRC, "libxattn_hip.so")
    tools = [os.path.join(LLVM, t) for t in ("clang-offload-bundler", "llvm-readelf")]
    if not os.path.exists(lib) or not shutil.which("objcopy") or not all(map(os.path.exists, tools)):
        pytest.skip("needs the built library and the ROCm tools")
    fused = {n: s for n, s in _kernel_sizes(lib, str(tmp_path)).items() if "estimate_small_kernel" in n and "Lb1E" in n}
    assert len(fused) == 3 and max(fused.values()) <= 15000, fused
