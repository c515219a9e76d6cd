"""CPU: the rule by which the attention kernel's long lists are cut keeps every q-block within its share of the pieces, covers
every list exactly once and needs a bounded workspace.  Compiled for the host from the kernels' own header; nothing runs on
a GPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_cut_lists_fit_their_share(tmp_path):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not (os.path.exists(hipcc) or shutil.which(hipcc)):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "attn_plan_check")
    src = os.path.join(ROOT, "tests", "host", "attn_plan_check.cpp")
    cmd = [hipcc, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17",
           "-I" + os.path.join(ROOT, "x-attention_amd", "csrc"), "-I" + os.path.join(ROOT, "include"), src, "-o", exe]
    build = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert build.returncode == 0, build.stdout
    run = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    print(run.stdout)
    assert run.returncode == 0, run.stdout


def test_workspace_of_the_operator_is_bounded():
    """What lists to be cut add to the operator's temporaries, over the lengths they are cut for."""
    from xattn.src import hip_backend as hb

    lib = hb.lib()
    for heads in (1, 8, 24, 32, 64):
        for q_len in (64, 500, 2048, 4096, 8000, 8192, 16384, 32768):
            for cache in (0, 8192, 65536, 131072):
                q_blocks = (q_len + 127) // 128
                assert lib.xattn_block_sparse_workspace_bytes(heads, q_len, q_len + cache, q_blocks, q_blocks) <= 200 << 20
    # lists of a prompt of up to 8192 tokens
    assert lib.xattn_block_sparse_workspace_bytes(32, 4096, 4096, 32, 32) <= 90 << 20
