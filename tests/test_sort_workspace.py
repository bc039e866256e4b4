"""The sort workspace's sizes, checked on the host (no GPU): a workspace that
segmented sorts used before must still hold all buffers of a large sort."""
import os
import subprocess

from gsparc_amd import build as b
from gsparc_amd import sptc

HERE = os.path.dirname(os.path.abspath(__file__))


def test_large_sort_after_segmented_sorts(tmp_path):
    sptc.lib()
    exe = str(tmp_path / "workspace_check")
    subprocess.run([b.HIPCC, "-x", "hip", "--offload-host-only", f"--offload-arch={b.ARCH}",
                    "-O1", "-std=c++17", "-I", b.CSRC, "-I",
                    os.path.join(b.REPO_DIR, "include"), os.path.join(HERE, "workspace_check.cpp"),
                    "-o", exe, "-L", b.LIB_DIR, "-lsptc_hip", f"-Wl,-rpath,{b.LIB_DIR}"],
                   check=True, capture_output=True, text=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60,
                       env={k: v for k, v in os.environ.items() if not k.startswith("SPTC_")})
    assert p.returncode == 0, p.stdout + p.stderr
    assert "BAD" not in p.stdout and "ok" in p.stdout
