"""Device buffers checked on the host (no GPU), in small programs that link the
library and replace its device pool (and, where needed, launches and waits)."""
import os
import subprocess

from gsparc_amd import build as b
from gsparc_amd import sptc

HERE = os.path.dirname(os.path.abspath(__file__))


def _run(source, tmp_path):
    sptc.lib()
    exe = str(tmp_path / source.split(".")[0])
    subprocess.run([b.HIPCC, "-x", "hip", "--offload-host-only", f"--offload-arch={b.ARCH}",
                    "-O1", "-std=c++17", "-I", b.CSRC, "-I",
                    os.path.join(b.REPO_DIR, "include"), os.path.join(HERE, source),
                    "-o", exe, "-L", b.LIB_DIR, "-lsptc_hip", f"-Wl,-rpath,{b.LIB_DIR}"],
                   check=True, capture_output=True, text=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=60,
                       env={k: v for k, v in os.environ.items() if not k.startswith("SPTC_")})
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout


def test_large_sort_after_segmented_sorts(tmp_path):
    """A workspace that segmented sorts used before must still hold all buffers of
    a large sort."""
    out = _run("workspace_check.cpp", tmp_path)
    assert "BAD" not in out and "ok" in out


def test_growing_plan_waits_for_the_chunk_before(tmp_path):
    """A chunk whose tables outgrow the plan's gives the old ones back only after
    the kernels of the chunk before have been waited for."""
    assert "0 of them too early" in _run("plan_growth_check.cpp", tmp_path)
