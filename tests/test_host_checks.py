"""Checks of the engines' host code on a HIP runtime in host memory
(tests/native/fake_hip.hpp): allocations that fail, in which order buffers
come and go, and which device launches are made on."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CHECKS = {"rank_memory_check": "rank memory ok", "sorted_memory_check": "sorted memory ok",
          "batch_layout_check": "batch layout ok", "rebind_check": "rebind ok",
          "group_check": "groups ok"}


@pytest.mark.parametrize("name", list(CHECKS))
def test_host_code_on_a_runtime_in_host_memory(name, tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not installed")
    exe = tmp_path / name
    # Wrappers of kernels that a check never calls stay unresolved.
    subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-std=c++17", "-O1",
                    "-I", str(ROOT / "multigpubfs_amd" / "csrc"), "-I", str(ROOT / "include"),
                    str(ROOT / "tests" / "native" / f"{name}.cpp"), "-o", str(exe),
                    "-Wl,--unresolved-symbols=ignore-all"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert CHECKS[name] in out.stdout
