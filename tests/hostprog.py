"""Small programs over the functions that the kernels share with the host,
compiled for the CPU and run there."""
import os
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "sonicsolver_amd" / "csrc"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def run(tmp_path, source: str) -> list:
    """The lines that the program prints."""
    if not shutil.which(HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "prog.hip", tmp_path / "prog"
    src.write_text(source)
    subprocess.run([HIPCC, "--offload-host-only", "-O1", "-std=c++17", f"-I{CSRC}",
                    f"-I{CSRC.parent.parent / 'include'}", "-o", str(exe), str(src)], check=True,
                   capture_output=True, text=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")[:-1]
