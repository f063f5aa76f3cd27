"""CAM_MI355X_LIB names the build of the kernel library that everything in the package calls: the ctypes binding, the C++
module behind ops.py and the torch operators.  No GPU is needed: which file is mapped is what counts."""
import os
import shutil
import subprocess
import sys

import pytest

import umdk_original_amd
from umdk_original_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(umdk_original_amd.__file__)))

PROGRAM = """
import umdk_original_amd as cam
from umdk_original_amd import ops
ops._native()
print("torch ops:", ops._torch_lib if isinstance(ops._torch_lib, str) else "python")
with open("/proc/self/maps") as f:
    for path in sorted({line.split()[-1] for line in f if "libcam_" in line}):
        print("mapped:", path)
"""


def _run(lib):
    env = dict(os.environ, CAM_MI355X_LIB=str(lib))
    return subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, env=env, stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                          text=True, timeout=300)


@pytest.mark.parametrize("torch_ops", [True, False])
def test_the_named_library_is_the_only_one(tmp_path, torch_ops):
    other = tmp_path / "libcam_other.so"
    shutil.copy(build.LIB_PATH, other)
    if torch_ops:
        shutil.copy(build.TORCH_OPS_PATH, tmp_path)
    p = _run(other)
    assert p.returncode == 0, p.stderr
    mapped = [line.split()[-1] for line in p.stdout.splitlines() if line.startswith("mapped:")]
    assert str(other) in mapped and build.LIB_PATH not in mapped
    assert ("torch ops: cpp" if torch_ops else "torch ops: python") in p.stdout
