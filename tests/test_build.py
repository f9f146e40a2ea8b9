"""What the build needs, and what is said when the torch helpers' native side is missing."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _dry_run(*targets):
    return subprocess.run(["make", "-C", os.path.join(ROOT, "ops_cv_amd", "csrc"), "-n", "-B", "PYTHON=/nonexistent", *targets],
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, check=True).stdout


def test_library_builds_without_pytorch():
    out = _dry_run()
    assert "libopscv_amd.so" in out and "libopscv_bench.so" in out
    assert "torch_helpers" not in out and "/nonexistent" not in out
    assert "torch_helpers" in _dry_run("all", "helpers")


@pytest.mark.parametrize("content,said", [(None, "is not built"), (b"not a library", "does not load")])
def test_missing_and_unloadable_helpers(tmp_path, content, said):
    package = tmp_path / "ops_cv_amd"
    package.mkdir()
    for name in ("__init__.py", "aclnn.py", "libopscv_amd.so"):
        shutil.copy(os.path.join(ROOT, "ops_cv_amd", name), package / name)
    if content is not None:
        (package / "_torch_helpers.so").write_bytes(content)
    code = "import torch; from ops_cv_amd import aclnn; t = torch.zeros(1, 1, 2, 2); aclnn.grid_sampler2d(t, t)"
    p = subprocess.run([sys.executable, "-c", code], cwd=tmp_path, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    last = p.stderr.strip().splitlines()[-1]
    assert p.returncode != 0 and last.startswith("RuntimeError") and said in last and "ops_cv_amd.build" in last
