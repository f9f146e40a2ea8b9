"""What the build needs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _dry_run(*targets):
    return subprocess.run(["make", "-C", os.path.join(ROOT, "ops_cv_amd", "csrc"), "-n", "-B", "PYTHON=/nonexistent", *targets],
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, check=True).stdout


def test_library_builds_without_pytorch():
    out = _dry_run()
    assert "libopscv_amd.so" in out and "libopscv_bench.so" in out
    assert "torch_helpers" not in out and "/nonexistent" not in out
    assert "torch_helpers" in _dry_run("all", "helpers")
