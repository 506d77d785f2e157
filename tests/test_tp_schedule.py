"""Automatic schedules of the tensor-product kernel are resolved once, not at
every launch, and sfk_op_tile_shape names their tile (CPU: the launch
descriptors an operator makes)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sum_factorization_kernels_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def run_check(name, tmp_path):
    if not os.path.exists(os.path.join(PKG, "libsfk.so")):
        pytest.skip("libsfk.so not built")
    exe = str(tmp_path / name)
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(PKG, "csrc"), "-isystem", os.path.join(ROCM, "include"),
                        os.path.join(ROOT, "tests", "cpp", name + ".cc"), "-o", exe, "-L" + PKG, "-lsfk",
                        "-L" + os.path.join(ROCM, "lib"), "-lamdhip64", "-Wl,-rpath," + PKG,
                        "-Wl,-rpath," + os.path.join(ROCM, "lib")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_automatic_schedules(tmp_path):
    run_check("tp_schedule_check", tmp_path)


def test_planned_tile_is_accepted(tmp_path):
    run_check("tp_plan_check", tmp_path)
