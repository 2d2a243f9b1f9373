"""The rule that chooses the small-tile GEMM's launch, on the CPU over the
extremes of its range (tests/cpp/gemm_plan.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_gemm_plans_stay_launchable(tmp_path):
    exe, pkg = str(tmp_path / "gemm_plan"), os.path.join(ROOT, "lite_ssm_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROOT}/include", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "gemm_plan.cpp"), "-o", exe, f"-L{pkg}", "-llssm_hip",
                    "-L/opt/rocm/lib", "-lamdhip64", f"-Wl,-rpath,{pkg}", "-Wl,-rpath,/opt/rocm/lib"],
                   check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
