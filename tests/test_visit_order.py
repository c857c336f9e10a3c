"""The 4-wide triangle records visit leaves in the reference's depth-first order for every direction octant
(tests/cpp/visit_order.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "cpp", "visit_order.cpp")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_wide_records_keep_the_reference_order(tmp_path):
    exe = str(tmp_path / "visit_order")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                    f"-I{ROCM}/include", SRC, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "visit the leaves in the reference's order" in r.stdout
