"""A traversal step at a leaf reads records of that leaf only (tests/cpp/leaf_record.cpp)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "cpp", "leaf_record.cpp")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def test_records_read_lie_in_the_leaf(tmp_path):
    exe = str(tmp_path / "leaf_record")
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", SRC, "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "every record read lies in its leaf" in r.stdout
