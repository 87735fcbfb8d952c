"""What wide rows do as device memory runs out: the column index of B, then the windows' lists are
done without, in a plan's recording and capture passes alike (tests/sanitize/wide_memory.cpp runs
the host orchestrator with host memory and no kernels, under ASan and UBSan).  No GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_forms_of_wide_rows_by_memory(tmp_path):
    exe = tmp_path / "wide_memory"
    subprocess.check_call(["g++", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-g", "-O1",
                           "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                           os.path.join(ROOT, "tests", "sanitize", "wide_memory.cpp"),
                           os.path.join(ROOT, "hsmu-spgemm_amd", "csrc", "api.cpp"), "-o", str(exe), "-pthread"])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "WIDE_MEMORY_OK" in out.stdout
