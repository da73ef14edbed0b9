"""The batched GEMM's workspace on the host (tests/c/gemm_workspace.cpp, which
includes csrc/capi_gemm.cpp and counts the allocations and launches): sized to
the call, captured or not, and a call that cannot have it runs on what is there
instead of failing; and how many rows the prefill's buffers get."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_workspace_is_sized_to_the_call_and_never_needed(tmp_path):
    exe = str(tmp_path / "gemm_workspace")
    rocm = os.environ.get("ROCM", "/opt/rocm")
    r = subprocess.run([rocm + "/llvm/bin/clang++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I" + rocm + "/include",
                        os.path.join(ROOT, "tests", "c", "gemm_workspace.cpp"), "-o", exe, "-lpthread"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "workspace ok" in r.stdout, r.stdout + r.stderr
