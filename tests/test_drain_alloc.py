"""Downloads that run out of memory end in an exception or with fewer threads,
never in an abort (cpp/drain_alloc.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_allocation_of_a_download_may_fail(tmp_path):
    exe = str(tmp_path / "drain_alloc")
    r = subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", "-o", exe, os.path.join(HERE, "cpp", "drain_alloc.cpp")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
