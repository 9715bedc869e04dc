"""The packing threads of the host-array entries (mg_hostpack.hpp), compiled for
the CPU: fields through two buffers in turn with one to eight threads, and with
threads (EAGAIN) or memory (std::bad_alloc) refused after some have started, which
must neither end the process nor lose a piece."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_packing_threads(tmp_path):
    exe = tmp_path / "hostpack_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-pthread", "-I", os.path.join(ROOT, "multiflow3d_amd", "csrc"),
                    os.path.join(ROOT, "tests", "hostpack_check.cpp"), "-o", str(exe), "-ldl"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
