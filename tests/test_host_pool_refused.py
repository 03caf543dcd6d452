"""The worker pool where the system refuses threads (tests/host_pool_refused_main.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_pool_works_with_the_threads_it_got(tmp_path):
    exe = str(tmp_path / "pool")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "ramses-cpp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host_pool_refused_main.cpp"), "-o", exe], check=True)
    env = dict(os.environ)
    env.pop("LD_PRELOAD", None)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60, env=env)
    assert out.returncode == 0 and "pool ok" in out.stdout, (out.returncode, out.stderr)
