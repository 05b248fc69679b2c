"""Host copies cut between threads, also where a thread cannot be started (tests/native/ranges_host.cpp)."""

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_element_once_when_threads_fail(tmp_path):
    program = str(tmp_path / "ranges")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-o", program, os.path.join(HERE, "native", "ranges_host.cpp")],
                   check=True)
    subprocess.run([program], check=True, timeout=60)
