"""The threads that move large fields to the host are the process's, not a
context's (lulesh_copypool.h): a few whatever the number of contexts, given
back with the last of them, and free of data races."""
import os
import subprocess
import time

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_pool_under_the_thread_sanitizer(tmp_path):
    exe = tmp_path / "pool_check"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-fsanitize=thread", "-Wall", "-Wextra",
                    "-I", os.path.join(os.path.dirname(HERE), "lulesh.jl_amd", "csrc"),
                    os.path.join(HERE, "host", "pool_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "failures 0" in r.stdout, r.stdout + r.stderr[-3000:]


@pytest.mark.gpu
def test_contexts_share_the_threads():
    from lulesh_amd import Domain, LuleshProblem
    print("[copy pool] five contexts", flush=True)

    def threads():
        return len(os.listdir("/proc/self/task"))

    held, counts = [], []
    for _ in range(5):
        d = Domain(LuleshProblem(10, True, 60, 1, 1, 1))
        d.get("e")  # 1.7 MB
        held.append(d)
        counts.append(threads())
    assert counts[-1] - counts[0] < 7, counts
    for d in held:
        d.close()
    for _ in range(100):  # a joined thread's entry may outlive the join for a moment
        if threads() < counts[-1]:
            break
        time.sleep(0.01)
    assert threads() < counts[-1], (threads(), counts)
