"""Which tasks the scheduler takes as independent of each other (csrc/hpx_task_ranges.h): those that share no byte of any
buffer they name, views at different addresses into one tensor included.  The header has no GPU dependency; the test
compiles tests/host_task_ranges.cpp with the host compiler and runs it."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tasks_share_memory_by_address_range(tmp_path):
    exe = str(tmp_path / "host_task_ranges")
    src = os.path.join(ROOT, "tests", "host_task_ranges.cpp")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-fsanitize=address,undefined",
                           "-I" + os.path.join(ROOT, "torch-hipress-extension_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                           src, "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "OK", (r.stdout, r.stderr)
