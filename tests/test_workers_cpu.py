"""The worker threads of the concurrent solves where the system refuses to
start some: the solves go on with those that run (no exception leaves a C
entry, no thread is left to end the process)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_workers_that_cannot_be_started_are_done_without(tmp_path):
    exe = str(tmp_path / "worker_limit")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread",
                    "-I" + os.path.join(ROOT, "primal-dual-toolbox_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "worker_limit.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, (run.returncode, run.stdout, run.stderr)
