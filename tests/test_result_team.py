"""The threads that help with a job's results, on the CPU: copies are whole whatever
number of threads can be had, and no failure to get one ends the process."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("team") / "team_test")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-pthread", "-Wl,--wrap=pthread_create", "-static-libstdc++",
                    "-o", path, os.path.join(HERE, "team", "team_test.cpp")], check=True)
    return path


@pytest.mark.parametrize("what", ["thread", "memory"])
@pytest.mark.parametrize("succeed", [0, 1, 2, 3, 4, 5, 6, 7, 9, 12, 15, 1000])
def test_copies_with_few_threads(program, what, succeed):
    r = subprocess.run([program, what, str(succeed)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "done\n", (r.returncode, r.stdout, r.stderr)
