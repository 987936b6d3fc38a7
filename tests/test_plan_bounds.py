"""The words that the device's matching reads for the terms of compiled plans lie inside a wave's region and the image
(plan_bounds.cpp, built with the task compiler's own source; no GPU needed)."""

import os
import subprocess

import pytest

from mymyr_amd import gen

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "mymyr_amd", "csrc")


def short_last_row(objects: int, marked: int) -> str:
    """A fluent of few objects whose row is the state's last, tested (negated) for a parameter of all objects: the
    parameter's window is far longer than the row."""
    lines = [f"O {objects}", "P 3", "S 1 item", "F 1 other", "F 1 mark", f"SI {marked}", *(f"0 {o}" for o in range(marked)),
             "FI 1", "1 0", "G 1", "1 1 5", "A 2", "mark 1", "L 1", "0 1 0", "E 1", "0", "L 0", "F 1", "2 1 0",
             "act 1", "L 1", "2 0 0", "E 1", "0", "L 0", "F 1", "1 1 0"]
    return "\n".join(lines) + "\n"


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plans") / "plan_bounds")
    subprocess.run(["g++", "-O1", "-std=c++20", "-I", CSRC, os.path.join(HERE, "plan_bounds.cpp"), "-o", exe], check=True)
    return exe


def test_plans_read_inside_the_region(checker, golden, tmp_path):
    files = []
    for k, (objects, marked) in enumerate([(6000, 10), (130, 10), (200, 70), (64, 64), (65, 1)]):
        files.append(tmp_path / f"short_{k}.txt")
        files[-1].write_text(short_last_row(objects, marked))
    files.append(tmp_path / "transport.txt")
    files[-1].write_text(gen.transport(24, 6, 40, goals=6, seed=0))
    tasks = os.path.dirname(golden.task_path("strips"))
    # (the organic synthesis task takes minutes to compile; its schemas have more literals of the same forms)
    files += [os.path.join(tasks, f) for f in sorted(os.listdir(tasks)) if not f.startswith("organic")]
    r = subprocess.run([checker, *map(str, files)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, "\n".join(x for x in r.stdout.splitlines() if not x.endswith("reads"))
