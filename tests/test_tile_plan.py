"""What the plan of the prompt-row products (csrc/tile_plan.h) can return, and
sizes that reach all of it: test_gpu_tiles.py runs SIZES on the GPU."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

# (gated, m, n, k): every tile shape, gated and with a residual, whole with one
# step of k and with many, and split; the last row and column tiles are ragged
# and k's pieces uneven.
SIZES = [
    (0, 65, 204, 64), (0, 65, 204, 832), (1, 65, 68, 64), (1, 65, 68, 832),
    (0, 2694, 660, 64), (0, 321, 280, 1984), (1, 1602, 584, 64), (1, 839, 68, 1344),
    (0, 129, 12_364, 64), (0, 839, 888, 2944), (1, 643, 2028, 64), (1, 769, 584, 2624),
    (0, 2694, 1420, 64), (0, 580, 3244, 3904), (1, 3268, 584, 64), (1, 1476, 660, 3904),
    (0, 391, 12_364, 64), (0, 1154, 1192, 5824), (1, 2946, 964, 64), (1, 1154, 584, 5824),
    (0, 257, 16_392, 64), (0, 1217, 1572, 4864), (1, 257, 8260, 64), (1, 1602, 584, 5824),
    (0, 65, 204, 576), (1, 65, 68, 576), (0, 1350, 1420, 576), (1, 1602, 584, 576),
    (0, 1154, 2408, 576), (1, 1665, 888, 576), (0, 1665, 2332, 576), (1, 2050, 964, 576),
    (0, 2435, 2332, 576), (1, 2946, 964, 576), (0, 1539, 4612, 576), (1, 2050, 1800, 576),
]


@pytest.fixture(scope="module")
def printer(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ is not available")
    out = str(tmp_path_factory.mktemp("plan") / "print_plan")
    subprocess.run([cxx, "-std=c++17", "-O2", os.path.join(HERE, "tile_plan", "print_plan.cpp"), "-o",
                    out], check=True, capture_output=True, text=True)
    return out


def numbers(text):
    return [tuple(map(int, line.split())) for line in text.split("\n") if line]


def test_the_sizes_reach_every_plan(printer):
    run = lambda *a, **k: subprocess.run([printer, *a], check=True, capture_output=True, text=True,
                                         timeout=300, **k).stdout
    reachable = set(numbers(run("all")))
    plans = numbers(run(input="".join(f"{m} {n} {k} {g}\n" for g, m, n, k in SIZES)))
    reached = set()
    for (gated, m, n, k), (shape, rows, cols, splits) in zip(SIZES, plans, strict=False):
        assert m % rows and n % cols and m > rows and n > cols, (m, n, k)
        assert splits == 1 or (k // 64) % splits, (m, n, k)
        reached.add((shape, gated, int(splits > 1), k > 64))
    assert {r[:3] for r in reached} == reachable
    # whole products of one step and of many
    assert {r[:2] for r in reached if not r[2] and r[3]} == {r[:2] for r in reachable}
    assert {r[:2] for r in reached if not r[2] and not r[3]} == {r[:2] for r in reachable}
