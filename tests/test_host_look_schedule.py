"""When the host looks at a queued solve (csrc/look_schedule.hpp), compiled alone
with g++: whatever the handle solved before, a solve of c iterations launches at
most max(128, 2 c) + 16 of them, and one like the last needs two looks or three."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "soft-body-simulation-cuda_amd", "csrc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("ls") / "look_schedule_driver")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", CSRC, os.path.join(HERE, "host", "look_schedule_driver.cpp"),
                    "-o", exe], check=True)

    def run(solves):
        text = "\n".join(" ".join(map(str, s)) for s in solves)
        p = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
        return np.array([list(map(int, l.split())) for l in p.stdout.split("\n") if l])
    return run


def test_surplus_is_bounded_whatever_came_before(driver):
    rng = np.random.default_rng(0)
    its = np.exp(rng.uniform(0, np.log(20000), 400)).astype(int)
    same = driver([(1000, 5000, 0, c, 20000) for c in its])
    assert np.all(same[:, 0] <= np.maximum(128, 2 * its) + 16)
    assert np.all(same[:, 0] > np.minimum(its, 19999))
    # another size, another start, or a solve cut by its limit: nothing is learned from it
    for before in ((1001, 5000, 0, 3000, 20000), (1000, 5001, 0, 3000, 20000), (1000, 5000, 1, 3000, 20000),
                   (1000, 5000, 0, 30000, 20000)):
        assert driver([before, (1000, 5000, 0, 12, 20000)])[1, 0] == 16


@pytest.mark.parametrize("its", [1, 15, 16, 40, 100, 128, 152, 250])
def test_a_repeated_solve_needs_few_looks(driver, its):
    launched, looks = driver([(1000, 5000, 0, its, 20000)] * 2)[1]
    assert looks <= (2 if its <= 152 else 3) and launched <= its + max(16, its // 4) + 1


@pytest.mark.parametrize("limit", [0, 1, 16, 17, 300])
def test_limit(driver, limit):
    assert np.all(driver([(1, 1, 0, 1000, limit)] * 3)[:, 0] == limit)
