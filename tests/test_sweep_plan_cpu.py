"""The choice of two or many steps per launch, its tiles and its chunk heights
(csrc/sweep_plan.cpp), without a GPU: the driver checks every work list against
the kernel's limits; here, which lattices get one."""
import os
import random
import shutil
import subprocess

import pytest

import nflow

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CAV, CH = nflow.CAVITY, nflow.CHANNEL


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = str(tmp_path_factory.mktemp("plan") / "driver")
    csrc = os.path.join(ROOT, "nflow-red-poplar_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "include"), "-I", csrc,
                    os.path.join(ROOT, "tests", "sweep_plan_driver.cpp"), os.path.join(csrc, "sweep_plan.cpp"),
                    "-o", exe], check=True)

    def run(lats, temporal=-1, cus=256):
        r = subprocess.run([exe, str(cus), str(temporal)] + [str(v) for s in lats for v in s], capture_output=True,
                           text=True, timeout=60)
        assert r.returncode == 0, (lats, temporal, r.stderr)
        if r.stdout.startswith("small"):
            return int(r.stdout.split()[1])
        return None if r.stdout == "none\n" else [tuple(map(int, w.split())) for w in r.stdout.splitlines()]

    return run


LARGE = [(576, 576, 576, CAV), (600, 600, 600, CAV), (640, 640, 640, CAV), (768, 768, 768, CAV),
         (1024, 1024, 1024, CAV), (1200, 1200, 1200, CAV), (512, 1600, 512, CAV), (984, 52, 1039, CAV),
         (1024, 512, 512, CH), (2048, 256, 256, CH), (2048, 512, 512, CH), (4096, 256, 256, CH), (2000, 20, 2500, CAV)]


@pytest.mark.parametrize("shape", LARGE)
def test_large_planes_take_chunks_that_a_window_holds(plan, shape):
    """The tiles of one plane are as many as the CUs: chunks for up to five
    rounds of the CUs are taller than 32-bit offsets reach."""
    (_, _, h, _), = plan([shape])
    most = (2 ** 30 - 2331) // 19 // (shape[0] * shape[2]) - 4
    assert 1 <= h <= most
    assert h == shape[1] or h > most // 2
    # in a batch too, and beside a lattice that fits as it is
    assert plan([shape, shape]) and plan([(128, 128, 128, CAV), shape])
    # a height that does not fit stays refused
    assert plan([shape], temporal=most) and plan([shape], temporal=most + 1) is None


def test_windows_that_end_at_32_bits(plan):
    """Heights whose h + 4 planes come within 59 nodes of what 32-bit byte
    offsets reach: the first plane starts up to 63 nodes into its block, and
    the last node's run 18 lies up to 1,152 elements on."""
    for nx, nz, h in ((1429, 557, 67), (557, 1429, 67), (1847, 1457, 17), (1457, 1847, 17), (2718, 2599, 4)):
        for below in (0, 1):
            plan([(nx, 5 * h + 3, nz, CAV)], temporal=h - below)
        plan([(nx, 5 * h + 3, nz, CAV)])


def test_any_box_within_the_kernel_limits(plan):
    rng = random.Random(1)
    for k in range(150):
        d = [int(2 ** rng.uniform(0, 10.5)) for _ in range(3)]
        lat = (*d, CH if rng.random() < 0.5 and d[0] > 2 else CAV)
        h = int(2 ** rng.uniform(0, 12))
        if d[0] * d[1] * d[2] < 2e9:
            plan([lat])
            plan([lat], temporal=h)
            plan([lat, (90, 80, 70, CAV)])


def test_not_where_it_does_not_apply(plan):
    big = (256, 256, 256, CAV)
    assert plan([big]) and plan([big], temporal=24)[0][2] == 24
    assert plan([big], temporal=0) is None
    assert plan([(256, 256, 256, nflow.PIPE)]) is None and plan([big, (256, 256, 256, nflow.PIPE)]) is None
    assert plan([big, big], temporal=16) is None  # a height is a choice for one lattice
    assert plan([(48, 48, 48, CAV)]) is None
    assert plan([(3700, 8, 3700, CAV)]) is None  # not a plane fits a window


# us per step of one and of two steps per launch, measured on 256 CUs with the
# tiles and heights that the plan picks
MEASURED = [
    ((274, 28, 24, CH), 8.1, 11.2), ((322, 47, 19, CH), 10.7, 14.9), ((142, 12, 110, CH), 7.8, 10.6),
    ((56, 52, 62, CH), 7.7, 9.7), ((30, 36, 245, CH), 11.5, 13.5), ((211, 5, 181, CH), 7.4, 10.4),
    ((170, 4, 248, CAV), 7.4, 8.6), ((306, 13, 44, CAV), 8.0, 9.6), ((59, 13, 217, CAV), 6.6, 7.9),
    ((194, 27, 32, CAV), 6.4, 8.3), ((64, 64, 64, CAV), 7.0, 7.8), ((128, 64, 32, CAV), 7.0, 7.8),
    ((61, 15, 213, CAV), 6.9, 8.1), ((64, 64, 64, CH), 8.8, 9.8), ((72, 72, 72, CAV), 12.3, 10.1),
    ((60, 60, 60, CAV), 8.9, 7.9), ((76, 76, 76, CH), 15.6, 14.0),
    ((96, 96, 96, CAV), 25.6, 16.6), ((101, 67, 83, CAV), 17.9, 13.6), ((128, 128, 128, CAV), 53.5, 33.8),
    ((66, 62, 233, CH), 30.1, 22.7), ((44, 98, 246, CH), 34.2, 24.9), ((512, 128, 128, CH), 215.0, 125.4),
    ((30, 150, 104, CAV), 16.6, 12.4), ((179, 32, 154, CAV), 26.4, 18.1), ((28, 323, 96, CH), 27.8, 17.1),
]


@pytest.mark.parametrize("lat,one,two", MEASURED)
def test_two_steps_per_launch_only_where_they_are_faster(plan, lat, one, two):
    assert (plan([lat]) is not None) == (two < one)


def test_batches_take_two_steps_only_where_they_are_faster(plan):
    assert plan([(35, 35, 35, CH)] * 57) is None  # 78.6 us a step, 105.5 in pairs
    assert plan([(47, 47, 47, CH)] * 26) is None  # 79.8 and 88.8
    assert plan([(48, 48, 48, CAV)] * 16)  # 51.7 and 39.4
    assert plan([(77, 77, 77, CH)] * 6)  # 0.82 of one step's time


def test_lattices_in_lds_only_where_they_are_faster(plan):
    small = (10, 10, 10, CAV)
    assert plan([small]) == 1000 and plan([small], temporal=0) is None
    assert plan([(1920, 1, 1, CAV)]) == 1920 and plan([(1921, 1, 1, CAV)]) is None
    assert plan([small, (12, 12, 12, CAV)]) == 1728
    assert plan([small, (10, 10, 10, CH)]) is None and plan([small, (16, 16, 16, CAV)]) is None
    # us per step of one step per launch / k_small
    assert plan([(4, 4, 4, CAV)] * 1024) == 64  # 3.8 / 3.7
    assert plan([(4, 4, 4, CAV)] * 4096) is None  # 9.4 / 14.7
    assert plan([(3, 3, 3, CAV)] * 2048) is None  # 5.0 / 8.2
    assert plan([(5, 5, 5, CAV)] * 4096) == 125  # 19.3 / 15.8
    assert plan([(8, 8, 8, CAV)] * 4096) == 512  # 59 / 20
