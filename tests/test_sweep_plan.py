"""The sweeps' layouts and plans (csrc/cd_plan.h), checked over many sizes by a
host program (tests/plan/plan_check.cpp) that this test compiles."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "poisson_caustic_design_amd", "csrc")


@pytest.fixture(scope="module")
def plan_check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "plan_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + CSRC, "-Wno-unused-function",
                    os.path.join(ROOT, "tests", "plan", "plan_check.cpp"), "-o", exe], check=True)

    def run(name):
        r = subprocess.run([exe, name], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout
    return run


def test_region_rows_lie_in_the_plane(plan_check):
    plan_check("rows_in_plane")


def test_tracking_words_fit_on_every_shape(plan_check):
    plan_check("tracking_room")


def test_launches_are_bounded(plan_check):
    plan_check("launch_length")


def test_tracking_launches_do_not_write_what_they_read(plan_check):
    plan_check("track_words")


def test_the_early_launch_is_one_launch(plan_check):
    plan_check("early_launch")
