"""The multigrid kernels on the CPU, for what depends on the order in which waves run or on values that a scene meets
rarely (tests/cpp/cpu_kernels/multigrid_check.cpp)."""

import subprocess

import pytest

from tests import cpu_kernels


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = cpu_kernels.build("multigrid_check", ["k_sort", "k_multigrid"], str(tmp_path_factory.mktemp("mg")))

    def run(name):
        r = subprocess.run([exe, name], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_a_solve_that_ends_during_a_launch_leaves_no_partial_sums(check):
    check("late_end")


def test_a_right_hand_side_that_is_not_a_number_is_not_solved(check):
    check("not_a_number")


def test_regions_without_air_converge(check):
    check("pockets")


def test_a_solve_does_not_depend_on_the_one_before(check):
    check("history")
