"""The shapes of the surrogate's convolution kernels (csrc/lbmib_conv_plan.h),
walked on the host by tests/conv_plan_check.cpp."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "conv_plan_check")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-o", exe,
                           os.path.join(REPO, "tests", "conv_plan_check.cpp")])

    def run(what):
        r = subprocess.run([exe, what], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_every_voxel_of_a_tile_has_one_position(check):
    check("tiles")


def test_every_piece_of_a_weight_gradient_unit_is_the_one_its_readers_expect(check):
    check("pieces")


def test_every_launch_has_fewer_threads_than_the_runtime_takes(check):
    check("grids")


def test_z_ranges_are_the_best_and_quickly_found(check):
    check("ranges")


def test_layers_take_the_form_that_suits_them(check):
    check("forms")


def test_the_gradient_of_a_view_is_the_volumes(check):
    check("views")
