"""The library's host code on a HIP runtime without a GPU (tests/fake): which
kernels the calls launch, on which devices, and what happens when an allocation
is refused."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
FAKE = os.path.join(HERE, "fake")
ROCM = os.environ.get("ROCM", "/opt/rocm")


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-o", out, os.path.join(FAKE, "fake_hip.cpp")], check=True)
    return out


def _run(fake, scenario):
    r = subprocess.run([sys.executable, os.path.join(FAKE, "scenarios.py"), fake, scenario], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr


def test_held_grid_pointer(fake):
    _run(fake, "held_grid_pointer")


def test_calls_on_a_plan_of_another_device(fake):
    _run(fake, "other_device")


def test_refused_memory_of_the_faster_paths(fake):
    _run(fake, "refused_memory")


def test_more_chunks_than_a_launch_has_threads(fake):
    _run(fake, "many_short_subgrids")


def test_deconvolver_beside_other_kernels(fake):
    _run(fake, "crowded_descent")


def test_layer_sum_without_line_transform(fake):
    _run(fake, "layer_sum_without_line_transform")


def test_direct_launches_of_a_resampled_plan(fake):
    _run(fake, "direct_launches_of_a_resampled_plan")


def test_preparation_is_left_to_the_calls_that_need_it(fake):
    _run(fake, "preparation")


def test_short_direct_launches(fake):
    _run(fake, "short_direct_launches")
