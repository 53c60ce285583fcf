"""What the library does on the host when something fails or several callers meet, without a device: a check program
defines the HIP runtime's functions itself (tests/cpp/host)."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOST = os.path.join(ROOT, "tests", "cpp", "host")
LIB = os.path.join(ROOT, "flipengine3d_amd")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "host_check")
    if not os.path.exists(os.path.join(LIB, "libflipmi.so")):
        import flipengine3d_amd.build
        flipengine3d_amd.build.build()
    # The HIP runtime itself is the library's to load, and hidden by these definitions.
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-w", "-rdynamic", "-pthread", "-I",
                    "/opt/rocm/include", os.path.join(HOST, "host_check.cpp"), os.path.join(HOST, "fake_hip.cpp"), "-o",
                    exe, "-L", LIB, "-lflipmi", "-Wl,-rpath," + LIB, "-Wl,--allow-shlib-undefined"], check=True)

    def run(name):
        r = subprocess.run([exe, name], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_a_fallback_without_room_is_an_error_each_time(check):
    check("no_room_to_fall_back")


def test_multigrid_is_tried_again_after_a_fallback(check):
    check("multigrid_again")


def test_idle_pool_memory_is_there_for_others(check):
    check("pool_gives_way")


def test_results_come_without_pinned_memory(check):
    check("no_pinned_memory")


def test_a_buffer_is_given_back_without_host_memory(check):
    check("give_back_without_host_memory")


def test_calls_of_two_contexts_do_not_wait_for_each_other(check):
    check("calls_do_not_wait_for_each_other")


def test_results_are_read_while_another_device_is_current(check):
    check("another_device_is_current")


def test_few_batch_sizes_are_captured(check):
    check("few_graphs")
