"""The logic of the device-to-host copies (nlm_copy.hip) on a CPU: the file is compiled with g++
over a small runtime whose device memory is host memory (fake_hip/), and each scenario of
copy_host_driver.cpp is run in a process of its own."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = [pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available"),
              pytest.mark.skipif(len(os.sched_getaffinity(0)) < 3, reason="helpers need three CPUs")]


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("copies") / "driver")
    r = subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-I" + os.path.join(HERE, "fake_hip"),
                        "-I" + os.path.join(HERE, "..", "include"), os.path.join(HERE, "copy_host_driver.cpp"),
                        "-o", exe, "-lpthread", "-ldl"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout
    return exe


def run(driver, scenario):
    r = subprocess.run([driver, scenario], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_every_size_arrives(driver):
    run(driver, "sizes")


def test_helpers_that_start_late(driver):
    """A helper thread that cannot be started is started by a later copy, the others not again."""
    run(driver, "helpers")


def test_no_pinned_memory(driver):
    """Where no staging area can be allocated the copies are the runtime's own, with no error left."""
    run(driver, "no area")


def test_stream_of_another_device(driver):
    """A plan's results while another device is the current one, which stays so."""
    run(driver, "device")


def test_results_in_pinned_memory(driver):
    """A caller's pinned memory is filled by one copy of the runtime's each, not by way of the area."""
    run(driver, "pinned")


def test_second_caller_takes_the_plain_copy(driver):
    """While one caller's copy goes by way of the area, another's is the runtime's."""
    run(driver, "two callers")


def test_one_cpu(driver):
    """A process on one CPU starts no helpers, its copies are the runtime's."""
    run(driver, "one cpu")
