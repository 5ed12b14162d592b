"""The library's host code on a stand-in for the HIP runtime (hip_stub.cpp):
failed allocations, what a call allocates, the order of calls.  No GPU; each
scenario of stub_cases.py runs in a process of its own."""
import os
import subprocess
import sys

import pytest

from magic_amd import sht
from stub_cases import FP64, SPLIT16, SPLIT16_REC

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def scenario(tmp_path_factory):
    if not os.path.exists(sht.LIB_PATH):
        pytest.skip("libmhx.so not built")
    stub = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I", ROCM + "/include",
                           "-o", stub, os.path.join(HERE, "hip_stub.cpp")])

    def run(*args):
        r = subprocess.run([sys.executable, os.path.join(HERE, "stub_cases.py"), stub, sht.LIB_PATH, *map(str, args)],
                           capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-2000:]
    return run


@pytest.mark.parametrize("precision,name", [
    (FP64, "axi_to_spat"), (FP64, "toraxi_to_spat"), (FP64, "tables"), (SPLIT16, "scal_to_spat"),
    (SPLIT16_REC, "scal_to_spat"), (SPLIT16_REC, "axi_to_spat"), (SPLIT16_REC, "toraxi_to_spat"), (SPLIT16_REC, "tables")])
def test_tables_of_a_failed_first_call_are_built_by_the_next(scenario, precision, name):
    """A plan whose tables could not be built by a first call builds them in
    the next: no kernel reads a missing or an unfilled one."""
    scenario("failed_first_call", precision, name)


@pytest.mark.parametrize("precision", [FP64, SPLIT16])
def test_calls_after_plan_creation_build_no_tables(scenario, precision):
    """Plans that store tables have all of them from their creation on: no first
    call allocates, launches a table kernel or waits for the device."""
    scenario("tables_at_creation", precision)


def test_split_plan_holds_no_tables_it_does_not_read(scenario):
    scenario("analysis_pair_given_up")


def test_lds_sizes_are_set_on_every_device(scenario):
    scenario("lds_per_device")


@pytest.mark.parametrize("precision", [FP64, SPLIT16, SPLIT16_REC])
def test_captured_step_is_destroyed_before_what_it_uses(scenario, precision):
    scenario("graph_destroyed_first", precision)


@pytest.mark.parametrize("precision", [FP64, SPLIT16, SPLIT16_REC])
def test_step_after_a_failed_growth_of_the_workspaces(scenario, precision):
    scenario("failed_growth", precision)


def test_radial_loop_after_a_failed_first_call(scenario):
    scenario("failed_rloop")
