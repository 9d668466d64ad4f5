"""Host side of the C API (buffers, their growth and what happens when memory
runs out) on a stand-in for the HIP runtime: pw_capi.hip and pw_ff.hip built
with the host compiler against tests/cpp/host_logic.cpp, whose launchers check
the buffers they are given."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="session")
def host_logic(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host_logic") / "host_logic")
    csrc = os.path.join(ROOT, "pawan_amd", "csrc")
    # tree and network kernels are not reached here: their launchers stay unresolved
    subprocess.run(
        ["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-D__device__=",
         "-D__align__(x)=__attribute__((aligned(x)))", "-DHIP_SYMBOL(x)=(&x)", "-I", os.path.join(ROCM, "include"),
         "-I", os.path.join(ROOT, "include"), "-I", csrc, "-x", "c++", os.path.join(csrc, "pw_capi.hip"),
         os.path.join(csrc, "pw_ff.hip"), os.path.join(ROOT, "tests", "cpp", "host_logic.cpp"),
         "-Wl,--unresolved-symbols=ignore-all", "-o", exe], check=True)
    return exe


def _run(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120)
    print(r.stdout + r.stderr, flush=True)
    assert r.returncode == 0, r.stdout


def test_partial_buffer_that_does_not_fit(host_logic):
    """A precision whose partial-sum rows do not fit runs in one part or
    reports it; the other precisions' launches still get rows of their own."""
    _run(host_logic, "partial_buffer")


def test_diagnostics_of_wake_blocks_stay_bounded(host_logic):
    """However large two wakes are, their block is a bounded number of items
    that cover it, and its sums come from all of them."""
    _run(host_logic, "diagnose_items")


def test_transfers_with_little_pinned_memory(host_logic):
    """States, rates and training samples pass where the staging of their
    whole size cannot be pinned."""
    _run(host_logic, "little_pinned_memory")


def test_pair_timing_holds_the_sum_of_partial_rates(host_logic):
    _run(host_logic, "timed_launches")


def test_items_name_their_chunks(host_logic):
    """Coupled and independent wakes, the default launch and source parts."""
    _run(host_logic, "item_chunks")


def test_state_vectors_of_many_wakes_in_one_launch(host_logic):
    """pw_set_states, pw_get_states and pw_get_rates of 500 wakes, empty ones
    and unused rows among them."""
    _run(host_logic, "state_vectors")
