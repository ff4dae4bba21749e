"""The engine's host side on the CPU, over a stand-in for the HIP runtime
(tests/hip_stub_driver.cpp): what refused calls touch, and what is held and
refused when device memory runs out."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "bfs-gpu-sycl_amd")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    out = tmp_path_factory.mktemp("stub") / "hip_stub_driver"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-rdynamic",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"),
                    "-isystem", os.path.join(ROCM, "include"),
                    os.path.join(ROOT, "tests", "hip_stub_driver.cpp"), "-o", str(out), "-L", PKG,
                    "-lbfsx", f"-Wl,-rpath,{PKG}", f"-Wl,-rpath-link,{os.path.join(ROCM, 'lib')}"],
                   check=True)
    return str(out)


def check(driver, what):
    p = subprocess.run([driver, what], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr)


def test_wrong_nnz_is_refused_before_row_idx_is_read(driver):
    check(driver, "wrong_nnz")


def test_replaced_arrays_leave_before_the_search_state_comes(driver):
    check(driver, "replace")


def test_no_graph_after_a_failure_to_allocate_its_search_state(driver):
    check(driver, "state_oom")


def test_nothing_of_a_bottom_up_copy_stays_after_a_failure(driver):
    check(driver, "order_oom")


def test_shared_tiles_fit_a_launch(driver):
    check(driver, "launch_size")


def test_upload_without_room_for_both_graphs(driver):
    check(driver, "no_room")


def test_temporaries_are_given_back_where_memory_ends(driver):
    check(driver, "leaks")
