"""What the library does on the host around its kernels, on a HIP runtime in
host memory (cxx/fake_hip.cpp) that a small C++ program brings along: failing
allocations, routes and launch shapes. CPU only, no kernel runs."""
import os
import subprocess

import pytest

from nopt_amd import _lib as L

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_runtime")

    def go(name, *args):
        exe = str(out / name)
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-rdynamic", os.path.join(HERE, "cxx", name + ".cpp"),
                               os.path.join(HERE, "cxx", "fake_hip.cpp"), L.LIB_PATH,
                               "-Wl,-rpath," + os.path.dirname(L.LIB_PATH), "-Wl,--allow-shlib-undefined", "-o", exe])
        r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=100)
        print(r.stdout[-3000:], r.stderr[-2000:])
        assert r.returncode == 0 and r.stdout.endswith("ok\n")
    return go


def test_failed_allocation_and_retry(run):
    run("host_alloc_retry")


def test_device_bytes_are_those_held(run):
    run("host_device_bytes")


def test_autotuner_leaves_unused_settings(run):
    run("host_autotune")


def test_stored_exchange_splits_are_those_launched(run):
    run("host_exchange_splits")


def test_matrix_product_over_no_terms_is_refused(run):
    run("host_gemm_empty")


def test_pinned_memory_is_kept(run):
    run("host_pinned")
