"""The library's host sources (planning, allocation, copies, the server) compiled
for the CPU with g++ against a HIP runtime on host memory
(tests/cpp/fake_hip.cpp), to drive what a device cannot be driven into: exhausted
memory, failed allocations. Kernels do nothing there."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "bnmf-algs_amd", "csrc")
CPP = os.path.join(ROOT, "tests", "cpp")
FLAGS = ["-std=c++17", "-O1", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
         "-fsanitize=address,undefined"]
SOURCES = ["bld_batch", "live", "hostcopy", "bld_appr_host", "tune", "sampler", "serving", "capi"]


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    out = tmp_path_factory.mktemp("host")
    files = [os.path.join(SRC, s + ".cpp") for s in SOURCES] + [os.path.join(CPP, "fake_hip.cpp")]
    jobs = [subprocess.Popen(["g++", *FLAGS, "-c", f, "-o", str(out / (os.path.basename(f) + ".o"))]) for f in files]
    assert all(j.wait() == 0 for j in jobs)
    return [str(out / (os.path.basename(f) + ".o")) for f in files]


def _run(objects, tmp_path, name, *args):
    exe = str(tmp_path / name)
    subprocess.run(["g++", *FLAGS, os.path.join(CPP, name + ".cpp"), *objects, "-o", exe, "-lpthread", "-ldl"], check=True)
    env = {**os.environ, "ASAN_OPTIONS": "verify_asan_link_order=0"}
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert " ok" in r.stdout


def test_batches_at_the_limit_of_memory(objects, tmp_path):
    _run(objects, tmp_path, "test_batch_memory")


def test_results_where_host_memory_runs_out(objects, tmp_path):
    _run(objects, tmp_path, "test_host_copy_alloc")


def test_results_to_host_memory(objects, tmp_path):
    _run(objects, tmp_path, "test_host_copy")


def test_calls_of_few_iterations(objects, tmp_path):
    _run(objects, tmp_path, "test_few_iterations")


def test_share_from_a_sample(objects, tmp_path):
    _run(objects, tmp_path, "test_worth")


@pytest.mark.parametrize("what", ["few", "full", "later", "small", "streams"])
def test_server_memory(objects, tmp_path, what):
    _run(objects, tmp_path, "test_server_memory", what)


@pytest.mark.parametrize("what", ["length", "route"])
def test_tiny_batches(objects, tmp_path, what):
    _run(objects, tmp_path, "test_tiny_batches", what)
