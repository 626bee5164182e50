"""The library's host paths on a stand-in for the HIP runtime (cpp/host_paths.cpp):
device memory is host memory, kernels are counted and not run.  What happens
when an allocation fails, when a result does not arrive and on which stream a
copy goes can be checked there without a GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host_paths(tmp_path_factory):
    import stratiflow_amd as sf
    if not os.path.exists(sf.LIB_PATH):
        pytest.skip("libsfhip.so not built")
    exe = str(tmp_path_factory.mktemp("host_paths") / "host_paths")
    lib = os.path.dirname(sf.LIB_PATH)
    subprocess.check_call(["g++", "-std=c++14", "-O1", "-Wall", "-rdynamic", "-I" + os.path.join(ROOT, "include"), "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", "host_paths.cpp"), "-L" + lib, "-lsfhip",
                           "-Wl,-rpath," + lib, "-Wl,--allow-shlib-undefined"])
    return exe


@pytest.mark.parametrize("scenario", ["adjoint_memory", "inner_product_results", "batch_memory", "net_stream",
                                      "net_memory", "table_copies"])
def test_host_path(host_paths, scenario):
    r = subprocess.run([host_paths, scenario], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout[-3000:]
