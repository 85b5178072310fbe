"""How blocking calls end: a program that stands in for the HIP runtime looks at what the library asks of it
(tests/host/blocking_calls_test.cc). Needs no GPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    lib_dir = os.path.join(ROOT, "kraken_amd")
    if not os.path.exists(os.path.join(lib_dir, "libkraken_hip.so")):
        from kraken_amd import build
        build.build(verbose=False)
    exe = str(tmp_path_factory.mktemp("host") / "blocking_calls_test")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-I" + os.path.join(ROOT, "include"),
                           "-isystem", os.path.join(ROCM, "include"),
                           os.path.join(ROOT, "tests", "host", "blocking_calls_test.cc"), "-o", exe, "-L" + lib_dir,
                           "-lkraken_hip", "-Wl,-rpath," + lib_dir, "-Wl,-rpath," + os.path.join(ROCM, "lib")])
    return exe


# dense, sparse: a blocking call on pageable arrays synchronises after the copies that staged them
# words: no two calls wait on one word, and the calls that find none synchronise
# core: a waiting thread lets the other threads of its core run
# host_gradients: sparse gradients in host memory of small dense tables are read once
# gradients_order: which of them go tile by tile
# first_gradient: a table's first one in pageable memory takes few commands
# decodes: which of them leave bits of the elements, and what one keeps on the device is bounded
# old_words: a launch of a call that failed says something over the next call's word
@pytest.mark.parametrize("which", ["dense", "sparse", "words", "core", "host_gradients", "gradients_order",
                                   "first_gradient", "decodes", "old_words"])
def test_blocking_calls(program, which):
    r = subprocess.run([program, which], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout == which + " ok\n"
