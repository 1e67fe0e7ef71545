"""Runs tests/cpp/test_quant_kernel.bin: the reference crate's own unit tests replayed
through the C++ mirror of its interface (include/oxq/quant_kernel.hpp -> C ABI), and the
host tests beside it: the kernels' LDS limits asked for by several threads, the order
in which work groups take tiles, where weight requests ahead of the end reach, and the library's scratch on a full device."""
import os
import subprocess

import pytest

CPP = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp")
BIN = os.path.join(CPP, "test_quant_kernel.bin")


def _run(*args, binary=BIN):
    if not os.path.exists(binary):
        pytest.fail(f"{binary} is not built: run `python -m oxillama_amd.build`")
    p = subprocess.run([binary, *args], capture_output=True, text=True, timeout=120)
    print(p.stdout)
    print(p.stderr)
    assert p.returncode == 0, p.stdout[-4000:]
    assert "0 failed" in p.stdout.split("\n")[-2]


def test_lds_limits_are_only_raised():
    _run(binary=os.path.join(CPP, "test_lds_opt_in.bin"))


def test_tiles_are_dealt_evenly_to_the_xcds():
    _run(binary=os.path.join(CPP, "test_tile_order.bin"))


def test_requests_ahead_of_the_end_stay_in_the_matrix():
    _run(binary=os.path.join(CPP, "test_direct_window.bin"))


def test_scratch_falls_back_to_what_a_call_needs():
    _run(binary=os.path.join(CPP, "test_scratch.bin"))


def test_cpp_mirror_host_cases():
    _run("--host")


@pytest.mark.gpu
def test_cpp_mirror_gpu_cases():
    _run("--gpu")
