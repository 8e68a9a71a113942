"""The prefill kernel's host-side launch rules (eredu_amd/csrc/qmm_plan.hpp),
compiled for the CPU."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "eredu_amd", "csrc")
DRIVER = r"""
#include "qmm_plan.hpp"
extern "C" int param_words(int gs, int K, int cps, uint64_t s, uint64_t b) {
    return eq::qmm_param_words(gs, K, cps, reinterpret_cast<const void*>(s), reinterpret_cast<const void*>(b));
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("qmm_plan")
    src, lib = d / "driver.cpp", d / "driver.so"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", "-o", lib, src],
                   check=True, timeout=120)
    lib = ctypes.CDLL(str(lib))
    lib.param_words.argtypes = [ctypes.c_int] * 3 + [ctypes.c_uint64] * 2
    return lib


@pytest.mark.parametrize("gs", [16, 32, 64, 128])
def test_parameters_are_read_as_words_only_where_they_are_aligned(rules, gs):
    base = 0x7F0000000100
    for s, b, ok in ((0, 0, True), (4, 8, True), (2, 0, False), (0, 2, False), (6, 2, False)):
        assert bool(rules.param_words(gs, 4096, 64, base + s, base + b)) is ok, (s, b)
    assert rules.param_words(gs, 4096, 64, base, 0)  # no biases
    assert not rules.param_words(gs, 4096, 64, base + 2, 0)
    # rows of an odd number of groups, and splits that start at an odd group
    assert bool(rules.param_words(gs, 192 if gs < 128 else 384, 6, base, base)) is (gs < 64)
    assert bool(rules.param_words(gs, 4096, 66 if gs == 128 else 65, base, base)) is (gs < 64)
