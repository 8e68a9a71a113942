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
extern "C" int plan(int M, int N, int K, int gs, int bits) {
    const eq::QmmPlan p = eq::qmm_plan(M, N, K, gs, bits, true, 256);
    return p.tm * 10000 + p.tn * 1000 + p.splits;
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
    lib.tile = lambda *shape: ((v := lib.plan(*shape)) // 10000 * 32, v // 1000 % 10 * 128, v % 1000)
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


# (M, N, K, group size, bits) -> tile rows, tile columns, splits of K on 256 CUs:
# 8-bit codes above 96 rows on split 128 x 128 tiles, 4-bit ones and shorter K on
# unsplit 64 x 128 ones; group 16 split where unsplit tiles of many steps lost, and
# on 128 x 128 tiles above 128 rows where those keep 16 chunks to a piece.
@pytest.mark.parametrize("shape,tile", [
    ((128, 14336, 4096, 64, 8), (128, 128, 2)), ((97, 12288, 4096, 128, 8), (128, 128, 2)),
    ((128, 14336, 4096, 64, 4), (64, 128, 1)), ((96, 14336, 4096, 64, 8), (96, 128, 2)),
    ((120, 16384, 3072, 128, 8), (64, 128, 1)), ((120, 9216, 2048, 64, 8), (64, 128, 1)),
    ((87, 12160, 5248, 16, 4), (96, 128, 2)), ((128, 10240, 3072, 16, 8), (128, 128, 3)),
    ((955, 768, 13952, 16, 4), (128, 128, 5)), ((300, 1024, 4096, 16, 4), (64, 128, 6)),
    # the tiles that the GPU tests name
    ((66, 4224, 2048, 64, 4), (96, 128, 4)), ((96, 5504, 2112, 16, 8), (96, 128, 3)), ((77, 16512, 192, 32, 8), (96, 128, 1)),
    ((500, 3968, 4096, 128, 8), (128, 128, 2)), ((955, 768, 5120, 16, 8), (128, 128, 5)), ((65, 384, 2048, 64, 4), (64, 128, 4)),
    ((300, 512, 2048, 64, 8), (64, 128, 4)), ((1029, 5760, 1280, 64, 4), (128, 256, 1)), ((500, 3968, 4096, 16, 4), (128, 256, 4)),
])
def test_tiles_and_splits(rules, shape, tile):
    assert rules.tile(*shape) == tile


def test_short_k_needs_no_workspace(rules):
    """64 x 128 tiles that cover half the CUs at a short K stay unsplit (a call
    without workspace can be captured without an eager one before)."""
    for gs in (32, 64, 128):
        for bits in (4, 8):
            for M, N, K in ((17, 16512, 2048), (64, 16512, 1024), (77, 8320, 2048), (100, 9216, 2048), (70, 10240, 3072)):
                assert rules.tile(M, N, K, gs, bits)[2] == 1, (M, N, K, gs, bits)
