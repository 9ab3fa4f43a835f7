"""Which tile the fp32 GEMMs take (csrc/fp32_tiles.hpp), asked on the host: results do not depend on it, times do."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "accelerated-model-architectures_amd", "csrc")
PROGRAM = """#include <stdio.h>
#include "fp32_tiles.hpp"
int main() {
    long long dw, m, n, k, e;
    while (scanf("%lld %lld %lld %lld %lld", &dw, &m, &n, &k, &e) == 5) printf("%d ", dw ? f32_small_tile_dw(m, n, k, e) : f32_small_tile(m, n, k, e));
}
"""


@pytest.fixture(scope="module")
def small(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fp32_tiles") / "ask")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-x", "c++", "-", "-o", exe], input=PROGRAM, text=True, check=True)
    return lambda *shape: subprocess.run([exe], input=" ".join(map(str, shape)), text=True, capture_output=True, check=True).stdout == "1 "


@pytest.mark.parametrize(
    "M,N,K,E,want",
    [
        (64 * 30, 2048, 1024, 64, True),  # half a large tile of rows
        (64 * 90, 2048, 1024, 64, False),
        (128 * 250, 512, 576, 128, True),
        (128 * 1000, 512, 576, 128, False),
        (8 * 512, 512, 2048, 8, True),  # less than two large tiles per compute unit
        (7354, 1376, 72, 64, False),  # a short K, padded to 96 instead of 80: measured 37 against 44 us
        (45 * 346, 1456, 112, 45, False),
        (45 * 346, 1456, 96, 45, True),  # 96 in either
    ],
)
def test_forward(small, M, N, K, E, want):
    assert small(0, M, N, K, E) == want


@pytest.mark.parametrize(
    "M,N_out,K_in,E,want",
    [
        (30 * 300, 1200, 400, 30, True),  # padded by a fifth
        (128 * 500, 576, 512, 128, False),
        (434, 3568, 424, 45, False),  # few rows: measured 66 against 91 us
        (297, 448, 1080, 128, False),
        (297 * 100, 448, 1080, 128, True),
        (0, 448, 1080, 128, False),  # rows not known
        (0, 2048, 64, 64, True),
        (0, 512, 512, 16, True),  # less than two large tiles per compute unit
    ],
)
def test_weight_gradient(small, M, N_out, K_in, E, want):
    assert small(1, M, N_out, K_in, E) == want
