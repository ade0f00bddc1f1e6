"""CPU: which kernel a linear or P5 shape takes, on a chip of 256 CUs.

The GPU parity lists name the kernel each shape is for; here the same lists
are held against the dispatch without a GPU, and against the tables of
csrc/gemm_ks.hip and csrc/gemm_mid.hip: no tile of them is without a case.
"""

from __future__ import annotations

import os
import re

import pytest
import test_gpu_mid as mid
import test_gpu_split_k as ks
from conftest import PKG
from helpers import kernel_of

CUS = 256


def _source(name):
    return open(os.path.join(PKG, "csrc", name)).read()


def test_listed_shapes_take_the_kernels_they_name():
    for kernel, M, N, K in ks.ORACLE + ks.TILES:
        for act in (None, "gelu", "gelu_tanh"):
            assert kernel_of(M, N, K, act, cus=CUS) == kernel, (M, N, K, act)
    for kernel, M, N, K, act in mid.LINEAR + mid.LARGE:
        assert kernel_of(M, N, K, act, cus=CUS) == kernel, (M, N, K, act)
    for kernel, M, N, K in ks.P5_ORACLE + ks.P5_TILES + mid.P5 + mid.P5_LARGE:
        assert kernel_of(M, N, K, p5=True, cus=CUS) == kernel, (M, N, K)


def test_every_wave_split_k_tile_has_a_case():
    entries = re.findall(r"KS\((\d), (\d), (\d), (\d), \d\)", _source("gemm_ks.hip"))
    assert len(entries) == 25
    tiles = {nb: {20000000 + int(w) * 1000000 + int(fm) * 16000 + int(fn) * 16
                  for n, fm, fn, w in entries if int(n) == nb} for nb in (1, 2)}
    assert tiles[1] == {c[0] for c in ks.TILES}
    assert tiles[2] == {c[0] for c in ks.P5_TILES}


def test_every_tile_below_256_x_256_has_a_case():
    entries = re.findall(r"gemm_mid_kernel<(\d), (\d), (\d), (\d)>\}", _source("gemm_mid.hip"))
    assert len(entries) == 9
    tiles = {nb: {30000000 + int(g) * 4000000 + int(ax) * 32000 + int(aw) * 32
                  for n, ax, aw, g in entries if int(n) == nb} for nb in (1, 2)}
    assert tiles[1] == {c[0] for c in mid.LINEAR}
    assert tiles[2] == {c[0] for c in mid.P5 if c[0] >= 30000000}


@pytest.mark.parametrize("p5", [False, True])
def test_few_rows_and_refused_shapes(p5):
    """Two rows take the GEMV, three to eight where K % 64 != 0; from nine
    rows such K takes the eight-wave tiles.  0 for what the entry points refuse."""
    for M in range(1, 9):
        on_ks = M > 2
        assert kernel_of(M, 4096, 4096, p5=p5, cus=CUS) // 10000000 == (2 if on_ks else 1)
        assert kernel_of(M, 4096, 4128, p5=p5, cus=CUS) == 10000000
    assert kernel_of(9, 4096, 4128, p5=p5, cus=CUS) == 48256256
    for M, N, K in ((0, 64, 64), (4, 0, 64), (4, 64, 0), (4, 60, 64), (4, 64, 80), (-1, 64, 64)):
        assert kernel_of(M, N, K, p5=p5, cus=CUS) == 0
