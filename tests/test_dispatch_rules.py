"""The rules that choose between two forms of a call, at shapes where both were timed on MI355X
and one is clearly the faster (CPU only: no kernel runs)."""

import ctypes

import pytest
import torch

from ksdraft_amd import _lib
from ksdraft_amd.kernels.ks3_triton import _one_launch_pays


# (rows, charts, time without the table, time with it), microseconds
COMPOSED = [(1464, 1024, 10.7, 11.1), (2929, 1024, 17.1, 14.3), (28125, 256, 34.3, 19.0), (24000, 300, 43.5, 24.8),
            (424, 5888, 15.1, 20.3), (1222, 5888, 34.7, 26.3), (2574, 777, 14.4, 18.9), (4504, 777, 22.0, 19.9),
            (2049, 2049, 23.7, 27.5), (873, 6869, 31.5, 39.6), (240, 30000, 37.0, 46.0), (1, 1, 4.5, 29.9)]
FUSED = [(1464, 1024, 9.5, 13.0), (5859, 1024, 25.1, 19.6), (56250, 128, 30.0, 22.7), (24000, 300, 37.4, 25.7),
         (1019, 5888, 25.6, 28.9), (1222, 5888, 30.2, 28.9), (873, 6869, 28.3, 35.3), (240, 30000, 32.3, 45.7)]


@pytest.mark.parametrize("fused,M,F,direct,table", [(0, *r) for r in COMPOSED] + [(1, *r) for r in FUSED])
def test_spine_table(fused, M, F, direct, table):
    c = ctypes.c_int(-1)
    _lib.call("ksd_ks3_spine_needs_table", M, F, fused, ctypes.byref(c))
    assert c.value == int(table < direct)


# (rows, columns, K, the persistent kernel's time, the few-row kernel's), microseconds
FEW_ROWS = [(1, 1536, 1536, 11.6, 4.4), (16, 16384, 1920, 14.9, 12.9), (16, 16384, 2048, 14.1, 16.3),
            (12, 16384, 2048, 14.5, 15.4), (5, 16384, 2048, 14.1, 13.4), (16, 6144, 4096, 14.3, 15.8),
            (8, 8192, 4096, 14.9, 14.0), (16, 8192, 3840, 15.6, 13.5), (16, 1000, 8192, 16.1, 16.9),
            (5, 1024, 8192, 15.7, 14.6), (16, 2048, 7680, 16.6, 15.2), (32, 8192, 2048, 13.0, 12.2),
            (64, 4096, 2048, 13.4, 11.2), (512, 512, 2048, 13.3, 11.2), (4096, 64, 2048, 13.3, 11.3),
            (64, 5888, 1536, 11.2, 13.4)]


@pytest.mark.parametrize("M,N,K,persistent,few", FEW_ROWS)
def test_few_row_gemm(M, N, K, persistent, few):
    c = ctypes.c_int(-1)
    _lib.call("ksd_w8a8_gemm_few_rows", M, N, K, ctypes.byref(c))
    assert c.value == int(few < persistent)


# (M, K, N, time in one launch, time of the GEMM and the spine), microseconds
PROJECT = [(257, 128, 1536, 20.0, 11.0), (512, 1536, 5888, 34.0, 29.0),
           (700, 1536, 5888, 57.0, 44.0), (1024, 1536, 5888, 57.0, 51.0), (600, 128, 5888, 25.0, 28.0),
           (1024, 128, 4096, 24.0, 33.0), (1024, 512, 4096, 28.0, 35.0), (512, 512, 4096, 25.0, 21.0),
           (1024, 128, 3001, 22.0, 29.0), (512, 128, 3001, 20.0, 18.7), (512, 768, 5001, 25.1, 28.3),
           (700, 1792, 5001, 35.0, 38.7), (1024, 1536, 5001, 56.0, 52.0), (1024, 1792, 3001, 31.7, 33.5),
           (1024, 768, 6869, 52.6, 54.9), (896, 512, 6869, 44.0, 48.0), (700, 1536, 6869, 57.0, 49.0),
           (1024, 128, 6912, 41.0, 47.0), (1024, 512, 6912, 49.0, 47.0), (1025, 128, 3001, 24.0, 29.0)]


@pytest.mark.parametrize("M,K,N,one,two", PROJECT)
def test_one_launch_projection(M, K, N, one, two):
    a, w = (torch.empty(r, K, dtype=torch.int8, device="meta") for r in (M, N))
    assert _one_launch_pays(a, w) == (one < two and M <= 1024)  # never taken past 1024 rows
