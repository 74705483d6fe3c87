"""The rules that choose between two forms of a call, at shapes where both were timed on MI355X
and one is clearly the faster (CPU only: no kernel runs)."""

import ctypes

import pytest

from ksdraft_amd import _lib


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
