"""Which products with few tiles of outputs take a workgroup a tile (ti_dense_tile 0 x 0; host code, no GPU): calls whose measured times (us, beside each: blocks /
a workgroup a tile) its rule has to tell apart."""
from __future__ import annotations

import ctypes as C

import pytest

import turboinfer_amd as T

CALLS = [   # dtype, rows, N, K, a workgroup a tile
    (T.DT_BF16, 66, 1024, 2048, True),      # 8.5 / 5.7
    (T.DT_BF16, 2048, 64, 2048, True),      # 8.4 / 7.8
    (T.DT_BF16, 1000, 128, 2048, True),     # 8.4 / 7.6
    (T.DT_BF16, 700, 128, 3072, True),      # 10.6 / 10.1
    (T.DT_BF16, 1000, 64, 8192, True),      # 22.0 / 15.0
    (T.DT_BF16, 1200, 64, 8192, False),     # 22.0 / 23.6
    (T.DT_BF16, 2048, 64, 4096, False),     # 13.0 / 14.6
    (T.DT_BF16, 1000, 128, 4096, False),    # 12.9 / 14.6
    (T.DT_BF16, 500, 256, 8192, True),      # 22.9 / 21.4
    (T.DT_BF16, 250, 512, 4096, True),      # 12.9 / 11.2
    (T.DT_BF16, 640, 256, 2048, False),     # 13.2 / 15.9
    (T.DT_BF16, 300, 64, 256, False),       # 3.86 / 3.87
    (T.DT_F32, 2048, 64, 8192, True),       # 78.5 / 44.4
    (T.DT_F32, 2048, 128, 8192, False),     # 79.0 / 83.7
    (T.DT_F32, 2048, 128, 2048, True),      # 23.8 / 23.9
    (T.DT_F32, 1000, 256, 8192, True),      # 79.5 / 74.9
]


@pytest.mark.parametrize("dtype,M,N,K,few", CALLS)
def test_few_tiles(ti_host, dtype, M, N, K, few):
    rows, cols = C.c_int(0), C.c_int(0)
    d = T.DenseArgs(lda=K, ldo=N, M=M, N=N, K=K, batch=1, epi=T.DE_F32, dtype=dtype)
    T.check(T.lib().ti_dense_tile(C.byref(d), C.byref(rows), C.byref(cols)))
    assert ((rows.value, cols.value) == (0, 0)) == few
