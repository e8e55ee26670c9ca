"""Which kernel ti_gemm_rows takes (host code, no GPU): calls whose measured times (us, beside each) its rule has to tell apart."""
from __future__ import annotations

import pytest

import turboinfer_amd as T

WS = 64 << 20
# (bits, rows, N, K, epilogue, fold, kernel)
CALLS = [
    *[(4, m, 28672, 4096, T.EPI_SILU_MUL_F16, 1, T.ROWS_MANY) for m in (3, 8, 16)],     # few 17.9 .. 18.8, many 17.3 .. 17.5
    (4, 16, 32000, 4096, T.EPI_LOGITS_ARGMAX, 0, T.ROWS_FEW),                           # few 21.8, many 23.5
    *[(8, m, 28672, 4096, T.EPI_SILU_MUL_F16, 1, T.ROWS_MANY) for m in (17, 24, 32)],   # block 31, many 28.5 .. 29.9
    *[(8, m, 22016, 4096, T.EPI_SILU_MUL_F16, 1, T.ROWS_MANY) for m in (17, 22)],       # block 27.0 .. 27.4, many 25.9 .. 26.8
    (8, 32, 22016, 4096, T.EPI_SILU_MUL_F16, 1, T.ROWS_BLOCK),                          # block 27.0, many 27.9
    *[(36, m, 22016, 4096, T.EPI_SILU_MUL_F16, 1, T.ROWS_MANY) for m in (17, 24, 32)],  # few 23.7 .. 24.3, many 22
    *[(40, m, 4096, 11008, T.EPI_RESID_F32, 1, T.ROWS_FEW) for m in (3, 8)],            # few 12.7, many 15.5
    (16, 700, 2048, 5632, T.EPI_RESID_F32, 0, T.ROWS_MANY),                             # block 37.8, many 34.5
    (16, 384, 2048, 5632, T.EPI_RESID_F32, 0, T.ROWS_BLOCK),                            # block 24.0, many 25.5
    (4, 577, 2048, 5632, T.EPI_RESID_F32, 0, T.ROWS_BLOCK),                             # block 25.2, many 26.2
    (4, 32, 22016, 4096, T.EPI_SILU_MUL_F16, 1, T.ROWS_BLOCK),                          # block 18.3, few 21.5, many 19.9
    (4, 512, 22016, 4096, T.EPI_SILU_MUL_F16, 0, T.ROWS_BLOCK),                         # block 100, many 114
    (4, 512, 22016, 4096, T.EPI_STORE_F16, 0, T.ROWS_MANY),                             # (no output of the block kernel)
]


@pytest.mark.parametrize("bits,M,N,K,kind,fold,kernel", CALLS)
def test_rows_kernel(bits, M, N, K, kind, fold, kernel):
    assert T.lib().ti_gemm_rows_kernel(bits, M, N, K, WS, kind, fold) == kernel


def test_rows_kernel_refuses():
    L = T.lib()
    for a in [(5, 4, 64, 128, 0, 0, 0), (4, 0, 64, 128, 0, 0, 0), (4, 1025, 64, 128, 0, 0, 0), (4, 65, 64, 128, 0, 0, 1), (4, 4, 60, 128, 0, 0, 0), (4, 4, 64, 100, 0, 0, 0)]:
        assert L.ti_gemm_rows_kernel(*a) == 0, a


def test_rows_kernel_name():
    """The labels of a step of 64 int4 streams: three products on the block kernel, the split one and the logits on the many-rows one."""
    got = [T.rows_kernel_name(4, 64, n, k, kind, fold) for n, k, kind, fold in
           [(12288, 4096, T.EPI_QKV_ROPE_KV, True), (4096, 4096, T.EPI_RESID_F32, True), (22016, 4096, T.EPI_SILU_MUL_F16, True),
            (4096, 11008, T.EPI_RESID_F32, True), (32000, 4096, T.EPI_LOGITS_ARGMAX, False)]]
    assert got == ["gemm_block_kernel"] * 3 + ["gemm_wide_kernel"] * 2
    assert T.rows_kernel_name(4, 64, 60, 128, T.EPI_STORE_F32) == ""
