"""The shared-K/V prompt attention at head_dim 64 (4- and 8-wave workgroups) at any grid size: partial query blocks, GQA
groups of 1 .. 16, prefixes before the chunk, positions in any order, the prefix ending at the cache's last row --
against the decode kernel and, by row, float64 (bound of test_gpu_prefill_attn.py: fp16 output, rtol = atol = 4e-3)."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_prefill_attn import _case

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[2, 3], ids=["shared4", "shared8"])
def kernel(request, ti):
    L = ti.lib()
    assert L.ti_attn_prefill_set_kernel(request.param) == 0
    yield request.param
    assert L.ti_attn_prefill_set_kernel(0) == request.param


@pytest.mark.parametrize("M,nh,nkv,start,max_seq", [
    (1, 4, 4, 0, 16), (15, 8, 1, 0, 16), (37, 4, 4, 0, 64), (64, 8, 2, 5, 80), (129, 8, 4, 0, 129), (77, 32, 2, 3, 96),
    (300, 32, 4, 600, 900), (333, 8, 8, 1000, 1333), (1000, 32, 4, 0, 1001),
])
def test_shared_kv(ti, kernel, M, nh, nkv, start, max_seq):
    pos = (start + np.arange(M)).astype(np.int32)
    q, kc, vc, got, dec = _case(ti, M, nh, nkv, 64, pos, max_seq, seed=M + nh)
    if dec is not None:
        np.testing.assert_allclose(got, dec, rtol=4e-3, atol=4e-3)
    for m in sorted({0, M // 2, M - 1}):
        S, G = int(pos[m]) + 1, nh // nkv
        for h in (0, nh - 1):
            s = kc[h // G, :S].astype(np.float64) @ q[m].reshape(nh, 64)[h].astype(np.float64) / 8.0
            p = np.exp(s - s.max())
            ref = p @ vc[h // G, :S].astype(np.float64) / p.sum()
            np.testing.assert_allclose(got[m].reshape(nh, 64)[h], ref, rtol=4e-3, atol=4e-3)


def test_any_positions(ti, kernel):
    pos = np.random.RandomState(5).permutation(900)[:333].astype(np.int32)
    _, _, _, got, dec = _case(ti, 333, 8, 2, 64, pos, 1024, seed=9)
    np.testing.assert_allclose(got, dec, rtol=4e-3, atol=4e-3)
