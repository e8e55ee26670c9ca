"""Decode attention of GQA batches dealt evenly over the workgroups (ti_attn_decode_spread) against float64 on the fp16
cache: ragged lengths around the unit of 32 keys, streams that end and begin inside a workgroup's piece, one long stream
beside short ones, more pieces than units.  Bound: fp16 output, half a unit in the last place (2^-11 relative), plus the
fp32 and hi + lo roundings of scores below 2^-17 of the largest output."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_kernels import dev

pytestmark = pytest.mark.gpu


def reference(q, k, v, lens, G):
    out = np.zeros(q.shape)
    for m, L in enumerate(lens):
        for h in range(q.shape[1]):
            if L <= 0:
                continue
            s = k[m, h // G, :L].astype(np.float64) @ q[m, h].astype(np.float64) / np.sqrt(q.shape[2])
            p = np.exp(s - s.max())
            out[m, h] = p @ v[m, h // G, :L].astype(np.float64) / p.sum()
    return out


def run(ti, lens, kvh, G, hd, parts, max_seq, qscale=1.0, seed=0, calls=2):
    rng = np.random.default_rng(seed)
    M, heads, L_ = len(lens), kvh * G, ti.lib()
    q = (rng.standard_normal((M, heads, hd)) * qscale).astype(np.float32)
    k = rng.standard_normal((M, kvh, max_seq, hd)).astype(np.float16)
    v = rng.standard_normal((M, kvh, max_seq, hd)).astype(np.float16)
    for m, L in enumerate(lens):   # rows past a stream's keys are not to be used
        k[m, :, max(L, 0):], v[m, :, max(L, 0):] = np.nan, np.nan
    qd, kd, vd, pd = dev(ti, q), dev(ti, k), dev(ti, v), dev(ti, np.array(lens, np.int32) - 1)
    ws = ti.DeviceBuffer(L_.ti_attn_spread_workspace_bytes(M, heads, hd, parts))
    ws.zero()
    ref = reference(q, k, v, lens, G)
    got = []
    for _ in range(calls):
        out = ti.DeviceBuffer(M * heads * hd * 2)
        ti.check(L_.ti_memset(out.ptr, 0xff, out.nbytes, None))
        ti.check(L_.ti_attn_decode_spread(qd.ptr, kd.ptr, vd.ptr, kvh * max_seq * hd, max_seq, pd.ptr, M, heads, kvh, hd, parts, ws.ptr,
                                          out.ptr, None))
        ti.sync()
        got.append(out.download(np.float16, (M, heads, hd)).astype(np.float64))
        # scores of magnitude |s| carry 2^-20 |s| (q's split, fp32 sums): p and so o move by that much
        tol = 2.0**-11 * np.abs(ref) + (2.0**-17 * max(1.0, qscale * np.sqrt(hd) / 8)) * 4
        assert (np.abs(got[-1] - ref) <= tol).all(), np.abs(got[-1] - ref).max()
    assert all((g == got[0]).all() for g in got)   # tickets re-armed, merge order fixed


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("G", [4, 8])
@pytest.mark.parametrize("parts", [1, 5, 32])
def test_ragged_lengths(ti, hd, G, parts):
    run(ti, [1, 31, 32, 33, 64, 255, 256, 257, 288, 700, 2, 513], 2, G, hd, parts, 704)


@pytest.mark.parametrize("lens", [[1], [1500], [1500, 1], [1, 1500, 3], [40] * 70, [1] * 130 + [900] + [5] * 9])
def test_stream_counts(ti, lens):
    run(ti, lens, 1, 4, 64, 64, 1500)


def test_large_queries_and_an_empty_stream(ti):
    run(ti, [300, 0, 65], 2, 8, 128, 32, 320, qscale=40.0)


def test_queries_past_fp16(ti):
    """|q| / sqrt(hd) above fp16's largest value: the scores' order decides, as in fp32."""
    rng = np.random.default_rng(2)
    M, kvh, G, hd, S = 2, 1, 4, 64, 96
    q = (rng.standard_normal((M, kvh * G, hd)) * 4e6).astype(np.float32)
    k, v = (rng.standard_normal((M, kvh, S, hd)).astype(np.float16) for _ in range(2))
    L_, ws = ti.lib(), ti.DeviceBuffer(ti.lib().ti_attn_spread_workspace_bytes(M, kvh * G, hd, 4))
    ws.zero()
    out = ti.DeviceBuffer(M * kvh * G * hd * 2)
    bufs = [dev(ti, x) for x in (q, k, v, np.array([S - 1, S - 9], np.int32))]
    ti.check(L_.ti_attn_decode_spread(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, kvh * S * hd, S, bufs[3].ptr, M, kvh * G, kvh, hd, 4, ws.ptr,
                                      out.ptr, None))
    ti.sync()
    got = out.download(np.float16, (M, kvh * G, hd)).astype(np.float64)
    ref = reference(q, k, v, [S, S - 8], G)   # (a one-hot softmax: the gaps between scores are ~ 1e5)
    assert np.abs(got - ref).max() <= 2.0**-11 * np.abs(ref).max()


@pytest.mark.parametrize("hd,G", [(64, 4), (64, 8), (128, 4), (128, 8)])
@pytest.mark.parametrize("qscale", [0.01, 0.3, 1.0, 4.0])
def test_error_of_the_fp32_rows(ti, hd, G, qscale):
    """The segments' fp32 rows, merged in float64, against float64: no further off than ti_attn_decode's (fp32 throughout).
    Both add the same terms in another order, so their errors over 10^4 values agree to the scatter of such sums: a
    quarter, and a third where the scores' own roundings decide (|score| ~ 4)."""
    lens, kvh, parts, splits = [1000, 1400, 700, 900, 1200, 450], 2, 32, 4
    rng = np.random.default_rng(hd + G)
    M, heads, S, L_ = len(lens), kvh * G, max(lens), ti.lib()
    q = (rng.standard_normal((M, heads, hd)) * qscale).astype(np.float32)
    k, v = (rng.standard_normal((M, kvh, S, hd)).astype(np.float16) for _ in range(2))
    ref = reference(q, k, v, lens, G)
    bufs = [dev(ti, x) for x in (q, k, v, np.array(lens, np.int32) - 1)]
    a = (bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, kvh * S * hd, S, bufs[3].ptr, M, heads, kvh, hd)
    out, err = ti.DeviceBuffer(M * heads * hd * 2), []

    def merged(rows):   # rows [parts][heads][hd + 4]: o, maximum, sum
        f = np.exp(rows[..., hd] - rows[..., hd].max(axis=0))
        return (rows[..., :hd] * f[..., None]).sum(axis=0) / (rows[..., hd + 1] * f).sum(axis=0)[..., None]

    for spread in (False, True):
        n = L_.ti_attn_spread_workspace_bytes(M, heads, hd, parts) if spread else L_.ti_attn_workspace_bytes(M, heads, hd, splits)
        ws = ti.DeviceBuffer(n)
        ws.zero()
        ti.check((L_.ti_attn_decode_spread if spread else L_.ti_attn_decode)(*a, parts if spread else splits, ws.ptr, out.ptr, None))
        ti.sync()
        raw = ws.download(np.float32, (n // 4,)).astype(np.float64)
        if spread:
            rows = raw[n // 4 - (parts + M) * heads * (hd + 4):].reshape(parts + M, heads, hd + 4)
            units = [-(-x // 32) for x in lens]
            segs = [-(-u // max(12, -(-sum(units) // parts))) for u in units]
            first = np.cumsum([0] + segs)
            assert min(segs) > 1
            got = np.stack([merged(rows[first[m]:first[m + 1]]) for m in range(M)])
        else:
            rows = raw[n // 4 - M * heads * splits * (hd + 4):].reshape(M, heads, splits, hd + 4)
            got = np.stack([merged(rows[m].transpose(1, 0, 2)) for m in range(M)])
        err.append(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    assert err[1] <= (1.25 if qscale < 4 else 1.35) * err[0], err


def test_refusals(ti):
    f = ti.lib().ti_attn_decode_spread
    ok = [1, 1, 1, 8 * 64 * 64, 64, 1, 2, 32, 8, 64, 4, 1, 1, None]
    for i, bad in ((0, None), (3, 100), (6, 0), (7, 24), (8, 16), (9, 96), (10, 0), (11, None)):
        a = list(ok)
        a[i] = bad
        assert f(*a) != 0
