"""ti_gemm_rows: row-major fp16 rows against packed weights of every format, against the weights' exact values in float64
(test_gpu_kernels.py's bound: fp32 summation order).  Calls run on each of its kernels that has their rows, the few-rows one
(gemm_few.hip, up to 48), the many-rows one (gemm_wide.hip) and the block one (gemm_block.hip), whichever the call itself would take;
test_rows_each_shape takes them through every block shape by name."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from test_gpu_g32 import g32_weight, pack_g32
from test_gpu_kernels import assert_close_dot, deq, dev

pytestmark = pytest.mark.gpu
f16, f32 = np.float16, np.float32
G32, WS = 32, 64 << 20


@pytest.fixture(scope="module")
def ws(ti):
    b = ti.DeviceBuffer(WS)
    b.zero()
    return b


def weight(ti, oracle, bits, K, N, rng):
    """(device tiles, device scales, the weight's exact values [K][N])."""
    if bits & G32:
        q, d, w = g32_weight(rng, K, N, bits & 15)
        t, s = pack_g32(ti, q, d, bits & 15)
        return t, s, w.astype(f32)
    w = (rng.standard_normal((K, N)) * 0.03).astype(f32)
    t, s = ti.wpack_host(w, bits)
    return dev(ti, t), dev(ti, s), w.astype(f16).astype(f32) if bits == 16 else deq(oracle, w, bits)


def kernels(ti, M, bits, block=True):
    """The kernels of a call of M rows; block: an output that the block kernel writes."""
    if M <= 48:
        return ti.ROWS_FEW, ti.ROWS_MANY
    return (ti.ROWS_AUTO, ti.ROWS_MANY) + ((ti.ROWS_BLOCK,) if block and not bits & G32 else ())


def rows(ti, bits, td, sd, xd, M, N, K, ep, ldx=None, ws=None, kernel=0, h=None, norm_w=None):
    ep.splitk_ws, ep.splitk_bytes = (ws.ptr, ws.nbytes) if ws is not None else (None, 0)
    rc = ti.lib().ti_gemm_rows_on(kernel, td.ptr, sd.ptr, bits, xd.ptr, ldx or K, h, norm_w, 1e-5, M, N, K, C.byref(ep), None)
    ti.check(rc)
    ti.sync()
    if ws is not None:
        assert not ws.download(np.int32, (65536,)).any(), "split-K tickets not re-armed"


# rows at the edges of the 16-, 32- and 64-row blocks, ragged column tiles, one k-group, odd numbers of them, narrow
# outputs whose K is split, wide ones in several rounds
@pytest.mark.parametrize("M,K,N", [(1, 128, 16), (16, 384, 80), (17, 1152, 4000), (32, 4096, 4096 + 48), (33, 128, 64),
                                   (64, 1152, 6208), (65, 2048, 2560), (129, 384, 400), (333, 5632, 2048), (1000, 640, 11264),
                                   (1024, 256, 1040), (100, 14336, 512)])
@pytest.mark.parametrize("bits", [4, 8, 16, 4 | G32, 8 | G32])
def test_rows_store(ti, oracle, ws, bits, M, K, N):
    rng = np.random.RandomState(M * 7 + K + N + bits)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    ldx = K + 8 * (M % 3)
    x = rng.standard_normal((M, ldx)).astype(f16)
    xd, yd = dev(ti, x), ti.DeviceBuffer(M * N * 4)
    xa = x[:, :K].astype(f32)
    ref = xa.astype(np.float64) @ w.astype(np.float64)
    for kernel in kernels(ti, M, bits):
        for k in (None, ws):
            yd.zero()
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out = ti.EPI_STORE_F32, N, yd.ptr
            rows(ti, bits, td, sd, xd, M, N, K, ep, ldx, k, kernel)
            assert_close_dot(yd.download(f32, (M, N)), ref, xa, w)


# the few-rows kernel (gemm_few.hip): rows at the edges of its 16-, 32- and 48-row blocks, waves without a group of k (K below
# 1024), with one, two, three, four and five, columns of several rounds and a ragged last block of columns
@pytest.mark.parametrize("M,K,N", [(2, 128, 16), (3, 896, 48), (15, 1024, 4112), (16, 1152, 2048), (4, 2176, 8208), (17, 3072, 80),
                                   (31, 3968, 4112), (32, 2048, 2064), (33, 4224, 112), (47, 896, 1040), (48, 5120, 272)])
@pytest.mark.parametrize("bits", [4, 8, 16, 4 | G32, 8 | G32])
def test_rows_few(ti, oracle, bits, M, K, N):
    rng = np.random.RandomState(M * 11 + K + N + bits)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    ldx = K + 8 * (M % 2)
    x = rng.standard_normal((M, ldx)).astype(f16)
    xd, yd = dev(ti, x), ti.DeviceBuffer((M + 1) * N * 4)
    yd.zero()
    ep = ti.Epilogue()
    ep.kind, ep.ldo, ep.out = ti.EPI_STORE_F32, N, yd.ptr
    rows(ti, bits, td, sd, xd, M, N, K, ep, ldx, kernel=ti.ROWS_FEW)
    y, xa = yd.download(f32, (M + 1, N)), x[:, :K].astype(f32)
    assert_close_dot(y[:M], xa.astype(np.float64) @ w.astype(np.float64), xa, w)
    assert not y[M].any()


# (24 .. 47 rows by the few-rows kernel: waves with none to five groups of k, its 16- and 32-column blocks with a ragged last one)
@pytest.mark.parametrize("M,K,N", [(24, 384, 96), (100, 1152, 1040), (700, 2048, 512), (3, 2176, 4112), (16, 5120, 4112), (31, 2176, 4112),
                                   (47, 5120, 272)])
def test_rows_affine_blocks(ti, oracle, ws, M, K, N):
    """Q4_1 blocks (4 | 32 | 64): the offset term through the block's sum of x."""
    from test_gpu_g32 import pack_q1
    rng = np.random.RandomState(M)
    q = rng.randint(0, 16, (K, N)).astype(np.uint8)
    d = (rng.uniform(0.5, 1.5, (K // 32, N)) * 0.01).astype(f16)
    m = (rng.standard_normal((K // 32, N)) * 0.05).astype(f16)
    td, sd = pack_q1(ti, q, d, m)
    w = np.repeat(d.astype(np.float64), 32, 0) * q + np.repeat(m.astype(np.float64), 32, 0)
    parts = np.repeat(np.abs(d.astype(np.float64)), 32, 0) * 16 + np.repeat(np.abs(m.astype(np.float64)), 32, 0)
    x = rng.standard_normal((M, K)).astype(f16)
    xd, yd = dev(ti, x), ti.DeviceBuffer(M * N * 4)
    for kernel in kernels(ti, M, 4 | G32 | 64):
        yd.zero()
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = ti.EPI_STORE_F32, N, yd.ptr
        rows(ti, 4 | G32 | 64, td, sd, xd, M, N, K, ep, ws=ws, kernel=kernel)
        # fp32 sums of d (q - 8) x and (8 d + m) x: the bound is on the parts' magnitudes
        assert np.all(np.abs(yd.download(f32, (M, N)) - x.astype(np.float64) @ w) <= 2e-5 * (np.abs(x.astype(np.float64)) @ parts) + 1e-6)


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M", [5, 30, 57, 150])
def test_rows_epilogues(ti, oracle, ws, bits, M):
    """fp16 store, residual add, SiLU * up and logits + argmax; rows of an odd pitch take the per-element form."""
    K, N = 1152, 1056
    rng = np.random.RandomState(M + bits)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    x = rng.standard_normal((M, K)).astype(f16)
    xd, xa = dev(ti, x), x.astype(np.float64)
    ref = xa @ w.astype(np.float64)
    for kernel, ldo in [(k, l) for k in kernels(ti, M, bits, False) for l in (N, N + 3)]:   # (the block kernel: test_rows_block)
        r = rng.standard_normal((M, ldo)).astype(f32)
        rd = dev(ti, r)
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = ti.EPI_RESID_F32, ldo, rd.ptr
        rows(ti, bits, td, sd, xd, M, N, K, ep, ws=ws, kernel=kernel)
        got = rd.download(f32, (M, ldo))
        assert_close_dot(got[:, :N] - r[:, :N], ref, x.astype(f32), w, rel=5e-5)
        np.testing.assert_array_equal(got[:, N:], r[:, N:])
        sil = ref.reshape(M, N // 16, 2, 8)
        sil = (sil[:, :, 1] * (sil[:, :, 0] / (1 + np.exp(-sil[:, :, 0])))).reshape(M, N // 2)
        hd = ti.DeviceBuffer(M * ldo * 2)
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = ti.EPI_SILU_MUL_F16, ldo, hd.ptr
        rows(ti, bits, td, sd, xd, M, N, K, ep, ws=ws, kernel=kernel)
        np.testing.assert_allclose(hd.download(f16, (M, ldo))[:, : N // 2].astype(np.float64), sil, rtol=3e-3, atol=2e-3)
        ep.kind = ti.EPI_STORE_F16
        rows(ti, bits, td, sd, xd, M, N, K, ep, ws=ws, kernel=kernel)
        np.testing.assert_allclose(hd.download(f16, (M, ldo))[:, :N].astype(np.float64), ref, rtol=2e-3, atol=1e-4)
    for kernel in kernels(ti, M, bits, False):
        ld, am = ti.DeviceBuffer(M * N * 4), ti.DeviceBuffer(M * ti.ARGMAX_SLOTS * 8)
        am.zero()
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out, ep.argmax = ti.EPI_LOGITS_ARGMAX, N, ld.ptr, am.ptr
        rows(ti, bits, td, sd, xd, M, N, K, ep, ws=ws, kernel=kernel)
        lg = ld.download(f32, (M, N))
        keys = am.download(np.uint64, (M, ti.ARGMAX_SLOTS)).max(axis=1)
        np.testing.assert_array_equal((0xFFFFFFFF - (keys & 0xFFFFFFFF)).astype(np.int64), np.argmax(lg, axis=1))
        np.testing.assert_allclose(lg, ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("hd,M", [(64, 21), (128, 70)])
def test_rows_qkv(ti, oracle, ws, hd, M):
    """RoPE + KV append against the fused kernel's epilogue on the same products (int8, 16-row calls)."""
    heads, kvh, K, S = 4, 2, 512, 96
    qd, kd = heads * hd, kvh * hd
    N = qd + 2 * kd
    rng = np.random.RandomState(hd)
    td, sd, _ = weight(ti, oracle, 8, K, N, rng)
    xd = dev(ti, rng.standard_normal((M, K)).astype(f16))
    pos = rng.permutation(S)[:M].astype(np.int32)
    pd = dev(ti, pos)
    cs = dev(ti, ti.rope_table(np.arange(S), hd, 10000.0))
    outs = []
    for kernel in kernels(ti, M, 8) + (None,):
        q, k, v = ti.DeviceBuffer(M * qd * 4), ti.DeviceBuffer(kvh * S * hd * 2), ti.DeviceBuffer(kvh * S * hd * 2)
        for b in (k, v):
            b.zero()
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out, ep.q_dim, ep.kv_dim, ep.head_dim, ep.max_seq = ti.EPI_QKV_ROPE_KV, qd, q.ptr, qd, kd, hd, S
        ep.pos, ep.rope_cs, ep.k_cache, ep.v_cache, ep.kv_stream_stride = pd.ptr, cs.ptr, k.ptr, v.ptr, 0
        if kernel is not None:
            rows(ti, 8, td, sd, xd, M, N, K, ep, ws=ws, kernel=kernel)
        else:
            for m in range(0, M, 16):
                ep.out, ep.pos = q.ptr + m * qd * 4, pd.ptr + 4 * m
                ti.check(ti.lib().ti_gemm_wq_a16(td.ptr, sd.ptr, 8, xd.ptr + m * K * 2, ti.X_F16, K, None, 1e-5, min(16, M - m), N, K,
                                                 C.byref(ep), None))
            ti.sync()
        outs.append([q.download(f32, (M, qd)), k.download(f16, (kvh, S, hd)).astype(f32), v.download(f16, (kvh, S, hd)).astype(f32)])
    for out in outs[:-1]:
        for a, b in zip(out, outs[-1]):
            np.testing.assert_allclose(a, b, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("bits", [4, 8, 16, 4 | G32])
@pytest.mark.parametrize("M", [3, 16, 17, 45, 64])
def test_rows_fold(ti, oracle, ws, bits, M):
    """The batched fold: residual epilogue writes fp16(h * w) and sums of h^2, the next call divides by the rms."""
    L, K, H, N = ti.lib(), 1152, 1024, 768
    rng = np.random.RandomState(M + bits)
    to, so, wo = weight(ti, oracle, bits, K, H, rng)
    t2, s2, w2 = weight(ti, oracle, bits, H, N, rng)
    act = rng.standard_normal((M, K)).astype(f16)
    h0 = rng.standard_normal((M, H)).astype(f32)
    nw = (1 + 0.1 * rng.standard_normal(H)).astype(f32)
    ad, nwd = dev(ti, act), dev(ti, nw)
    for kernel, k in [(a, b) for a in kernels(ti, M, bits) for b in (ws, None)]:   # (the many-rows kernel splits K with a workspace)
        n_ss = L.ti_gemm_rows_fold_partials_on(kernel, bits, M, H, K, WS if k else 0)
        assert 1 <= n_ss <= 4096
        bits_out = []
        for _ in range(2):
            hd, fx, ss, yd = dev(ti, h0), ti.DeviceBuffer(M * H * 2), ti.DeviceBuffer(n_ss * 64 * 4), ti.DeviceBuffer(M * N * 4)
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out = ti.EPI_RESID_F32, H, hd.ptr
            ep.fold_w, ep.fold_x, ep.fold_ss = nwd.ptr, fx.ptr, ss.ptr
            rows(ti, bits, to, so, ad, M, H, K, ep, ws=k, kernel=kernel)
            h1 = hd.download(f32, (M, H))
            assert_close_dot(h1 - h0, act.astype(np.float64) @ wo.astype(np.float64), act.astype(f32), wo, rel=5e-5)
            np.testing.assert_array_equal(fx.download(np.uint16, (M, H)), (h1 * nw).astype(f16).view(np.uint16))
            np.testing.assert_allclose(ss.download(f32, (n_ss, 64))[:, :M].sum(axis=0), (h1.astype(np.float64) ** 2).sum(axis=1), rtol=1e-5)
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out, ep.ss_in, ep.n_ss = ti.EPI_STORE_F32, N, yd.ptr, ss.ptr, n_ss
            rows(ti, bits, t2, s2, fx, M, N, H, ep, ws=k, kernel=kernel)
            y = yd.download(f32, (M, N))
            bits_out.append(y.view(np.uint32))
        rms = np.sqrt((h1.astype(np.float64) ** 2).mean(axis=1) + 1e-5)
        xf = (h1 * nw).astype(f16).astype(np.float64) / rms[:, None]
        assert_close_dot(y, xf @ w2.astype(np.float64), xf.astype(f32), w2, rel=5e-5)
        np.testing.assert_array_equal(*bits_out)   # fixed-order sums


def test_rows_refusals(ti):
    L = ti.lib()
    b = ti.DeviceBuffer(1 << 20)
    ep = ti.Epilogue()
    ep.kind, ep.ldo, ep.out = ti.EPI_STORE_F32, 64, b.ptr
    ok = (b.ptr, b.ptr, 8, b.ptr, 256, 1e-5, 4, 64, 256)
    for i, v in [(2, 5), (2, 16 | G32), (3, b.ptr + 2), (4, 260), (4, 128), (6, 0), (6, 2000), (7, 60), (8, 200)]:
        a = list(ok)
        a[i] = v
        assert L.ti_gemm_rows(*a, C.byref(ep), None) != 0, (i, v)
    on = (b.ptr, b.ptr, 8, b.ptr, 256, None, None, 1e-5)
    S = ti.ROWS_SHAPE
    for kernel, M in [(ti.ROWS_BLOCK + 1, 40), (-1, 4), (ti.ROWS_FEW, 49), (ti.ROWS_BLOCK, 16), (S, 40), (ti.ROWS_FEW + 12 * S, 4), (ti.ROWS_MANY + 6 * S, 4),
                      (ti.ROWS_BLOCK + 13 * S, 40), (ti.ROWS_FEW + S, 17), (ti.ROWS_MANY + 5 * S, 17)]:
        assert L.ti_gemm_rows_on(kernel, *on, M, 64, 256, C.byref(ep), None) != 0, (kernel, M)
        assert L.ti_gemm_rows_fold_partials_on(kernel, 8, M, 64, 256, 0) == 0, (kernel, M)
    # what the block kernel does not take: few rows, blocks of 32, fp16 rows, logits, a pitch of no whole 16-byte pieces
    for bits, M, kind, ldo in [(4, 16, ti.EPI_STORE_F32, 64), (16, 32, ti.EPI_STORE_F32, 64), (8 | G32, 40, ti.EPI_STORE_F32, 64), (8, 40, ti.EPI_STORE_F16, 64),
                               (8, 40, ti.EPI_LOGITS_ARGMAX, 64), (8, 40, ti.EPI_STORE_F32, 65)]:
        e2 = ti.Epilogue()
        e2.kind, e2.ldo, e2.out, e2.argmax = kind, ldo, b.ptr, b.ptr
        assert L.ti_gemm_rows_on(ti.ROWS_BLOCK, b.ptr, b.ptr, bits, *on[3:], M, 64, 256, C.byref(e2), None) != 0, (bits, M, kind, ldo)
    ep.kind, ep.fold_x = ti.EPI_RESID_F32, b.ptr
    assert L.ti_gemm_rows(*ok, C.byref(ep), None) != 0


@pytest.mark.parametrize("M,K,N", [(300, 256, 11280), (129, 384, 22016), (1000, 128, 12304)])
def test_rows_fp16_wide_blocks(ti, oracle, ws, M, K, N):
    """fp16 outputs wide enough for 128 x 192 blocks: ragged last rows and columns."""
    test_rows_store(ti, oracle, ws, 16, M, K, N)


@pytest.mark.parametrize("bits", [4, 8, 16, 4 | G32])
@pytest.mark.parametrize("M", [6, 17, 33, 64])
def test_rows_fold_range(ti, oracle, ws, bits, M):
    """Rows whose h * w fp16 does not hold: past 65504 in a few columns or in all, or all of it in the subnormal steps.
    Their sums are negative, and the consumer normalises them first.  Bound: fp16 inputs, half a unit in
    the last place of every x (2^-11, or 2^-25 below the normal range), beside the fp32 sums."""
    L, K, H, N = ti.lib(), 256, 1024, 208
    rng = np.random.RandomState(M + bits)
    to, so, wo = weight(ti, oracle, bits, K, H, rng)
    t2, s2, w2 = weight(ti, oracle, bits, H, N, rng)
    act = rng.standard_normal((M, K)).astype(f16)
    h0 = rng.standard_normal((M, H)).astype(f32)
    nw = (1 + 0.1 * rng.standard_normal(H)).astype(f32)
    h0[1, [5, 700]] = 1e5, -3e5
    h0[M - 1] *= 1e6
    h0[2] *= 3e-7
    act[2] = 0
    h0[4], act[4] = 0, 0
    bad = np.isin(np.arange(M), [1, 2, 4, M - 1])
    ad, nwd = dev(ti, act), dev(ti, nw)
    for kernel, k in [(a, b) for a in kernels(ti, M, bits) for b in (ws, None)]:
        n_ss = L.ti_gemm_rows_fold_partials_on(kernel, bits, M, H, K, WS if k else 0)
        hd, fx, ss, yd = dev(ti, h0), ti.DeviceBuffer(M * H * 2), ti.DeviceBuffer(n_ss * 64 * 4), ti.DeviceBuffer(M * N * 4)
        out = []
        for _ in range(2):   # (the second call over rows that the first rewrote)
            ti.check(L.ti_memcpy_h2d(hd.ptr, h0.ctypes.data_as(C.c_void_p), h0.nbytes, None))
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out = ti.EPI_RESID_F32, H, hd.ptr
            ep.fold_w, ep.fold_x, ep.fold_ss = nwd.ptr, fx.ptr, ss.ptr
            rows(ti, bits, to, so, ad, M, H, K, ep, ws=k, kernel=kernel)
            np.testing.assert_array_equal(np.signbit(ss.download(f32, (n_ss, 64))[:, :M]).any(axis=0), bad)
            h1 = hd.download(f32, (M, H)).astype(np.float64)
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out, ep.ss_in, ep.n_ss = ti.EPI_STORE_F32, N, yd.ptr, ss.ptr, n_ss
            rows(ti, bits, t2, s2, fx, M, N, H, ep, ws=k, kernel=kernel, h=hd.ptr, norm_w=nwd.ptr)
            out.append(yd.download(f32, (M, N)))
        x = h1 / np.sqrt((h1**2).mean(axis=1) + 1e-5)[:, None] * nw
        err = np.abs(out[0] - x @ w2.astype(np.float64))
        assert np.all(err <= (2.0**-11 + H * 2.0**-24) * (np.abs(x) @ np.abs(w2)) + 2.0**-25 * np.abs(w2).sum(axis=0) + 1e-9)
        np.testing.assert_array_equal(*out)


@pytest.mark.parametrize("bits", [4, 8, 16, 4 | G32])
@pytest.mark.parametrize("M", [7, 24, 40, 64])
def test_rows_fold_small_columns(ti, oracle, ws, bits, M):
    """Small columns of a row are taken as they are unless most of the row is small, however wide the blocks that carry the marks
    are.  Bound: fp16 inputs, half a unit in the last place of every h w (2^-11, or 2^-25 below the normal range, over the rms)
    beside the fp32 sums; rows normalised first as in test_rows_fold_range."""
    L, K, H, N = ti.lib(), 256, 1024, 208
    rng = np.random.RandomState(M + bits)
    to, so, wo = weight(ti, oracle, bits, K, H, rng)
    t2, s2, w2 = weight(ti, oracle, bits, H, N, rng)
    act = np.zeros((M, K), f16)
    h = rng.standard_normal((M, H)).astype(f32)
    nw = (1 + 0.1 * rng.standard_normal(H)).astype(f32)
    h[1, 32:48] *= 1e-6    # a weight tile's columns
    h[2, 128:192] *= 1e-6
    h[3, :448] *= 1e-6     # nearly half
    h[4] *= 5e-4           # (all of it not far above 2^-11.5, nearly every h w below 2^-10)
    h[5, 64:] *= 1e-6
    h[M - 1] *= 2e-4
    first = np.isin(np.arange(M), [5, M - 1])
    plain = (h * nw).astype(f16).view(np.uint16)
    rms = np.sqrt((h.astype(np.float64) ** 2).mean(axis=1) + 1e-5)[:, None]
    x = h.astype(np.float64) / rms * nw
    step = 2.0**-25 / np.where(first[:, None], 1.0, rms)
    tol = (2.0**-11 + H * 2.0**-24) * (np.abs(x) @ np.abs(w2)) + step * np.abs(w2).sum(axis=0) + 1e-9
    ad, nwd = dev(ti, act), dev(ti, nw)
    for kernel in kernels(ti, M, bits):
        n_ss = L.ti_gemm_rows_fold_partials_on(kernel, bits, M, H, K, WS)
        hd, fx, ss, yd = dev(ti, h), ti.DeviceBuffer(M * H * 2), ti.DeviceBuffer(n_ss * 64 * 4), ti.DeviceBuffer(M * N * 4)
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = ti.EPI_RESID_F32, H, hd.ptr
        ep.fold_w, ep.fold_x, ep.fold_ss = nwd.ptr, fx.ptr, ss.ptr
        rows(ti, bits, to, so, ad, M, H, K, ep, ws=ws, kernel=kernel)
        np.testing.assert_allclose(np.abs(ss.download(f32, (n_ss, 64))[:, :M]).sum(axis=0), (h.astype(np.float64) ** 2).sum(axis=1), rtol=1e-5)
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out, ep.ss_in, ep.n_ss = ti.EPI_STORE_F32, N, yd.ptr, ss.ptr, n_ss
        rows(ti, bits, t2, s2, fx, M, N, H, ep, ws=ws, kernel=kernel, h=hd.ptr, norm_w=nwd.ptr)
        np.testing.assert_array_equal((fx.download(np.uint16, (M, H)) != plain).any(axis=1), first)
        assert np.all(np.abs(yd.download(f32, (M, N)) - x @ w2.astype(np.float64)) <= tol)


@pytest.mark.parametrize("bits", [4, 8, 16, 4 | G32, 8 | G32])
def test_step_with_large_residuals(ti, bits):
    """An embedding whose product with the norm weight passes fp16's range, or lies in its subnormal steps: steps of 9 streams and
    prompts with the norms folded against the same with the fold off (ti_rmsnorm_f16 in front of every product).  Both round
    the same fp16 inputs: 1e-2 of the largest logit."""
    V, H, layers, heads, kv, hd, inter = 512, 256, 2, 4, 2, 64, 512
    e = ti.Engine(V, H, layers, heads, kv, hd, inter, bits=bits, max_seq=96, max_batch=9)
    rng = np.random.RandomState(bits)
    if bits & G32:
        for i in range(layers + 1):
            for slot, K, N in [(ti.W_Q, H, heads * hd), (ti.W_K, H, kv * hd), (ti.W_V, H, kv * hd), (ti.W_O, heads * hd, H), (ti.W_GATE, H, inter),
                               (ti.W_UP, H, inter), (ti.W_DOWN, inter, H)] if i < layers else [(ti.W_LM_HEAD, H, V)]:
                q, d, _ = g32_weight(rng, K, N, bits & 15)
                e.set_tensor_q(slot, i % layers if i < layers else 0, q, d)
    else:
        e.synth(5, 0.1)
    emb = (0.02 * rng.standard_normal((V, H))).astype(f32)
    emb[::3, 7] = 6e4
    emb[1::3] *= 5e-5
    e.set_tensor(ti.E_EMBED, 0, emb)
    for slot, i in [(ti.V_ATTN_NORM, 0), (ti.V_ATTN_NORM, 1), (ti.V_FFN_NORM, 0), (ti.V_FFN_NORM, 1), (ti.V_OUT_NORM, 0)]:
        nw = rng.uniform(0.7, 1.3, H).astype(f32)   # (each its own)
        nw[7] = 2
        e.set_tensor(slot, i, nw)
    tok = rng.randint(0, V, (3, 9)).astype(np.int32)
    tok[0] = np.arange(9)
    prompts = [rng.randint(0, V, n).astype(np.int32) for n in (3, 17, 48, 64)]
    out = []
    for on in (True, False):
        e.set_fold(on)
        out.append([e.step(t, np.full(9, i, np.int32)) for i, t in enumerate(tok)] +
                   [e.prefill(1, p, want=[0, p.size // 2, p.size - 1]) for p in prompts])
    e.close()
    for got, ref in zip(*out):
        assert np.isfinite(got).all() and np.isfinite(ref).all()
        assert np.abs(got - ref).max() <= 1e-2 * np.abs(ref).max(), (np.abs(got - ref).max(axis=1), np.abs(ref).max())


# the block kernel (gemm_block.hip): the fewest rows, the last block of rows by one row, one group of k (waves without one of their
# own), 2, 3, 5, 7, 9, 11, 17, 23 and 24 of them (its ring of 2 or 3 slots and the last stages, of up to 4 groups), a last block of
# columns of 1 .. 15 tiles, most block shapes as the call itself would take them; the outputs it writes, rows of a pitch of their own, with fp16 rows of one where 16-byte pieces are not aligned
@pytest.mark.parametrize("M,K,N", [(65, 128, 16), (97, 384, 1040), (129, 256, 4112), (500, 2176, 2064), (97, 896, 16400), (257, 640, 12304),
                                   (512, 640, 12304), (577, 640, 16400), (1024, 1408, 2576), (97, 3072, 8208), (161, 3072, 11280),
                                   (65, 1152, 400), (66, 384, 3088), (70, 2944, 3088), (97, 2944, 4112)])
@pytest.mark.parametrize("bits", [4, 8, 16])
def test_rows_block(ti, oracle, bits, M, K, N):
    rng = np.random.RandomState(M * 3 + K + N + bits)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    ldx, ldo = K + 8 * (M % 3), N + 4
    x = rng.standard_normal((M, ldx)).astype(f16)
    xd, xa = dev(ti, x), x[:, :K].astype(f32)
    ref = xa.astype(np.float64) @ w.astype(np.float64)

    def run(kind, out):
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = kind, ldo, out.ptr
        rows(ti, bits, td, sd, xd, M, N, K, ep, ldx, kernel=ti.ROWS_BLOCK)

    r = rng.standard_normal((M + 1, ldo)).astype(f32)
    yd, rd, hd = ti.DeviceBuffer(r.nbytes), dev(ti, r), ti.DeviceBuffer(r.nbytes // 2)
    yd.zero()
    hd.zero()
    run(ti.EPI_STORE_F32, yd)
    run(ti.EPI_RESID_F32, rd)
    run(ti.EPI_SILU_MUL_F16, hd)
    y, h = yd.download(f32, r.shape), hd.download(f16, r.shape)
    assert_close_dot(y[:M, :N], ref, xa, w)
    assert not y[M].any() and not y[:, N:].any()
    np.testing.assert_array_equal(rd.download(f32, r.shape), r + y)   # one addition to the same sums
    g = y[:M, :N].astype(np.float64).reshape(M, N // 16, 2, 8)
    sil = (g[:, :, 1] * (g[:, :, 0] / (1 + np.exp(-g[:, :, 0])))).reshape(M, N // 2)
    # (fp32 arithmetic of ~ 1e-6 and fp16's rounding, 2^-11)
    np.testing.assert_allclose(h[:M, : N // 2].astype(np.float64), sil, rtol=2.0 ** -11 + 1e-5, atol=2.0 ** -25)
    assert not h[M].any() and not h[:, N // 2:].any()


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("hd,M", [(16, 65), (48, 200), (128, 130)])
def test_rows_block_qkv(ti, oracle, bits, hd, M):
    """Queries, keys and values of a prompt chunk: the many-rows kernel's on the same rows, to the order of the sums; streams of
    their own where the rows belong to several."""
    heads, kvh, K, S = 6, 2, 640, 256
    qd, kd = heads * hd, kvh * hd
    N, rng = qd + 2 * kd, np.random.RandomState(hd + bits)
    td, sd, _ = weight(ti, oracle, bits, K, N, rng)
    xd, pd = dev(ti, rng.standard_normal((M, K)).astype(f16)), dev(ti, rng.permutation(S)[:M].astype(np.int32))
    cs = dev(ti, ti.rope_table(np.arange(S), hd, 10000.0))
    stride = kvh * S * hd if M < 100 else 0
    outs = []
    for kernel in (ti.ROWS_MANY, ti.ROWS_BLOCK):
        n = kvh * S * hd * (M if stride else 1)
        q, k, v = ti.DeviceBuffer(M * qd * 4), ti.DeviceBuffer(n * 2), ti.DeviceBuffer(n * 2)
        for b in (k, v):
            b.zero()
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out, ep.q_dim, ep.kv_dim, ep.head_dim, ep.max_seq = ti.EPI_QKV_ROPE_KV, qd, q.ptr, qd, kd, hd, S
        ep.pos, ep.rope_cs, ep.k_cache, ep.v_cache, ep.kv_stream_stride = pd.ptr, cs.ptr, k.ptr, v.ptr, stride
        rows(ti, bits, td, sd, xd, M, N, K, ep, kernel=kernel)
        outs.append([q.download(f32, (M, qd)), k.download(f16, (n,)).astype(f32), v.download(f16, (n,)).astype(f32)])
    # (sums of 640 products of ~ 0.03: their fp32 rounding in either order is below 1e-5; fp16 rows may round apart by a step)
    np.testing.assert_allclose(outs[0][0], outs[1][0], rtol=1e-5, atol=1e-5)
    for a, b in zip(outs[0][1:], outs[1][1:]):
        np.testing.assert_allclose(a, b, rtol=2.0 ** -10, atol=1e-5)


# the few-rows kernel's blocks of 3 and 6 tiles, and of 2 at 48 rows (other formats of a size: of 3), a last block short by 1 .. 5
@pytest.mark.parametrize("M,K,N", [(16, 384, 11296), (13, 2176, 12336), (5, 896, 22064), (31, 1152, 11296), (32, 384, 16432), (47, 2176, 5648)])
@pytest.mark.parametrize("bits", [4, 8, 4 | G32, 8 | G32])
def test_rows_few_wide_blocks(ti, oracle, bits, M, K, N):
    """A folded input into the residual with a folded output."""
    rng = np.random.RandomState(M + K + N + bits)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    h, r = rng.standard_normal((M, K)).astype(f32), rng.standard_normal((M + 1, N)).astype(f32)
    nw, ow = (1 + 0.1 * rng.standard_normal(K)).astype(f32), (1 + 0.1 * rng.standard_normal(N)).astype(f32)
    x, sq = (h * nw).astype(f16), np.zeros((1, 64), f32)
    sq[0, :M] = (h.astype(np.float64) ** 2).sum(axis=1)
    xd, sqd, rd, owd, fx = dev(ti, x), dev(ti, sq), dev(ti, r), dev(ti, ow), ti.DeviceBuffer(M * N * 2)
    n_ss = ti.lib().ti_gemm_rows_fold_partials_on(ti.ROWS_FEW, bits, M, N, K, 0)
    assert n_ss < N // 16   # (blocks of more than a tile)
    ss = ti.DeviceBuffer(n_ss * 64 * 4)
    ep = ti.Epilogue()
    ep.kind, ep.ldo, ep.out, ep.ss_in, ep.n_ss = ti.EPI_RESID_F32, N, rd.ptr, sqd.ptr, 1
    ep.fold_w, ep.fold_x, ep.fold_ss = owd.ptr, fx.ptr, ss.ptr
    rows(ti, bits, td, sd, xd, M, N, K, ep, kernel=ti.ROWS_FEW)
    got = rd.download(f32, (M + 1, N))
    xf = x.astype(np.float64) / np.sqrt(sq[0, :M, None].astype(np.float64) / K + 1e-5)
    assert_close_dot(got[:M] - r[:M], xf @ w.astype(np.float64), xf.astype(f32), w, rel=5e-5)
    np.testing.assert_array_equal(got[M], r[M])
    np.testing.assert_array_equal(fx.download(np.uint16, (M, N)), (got[:M] * ow).astype(f16).view(np.uint16))
    np.testing.assert_allclose(ss.download(f32, (n_ss, 64))[:, :M].sum(axis=0), (got[:M].astype(np.float64) ** 2).sum(axis=1), rtol=1e-5)


# (block kernel: one and two row blocks of 32, the last one by a row, one of 64; 1, 2 and 4 groups of waves)
@pytest.mark.parametrize("M,K,H,N", [(33, 384, 1152, 80), (40, 256, 1024, 4112), (33, 1152, 2048, 400), (50, 640, 22016, 2064),
                                     (64, 2944, 4096, 12304), (64, 512, 12288, 208), (48, 384, 2944, 28688), (17, 1152, 2048, 4112), (32, 384, 1024, 28688)])
@pytest.mark.parametrize("bits", [4, 8, 16])
def test_rows_block_fold(ti, oracle, ws, bits, M, K, H, N):
    """Folds of up to 64 rows on the block kernel, into it and into the many-rows one, with rows that must be normalised first in its
    first and last block.  Bounds: test_rows_fold_range's."""
    L, rng = ti.lib(), np.random.RandomState(M + bits)
    if bits == 16 and M <= 32:
        assert L.ti_gemm_rows_fold_partials_on(ti.ROWS_BLOCK, bits, M, H, K, WS) == 0
        return
    to, so, wo = weight(ti, oracle, bits, K, H, rng)
    t2, s2, w2 = weight(ti, oracle, bits, H, N, rng)
    act = rng.standard_normal((M, K)).astype(f16)
    h0 = rng.standard_normal((M, H)).astype(f32)
    nw = (1 + 0.1 * rng.standard_normal(H)).astype(f32)
    nwd = dev(ti, nw)
    for marked in (False, True):
        if marked:
            h0[1, [5, 600]] = 1e5, -3e5
            h0[M - 1] *= 1e6
            h0[2] *= 3e-7
            act[2] = 0
        bad = np.isin(np.arange(M), [1, 2, M - 1]) & marked
        ad = dev(ti, act)
        n_ss = L.ti_gemm_rows_fold_partials_on(ti.ROWS_BLOCK, bits, M, H, K, WS)
        hd, fx, ss, yd = dev(ti, h0), ti.DeviceBuffer(M * H * 2), ti.DeviceBuffer(n_ss * 64 * 4), ti.DeviceBuffer(M * N * 4)
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = ti.EPI_RESID_F32, H, hd.ptr
        ep.fold_w, ep.fold_x, ep.fold_ss = nwd.ptr, fx.ptr, ss.ptr
        rows(ti, bits, to, so, ad, M, H, K, ep, ws=ws, kernel=ti.ROWS_BLOCK)
        h1 = hd.download(f32, (M, H))
        assert_close_dot(h1[~bad] - h0[~bad], act[~bad].astype(np.float64) @ wo.astype(np.float64), act[~bad].astype(f32), wo, rel=5e-5)
        sums, plain = ss.download(f32, (n_ss, 64))[:, :M], fx.download(np.uint16, (M, H))
        np.testing.assert_allclose(np.abs(sums).sum(axis=0), (h1.astype(np.float64) ** 2).sum(axis=1), rtol=1e-5)
        np.testing.assert_array_equal(np.signbit(sums).any(axis=0), bad)
        with np.errstate(over="ignore"):
            np.testing.assert_array_equal(plain, (h1 * nw).astype(f16).view(np.uint16))
        x = h1 / np.sqrt((h1.astype(np.float64) ** 2).mean(axis=1) + 1e-5)[:, None] * nw
        ref, tol = x @ w2, (2.0**-11 + H * 2.0**-24) * (np.abs(x) @ np.abs(w2)) + 2.0**-25 * np.abs(w2).sum(axis=0) + 1e-9
        for second in (ti.ROWS_MANY, ti.ROWS_BLOCK):
            out = []
            for _ in range(2):   # (the second call over rows that the first rewrote)
                ep = ti.Epilogue()
                ep.kind, ep.ldo, ep.out, ep.ss_in, ep.n_ss = ti.EPI_STORE_F32, N, yd.ptr, ss.ptr, n_ss
                rows(ti, bits, t2, s2, fx, M, N, H, ep, ws=ws, kernel=second, h=hd.ptr, norm_w=nwd.ptr)
                out.append(yd.download(f32, (M, N)))
            assert np.all(np.abs(out[0] - ref) <= tol), (marked, second)
            np.testing.assert_array_equal(*out)
        np.testing.assert_array_equal((fx.download(np.uint16, (M, H)) != plain).any(axis=1), bad)


@pytest.mark.parametrize("bits", [4, 8, 16])
@pytest.mark.parametrize("M,K,N", [(33, 640, 4112), (48, 384, 1040), (64, 1152, 12304)])
def test_rows_fold_divides(ti, oracle, bits, M, K, N):
    """A folded input's outputs are the plain ones divided by the row's rms, rounded once: the product with a rounded 1 / rms misses
    that in a fourth of the values, a quotient corrected by its remainder in next to none."""
    rng = np.random.RandomState(M + K + bits)
    td, sd, _ = weight(ti, oracle, bits, K, N, rng)
    h = rng.standard_normal((M, K)).astype(f32) * rng.uniform(0.3, 3, (M, 1)).astype(f32)
    sq = np.zeros((1, 64), f32)
    sq[0, :M] = (h.astype(np.float64) ** 2).sum(axis=1)
    xd, sqd, yd = dev(ti, h.astype(f16)), dev(ti, sq), ti.DeviceBuffer(M * N * 4)
    rms = np.sqrt(sq[0, :M] / f32(K) + f32(1e-5))[:, None]
    for kernel in (ti.ROWS_MANY, ti.ROWS_BLOCK) + ((ti.ROWS_FEW,) if M <= 48 else ()):
        out = []
        for fold in (False, True):
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out = ti.EPI_STORE_F32, N, yd.ptr
            if fold:
                ep.ss_in, ep.n_ss = sqd.ptr, 1
            rows(ti, bits, td, sd, xd, M, N, K, ep, kernel=kernel)
            out.append(yd.download(f32, (M, N)))
        ref = out[0] / rms
        assert (out[1] != ref).mean() < 1e-4, (kernel, (out[1] != ref).mean())
        np.testing.assert_allclose(out[1], ref, rtol=2.0 ** -23)


@pytest.mark.parametrize("bits", [4, 8, 16, 8 | G32])
@pytest.mark.parametrize("M,N", [(3, 48), (17, 4112), (48, 1040), (50, 400), (130, 2064)])
def test_rows_logits_keys(ti, oracle, bits, M, N):
    """Logits in 16-byte pieces and, at a pitch that is none, one by one: the plain product's values, and each row's key at the first
    of its largest columns where several are equal (columns of the same weights)."""
    K, rng = 512, np.random.RandomState(M + N + bits)
    w = np.tile(rng.standard_normal((K, 16)).astype(f32) * 0.03, (1, N // 16))
    if bits & G32:
        q, d, _ = g32_weight(rng, K, 16, bits & 15)
        td, sd = pack_g32(ti, np.tile(q, (1, N // 16)), np.tile(d, (1, N // 16)), bits & 15)
    else:
        td, sd = (dev(ti, a) for a in ti.wpack_host(w, bits))
    x = rng.standard_normal((M, K)).astype(f16)
    xd, yd = dev(ti, x), ti.DeviceBuffer(M * N * 4)
    for kernel in kernels(ti, M, bits, False):
        ep = ti.Epilogue()
        ep.kind, ep.ldo, ep.out = ti.EPI_STORE_F32, N, yd.ptr
        rows(ti, bits, td, sd, xd, M, N, K, ep, kernel=ti.ROWS_MANY if M > 48 else kernel)
        ref = yd.download(f32, (M, N))
        for ldo in (N, N + 4, N + 1):
            ld, am = ti.DeviceBuffer(M * ldo * 4), ti.DeviceBuffer(M * ti.ARGMAX_SLOTS * 8)
            ld.zero()
            am.zero()
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out, ep.argmax = ti.EPI_LOGITS_ARGMAX, ldo, ld.ptr, am.ptr
            rows(ti, bits, td, sd, xd, M, N, K, ep, kernel=kernel)
            lg = ld.download(f32, (M, ldo))
            np.testing.assert_array_equal(lg[:, :N], ref)
            assert not lg[:, N:].any()
            keys = am.download(np.uint64, (M, ti.ARGMAX_SLOTS)).max(axis=1)
            np.testing.assert_array_equal((0xFFFFFFFF - (keys & 0xFFFFFFFF)).astype(np.int64), np.argmax(lg[:, :N], axis=1))


# (kernel, format): how many block shapes it has
SHAPES = {("FEW", 4): 11, ("FEW", 8): 8, ("FEW", 16): 4, ("FEW", 36): 8, ("FEW", 40): 8, ("MANY", 4): 5, ("MANY", 8): 5, ("MANY", 16): 5, ("MANY", 36): 5,
          ("MANY", 40): 5, ("BLOCK", 4): 9, ("BLOCK", 8): 12, ("BLOCK", 16): 8}
FEW_ROWS = {4: [16] * 5 + [32] * 4 + [48] * 2, 16: [16, 16, 32, 48]}
EACH = [(k, b, i) for (k, b), n in SHAPES.items() for i in range(n) if not (k == "MANY" and b & G32 and i == 0)]   # (no such block of 32)


def each_rows(kernel, bits, i):
    """Rows of a shape's calls: a ragged block, and several where it has them."""
    if kernel == "FEW":
        r = FEW_ROWS.get(bits, [16] * 3 + [32] * 3 + [48] * 2)[i]
        return (r - 3, r)
    return ((50, 161) if i < 3 else (29,) if i == 3 else (13,)) if kernel == "MANY" else (50, 161)


def qkv_ref(ti, y, pos, cs, heads, kvh, hd):
    """RoPE of the products y, as (q, k, v) rows in float64."""
    qd, kd, (M, _) = heads * hd, kvh * hd, y.shape
    c = cs.reshape(-1, hd // 2, 2)[pos].astype(np.float64)
    p = y[:, : qd + kd].astype(np.float64).reshape(M, heads + kvh, hd // 2, 2)
    co, si = c[:, None, :, 0], c[:, None, :, 1]
    r = np.stack([p[..., 0] * co - p[..., 1] * si, p[..., 1] * co + p[..., 0] * si], -1).reshape(M, qd + kd)
    return r[:, :qd], r[:, qd:], y[:, qd + kd :].astype(np.float64)


@pytest.mark.parametrize("kernel,bits,i", EACH)
def test_rows_each_shape(ti, oracle, ws, kernel, bits, i):
    """Every block shape of each kernel by name, each output it writes: ragged rows and columns, k-groups that its waves or slices
    do not share evenly; the many-rows kernel with and without its split.  The other outputs follow from the plain one's values (same
    sums), which are within fp32 summation order of the weights' exact ones."""
    K, heads, kvh, hd, S = 1152, 39, 17, 16, 256
    qd, kd = heads * hd, kvh * hd
    N = qd + 2 * kd   # (73 tiles: no shape's blocks end with them)
    rng = np.random.RandomState(7 * bits + i)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    cs = ti.rope_table(np.arange(S), hd, 10000.0)
    csd, on = dev(ti, cs), getattr(ti, "ROWS_" + kernel) + (i + 1) * ti.ROWS_SHAPE
    for M in each_rows(kernel, bits, i):
        x, pos, r = rng.standard_normal((M, K)).astype(f16), rng.permutation(S)[:M].astype(np.int32), rng.standard_normal((M + 1, N)).astype(f32)
        xd, pd = dev(ti, x), dev(ti, pos)
        ref = x.astype(np.float64) @ w.astype(np.float64)
        for k in (None, ws) if kernel == "MANY" else (None,):
            yd, rd, hd_ = ti.DeviceBuffer(r.nbytes), dev(ti, r), ti.DeviceBuffer(r.nbytes // 2)
            q, kc, vc = ti.DeviceBuffer(M * qd * 4), ti.DeviceBuffer(S * kd * 2), ti.DeviceBuffer(S * kd * 2)
            for b in (yd, hd_, kc, vc):
                b.zero()
            for kind, out, ldo in ((ti.EPI_STORE_F32, yd, N), (ti.EPI_RESID_F32, rd, N), (ti.EPI_SILU_MUL_F16, hd_, N), (ti.EPI_QKV_ROPE_KV, q, qd)):
                ep = ti.Epilogue()
                ep.kind, ep.ldo, ep.out = kind, ldo, out.ptr
                if kind == ti.EPI_QKV_ROPE_KV:
                    ep.q_dim, ep.kv_dim, ep.head_dim, ep.max_seq = qd, kd, hd, S
                    ep.pos, ep.rope_cs, ep.k_cache, ep.v_cache, ep.kv_stream_stride = pd.ptr, csd.ptr, kc.ptr, vc.ptr, 0
                rows(ti, bits, td, sd, xd, M, N, K, ep, ws=k, kernel=on)
            y = yd.download(f32, r.shape)
            assert_close_dot(y[:M], ref, x.astype(f32), w, rel=5e-5)
            assert not y[M].any()
            np.testing.assert_array_equal(rd.download(f32, r.shape), r + y)
            h = hd_.download(f16, r.shape)
            g = y[:M].astype(np.float64).reshape(M, N // 16, 2, 8)
            sil = (g[:, :, 1] * (g[:, :, 0] / (1 + np.exp(-g[:, :, 0])))).reshape(M, N // 2)
            np.testing.assert_allclose(h[:M, : N // 2].astype(np.float64), sil, rtol=2.0 ** -11 + 1e-5, atol=2.0 ** -25)
            assert not h[M].any() and not h[:, N // 2 :].any()
            # (two products and a sum of fp32, of values of ~ 1; fp16 caches)
            rq, rk, rv = qkv_ref(ti, y[:M], pos, cs, heads, kvh, hd)
            np.testing.assert_allclose(q.download(f32, (M, qd)), rq, rtol=1e-6, atol=1e-6)
            for buf, rr in ((kc, rk), (vc, rv)):
                got = buf.download(f16, (kvh, S, hd)).astype(np.float64)
                np.testing.assert_allclose(got[:, pos].transpose(1, 0, 2).reshape(M, kd), rr, rtol=2.0 ** -11 + 1e-5, atol=2e-6)
                assert not np.delete(got, pos, axis=1).any()


@pytest.mark.parametrize("kernel,bits,i", EACH)
def test_rows_each_shape_fold(ti, oracle, ws, kernel, bits, i):
    """The folds of every block shape that has them: queries, keys and values, SiLU and plain outputs of a folded input with and without
    rows that are normalised first, in the first and the last block, and the folded output.  Bounds: test_rows_fold_range's, and
    test_rows_block_fold's."""
    K, heads, kvh, hd, S = 640, 39, 17, 16, 64
    qd, kd = heads * hd, kvh * hd
    N, M = qd + 2 * kd, each_rows(kernel, bits, i)[0]
    on, L = getattr(ti, "ROWS_" + kernel) + (i + 1) * ti.ROWS_SHAPE, ti.lib()
    n_out = L.ti_gemm_rows_fold_partials_on(on, bits, M, N, K, 0)
    wide = {"MANY": lambda: bits == 16 and i < 2, "BLOCK": lambda: no_fold_shape(bits, i), "FEW": lambda: False}[kernel]()
    assert (n_out == 0) == wide
    if wide:
        return
    rng = np.random.RandomState(11 * bits + i)
    td, sd, w = weight(ti, oracle, bits, K, N, rng)
    w = w.astype(np.float64)
    cs = ti.rope_table(np.arange(S), hd, 10000.0)
    csd, pos = dev(ti, cs), rng.permutation(S)[:M].astype(np.int32)
    pd, nw = dev(ti, pos), (1 + 0.1 * rng.standard_normal(K)).astype(f32)
    nwd = dev(ti, nw)
    h = rng.standard_normal((M, K)).astype(f32)
    for marked in (False, True):
        sq = np.zeros((1, 64), f32)
        if marked:   # (past 65504: the sum negative, its lowest bit 0)
            h[1, [5, 600]] = 1e5, -3e5
            h[M - 1] *= 1e6
        sq[0, :M] = (h.astype(np.float64) ** 2).sum(axis=1)
        if marked:
            b = sq.view(np.uint32)
            b[0, [1, M - 1]] = (b[0, [1, M - 1]] & ~np.uint32(1)) | np.uint32(0x80000000)
        with np.errstate(over="ignore"):
            xd = dev(ti, (h * nw).astype(f16))
        hd_, sqd = dev(ti, h), dev(ti, sq)
        yd, od, q = ti.DeviceBuffer(M * N * 4), ti.DeviceBuffer(M * N * 2), ti.DeviceBuffer(M * qd * 4)
        kc, vc = ti.DeviceBuffer(M * S * kd * 2), ti.DeviceBuffer(M * S * kd * 2)
        kc.zero()
        vc.zero()
        for kind, out, ldo in ((ti.EPI_QKV_ROPE_KV, q, qd), (ti.EPI_SILU_MUL_F16, od, N), (ti.EPI_STORE_F32, yd, N)):
            ep = ti.Epilogue()
            ep.kind, ep.ldo, ep.out, ep.ss_in, ep.n_ss = kind, ldo, out.ptr, sqd.ptr, 1
            if kind == ti.EPI_QKV_ROPE_KV:   # (decode rows: a cache of its own for each)
                ep.q_dim, ep.kv_dim, ep.head_dim, ep.max_seq = qd, kd, hd, S
                ep.pos, ep.rope_cs, ep.k_cache, ep.v_cache, ep.kv_stream_stride = pd.ptr, csd.ptr, kc.ptr, vc.ptr, S * kd
            rows(ti, bits, td, sd, xd, M, N, K, ep, kernel=on, h=hd_.ptr, norm_w=nwd.ptr)
        x = h / np.sqrt((h.astype(np.float64) ** 2).mean(axis=1) + 1e-5)[:, None] * nw
        y = yd.download(f32, (M, N))
        tol = (2.0**-11 + K * 2.0**-24) * (np.abs(x) @ np.abs(w)) + 2.0**-25 * np.abs(w).sum(axis=0) + 1e-9
        assert np.all(np.abs(y - x @ w) <= tol), marked
        g = y.astype(np.float64).reshape(M, N // 16, 2, 8)   # (the other outputs from the same sums)
        sil = (g[:, :, 1] * (g[:, :, 0] / (1 + np.exp(-g[:, :, 0])))).reshape(M, N // 2)
        np.testing.assert_allclose(od.download(f16, (M, N))[:, : N // 2].astype(np.float64), sil, rtol=2.0 ** -11 + 1e-5, atol=2.0 ** -25)
        rq, rk, rv = qkv_ref(ti, y, pos, cs, heads, kvh, hd)
        np.testing.assert_allclose(q.download(f32, (M, qd)), rq, rtol=1e-6, atol=1e-6)
        for buf, rr in ((kc, rk), (vc, rv)):
            got = buf.download(f16, (M, kvh, S, hd)).astype(np.float64)
            np.testing.assert_allclose(got[np.arange(M), :, pos].reshape(M, kd), rr, rtol=2.0 ** -11 + 1e-5, atol=2e-6)
            got[np.arange(M), :, pos] = 0
            assert not got.any()
    act, r, ow = rng.standard_normal((M, K)).astype(f16), rng.standard_normal((M + 1, N)).astype(f32), (1 + 0.1 * rng.standard_normal(N)).astype(f32)
    ad, rd, owd, fx, ss = dev(ti, act), dev(ti, r), dev(ti, ow), ti.DeviceBuffer(M * N * 2), ti.DeviceBuffer(n_out * 64 * 4)
    ep = ti.Epilogue()
    ep.kind, ep.ldo, ep.out = ti.EPI_RESID_F32, N, rd.ptr
    ep.fold_w, ep.fold_x, ep.fold_ss = owd.ptr, fx.ptr, ss.ptr
    rows(ti, bits, td, sd, ad, M, N, K, ep, kernel=on)
    got = rd.download(f32, (M + 1, N))
    assert_close_dot(got[:M] - r[:M], act.astype(np.float64) @ w, act.astype(f32), w, rel=5e-5)
    np.testing.assert_array_equal(got[M], r[M])
    np.testing.assert_array_equal(fx.download(np.uint16, (M, N)), (got[:M] * ow).astype(f16).view(np.uint16))
    np.testing.assert_allclose(ss.download(f32, (n_out, 64))[:, :M].sum(axis=0), (got[:M].astype(np.float64) ** 2).sum(axis=1), rtol=1e-5)


def no_fold_shape(bits, i):
    """The block kernel's shapes of more than 64 rows, and int4's 64 x 256, have no folds."""
    return i in {4: (0, 1, 2), 8: (0, 1, 2, 3), 16: (0, 1, 2, 3)}[bits]
