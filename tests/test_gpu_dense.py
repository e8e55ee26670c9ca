"""Large tiles of the layer-stack products (ti_dense, dense_block_kernel) against float64: the tiles that the dispatch picks
(ti_dense_tile), ragged rows and columns, short k, the epilogues that run on them, grouped tiles whose experts hold from 1
row to a whole tile.  Bound: K roundings of 2^-24 of the sum of magnitudes (fp32 accumulation), and half a unit in the last
place of the stored type."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(M, N, K, dtype, batch=1, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn(M, K, device="cuda", generator=g).to(dtype)
    w = (torch.randn(batch, -(-N // 16) * 16, K, device="cuda", generator=g) * 0.05).to(dtype)
    vec = 8 if dtype == torch.bfloat16 else 4
    # fragment order: [column tile][k-tile][lane][vec], lane l: column l & 15, k from vec * (l >> 4)
    f = w.view(batch, -1, 16, K // (4 * vec), 4, vec).permute(0, 1, 3, 4, 2, 5).contiguous()
    return a, w[:, :N], f


def call(ti, d):
    torch.cuda.synchronize()
    ti.check(ti.lib().ti_dense(C.byref(d), None))
    ti.sync()


def check(got, a, w, dtype, out16=False):
    ref = a.double() @ w.double().T
    tol = a.shape[1] * 2.0**-24 * (a.double().abs() @ w.double().abs().T) + (2.0**-8 if out16 else 2.0**-23) * ref.abs()
    assert (got.double() - ref).abs().le(tol).all()


def tile(ti, d):
    rows, cols = C.c_int(0), C.c_int(0)
    ti.check(ti.lib().ti_dense_tile(C.byref(d), C.byref(rows), C.byref(cols)))
    return rows.value, cols.value


BLOCKS = [   # a tile's shape, and a call that runs on it: last rows and columns ragged
    ((256, 256), 1100, 8712, 2048, torch.bfloat16),   # last row tile 76 rows, last columns 8
    ((256, 256), 1281, 8193, 2048, torch.bfloat16),   # .. 1 row, 1 column
    ((128, 256), 700, 8708, 2048, torch.bfloat16),
    ((128, 128), 1100, 2051, 8192, torch.bfloat16),
    ((128, 128), 1100, 2051, 8256, torch.bfloat16),
    ((256, 256), 1601, 8705, 2048, torch.float32),
    ((128, 256), 2000, 4008, 512, torch.float32),
]


@pytest.mark.parametrize("shape,M,N,K,dtype", BLOCKS)
def test_blocks(ti, shape, M, N, K, dtype):
    a, w, f = operands(M, N, K, dtype)
    ldo = N + 5
    out = torch.full((M + 1, ldo), 7.0, device="cuda")
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=ldo, M=M, N=N, K=K, batch=1, epi=ti.DE_F32,
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    assert tile(ti, d) == shape
    call(ti, d)
    check(out[:M, :N], a, w[0], dtype)
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()


def swiglu(y):   # even columns gate, odd ones up
    g, u = y[:, 0::2], y[:, 1::2]
    return g * torch.sigmoid(g) * u


def check_swiglu(got, a, w, dtype):
    """|d silu| <= 1.1, so an output moves by the roundings of its two products, each times the other's size; and half a
    unit in the last place of the stored type."""
    y, mag = a.double() @ w.double().T, a.shape[1] * 2.0**-24 * (a.double().abs() @ w.double().abs().T)
    ref = swiglu(y)
    tol = 1.1 * mag[:, 0::2] * y[:, 1::2].abs() + mag[:, 1::2] * y[:, 0::2].abs() + (2.0**-8 if dtype == torch.bfloat16 else 2.0**-20) * ref.abs()
    assert (got.double() - ref).abs().le(tol + 1e-9).all()


@pytest.mark.parametrize("shape,M,N,K,dtype", [(s, m, n + n % 2, k, t) for s, m, n, k, t in BLOCKS])
def test_swiglu_blocks(ti, shape, M, N, K, dtype):
    a, w, f = operands(M, N, K, dtype)
    out = torch.full((M + 1, N // 2), 7.0, device="cuda").to(dtype)
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N // 2, M=M, N=N, K=K, batch=1, epi=ti.DE_SWIGLU,
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    assert tile(ti, d) == shape
    call(ti, d)
    check_swiglu(out[:M], a, w[0], dtype)
    assert (out[M] == 7).all()


@pytest.mark.parametrize("shape,M,N,K,dtype", [(s, m, (n + 31) // 32 * 32, k, t) for s, m, n, k, t in BLOCKS])
def test_rotary_blocks(ti, shape, M, N, K, dtype):
    """Rotary pairs of the last 16 of a head's 32 columns; bound: the pair's roundings of both products."""
    a, w, f = operands(M, N, K, dtype)
    pos = torch.randperm(M, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)).int()
    ang = torch.arange(M, device="cuda")[:, None].double() * 100.0 ** (-torch.arange(8, device="cuda").double() / 8)
    cs = torch.stack([ang.cos(), ang.sin()], -1).float().contiguous()
    out = torch.full((M + 1, N), 7.0, device="cuda").to(dtype)
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N, M=M, N=N, K=K, batch=1, epi=ti.DE_ROPE, head_w=32,
                     rot_off=16, rope_cs=cs.data_ptr(), pos=pos.data_ptr(), dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    assert tile(ti, d) == shape
    call(ti, d)
    y, mag = a.double() @ w[0].double().T, K * 2.0**-24 * (a.double().abs() @ w[0].double().abs().T)
    y, mag = y.view(M, -1, 32), mag.view(M, -1, 32)
    c, s = (cs[pos.long()].double()[:, None, :, i] for i in (0, 1))
    e, o = y[..., 16::2], y[..., 17::2]
    ref, tol = y.clone(), mag.clone()
    ref[..., 16::2], ref[..., 17::2] = e * c - o * s, o * c + e * s
    tol[..., 16:] = (mag[..., 16::2] + mag[..., 17::2]).repeat_interleave(2, -1) + 2.0**-22 * (e.abs() + o.abs()).repeat_interleave(2, -1)
    err = (out[:M].double().view(M, -1, 32) - ref).abs()
    assert err.le(tol + (2.0**-8 if dtype == torch.bfloat16 else 2.0**-23) * ref.abs()).all()
    assert (out[M] == 7).all()


@pytest.mark.parametrize("shape,M,N,K", [((256, 256), 1100, 8640, 2048), ((128, 256), 700, 8640, 2048), ((128, 128), 1100, 2112, 8192)])
@pytest.mark.parametrize("head_w,rot_off", [(192, 128), (96, 64), (32, 16), (64, 0)])
@pytest.mark.parametrize("pad", [0, 4])
def test_rotary_heads(ti, shape, M, N, K, head_w, rot_off, pad):
    """Pieces of 64 columns without a rotated part, all of it, both, and of two heads; rows that 16 bytes fit, and not.  A column in front of the
    rotated part is infinite: its neighbours are what they are without it.  Bound as above."""
    N = N // head_w * head_w
    a, w, _ = operands(M, N, K, torch.bfloat16)
    inf = head_w + 5
    a[:, 0] = 1.0
    w = torch.cat([w[0], w.new_zeros(-N % 16, K)])
    if rot_off:
        w[inf, 0] = float("inf")
    f = w.view(-1, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()
    pairs, ldo = (head_w - rot_off) // 2, N + pad
    pos = torch.randperm(M, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2)).int()
    ang = torch.arange(M, device="cuda")[:, None].double() * 100.0 ** (-torch.arange(pairs, device="cuda").double() / pairs)
    cs = torch.stack([ang.cos(), ang.sin()], -1).float().contiguous()
    out = torch.full((M + 1, ldo), 7.0, device="cuda").bfloat16()
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=ldo, M=M, N=N, K=K, batch=1, epi=ti.DE_ROPE, head_w=head_w,
                     rot_off=rot_off, rope_cs=cs.data_ptr(), pos=pos.data_ptr(), dtype=ti.DT_BF16)
    assert tile(ti, d) == shape
    call(ti, d)
    if rot_off:
        w[inf, 0] = 0.0
    y, mag = a.double() @ w[:N].double().T, K * 2.0**-24 * (a.double().abs() @ w[:N].double().abs().T)
    y, mag = y.view(M, -1, head_w), mag.view(M, -1, head_w)
    c, s = (cs[pos.long()].double()[:, None, :, i] for i in (0, 1))
    e, o = y[..., rot_off::2], y[..., rot_off + 1 :: 2]
    ref, tol = y.clone(), mag.clone()
    ref[..., rot_off::2], ref[..., rot_off + 1 :: 2] = e * c - o * s, o * c + e * s
    tol[..., rot_off:] = (mag[..., rot_off::2] + mag[..., rot_off + 1 :: 2]).repeat_interleave(2, -1) + 2.0**-22 * (e.abs() + o.abs()).repeat_interleave(2, -1)
    got, ref, tol = out[:M, :N].double(), ref.reshape(M, N), tol.reshape(M, N)
    if rot_off:
        assert (got[:, inf] == float("inf")).all()
        got[:, inf] = ref[:, inf]
    assert (got - ref).abs().le(tol + 2.0**-8 * ref.abs()).all()
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tile_rows", [128, 256])
@pytest.mark.parametrize("N,K", [(48, 64), (264, 128), (512, 192), (250, 448)])
def test_grouped_tiles(ti, dtype, tile_rows, N, K):
    counts = [1, 16, 17, 0, 31, 64, 65, 96, 127, 128, 129, 192, 193, 255, 256, 257]
    E, M = len(counts), sum(counts)
    a, w, f = operands(M, N, K, dtype, E, 3)
    order = torch.randperm(M, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).int()
    tiles, first = [], 0
    for e, c in enumerate(counts):
        tiles += [(e, first + i, min(tile_rows, c - i), 0) for i in range(0, c, tile_rows)]
        first += c
    tl = torch.zeros(len(tiles) + 9, 4, dtype=torch.int32, device="cuda")
    tl[:len(tiles)] = torch.tensor(tiles, dtype=torch.int32)
    n = torch.tensor([len(tiles)], dtype=torch.int32, device="cuda")
    out = torch.full((M + 1, N), 7.0, device="cuda").to(dtype)
    d = ti.DenseArgs(w=f.data_ptr(), w_batch=f[0].numel(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N, M=M, N=N, K=K, batch=1,
                     epi=ti.DE_T, dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32, tile_rows=tile_rows,
                     max_tiles=len(tl), tiles=tl.data_ptr(), n_tiles=n.data_ptr(), rows_in=order.data_ptr(), rows_out=order.data_ptr(),
                     row_div=1)
    call(ti, d)
    first = 0
    for e, c in enumerate(counts):
        r = order[first:first + c].long()
        check(out[r], a[r], w[e], dtype, dtype == torch.bfloat16)
        first += c
    assert (out[M] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tile_rows", [128, 256])
@pytest.mark.parametrize("N,K", [(48, 64), (264, 128), (512, 192), (250, 448)])
def test_grouped_swiglu(ti, dtype, tile_rows, N, K):
    counts = [1, 16, 17, 0, 31, 64, 65, 96, 127, 128, 129, 192, 193, 255, 256, 257]
    E, M = len(counts), sum(counts)
    a, w, f = operands(M, N, K, dtype, E, 3)
    order = torch.randperm(M, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).int()
    tiles, first = [], 0
    for e, c in enumerate(counts):
        tiles += [(e, first + i, min(tile_rows, c - i), 0) for i in range(0, c, tile_rows)]
        first += c
    tl = torch.zeros(len(tiles) + 9, 4, dtype=torch.int32, device="cuda")
    tl[:len(tiles)] = torch.tensor(tiles, dtype=torch.int32)
    n = torch.tensor([len(tiles)], dtype=torch.int32, device="cuda")
    out = torch.full((M + 1, N // 2), 7.0, device="cuda").to(dtype)
    d = ti.DenseArgs(w=f.data_ptr(), w_batch=f[0].numel(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N // 2, M=M, N=N, K=K, batch=1,
                     epi=ti.DE_SWIGLU, dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32, tile_rows=tile_rows,
                     max_tiles=len(tl), tiles=tl.data_ptr(), n_tiles=n.data_ptr(), rows_in=order.data_ptr(), rows_out=order.data_ptr(),
                     row_div=1)
    call(ti, d)
    first = 0
    for e, c in enumerate(counts):
        r = order[first:first + c].long()
        check_swiglu(out[r], a[r], w[e], dtype)
        first += c
    assert (out[M] == 7).all()


@pytest.mark.parametrize("epi", ["T", "SWIGLU"])
@pytest.mark.parametrize("tiles_n,N,K", [(122, 1072, 192), (77, 1024, 256), (9, 520, 320), (3, 2048, 1408)])
def test_expert_rounds(ti, epi, tiles_n, N, K):
    """256-row tiles on workgroups that stay: from one block for some of them to four each, of every height, the last columns
    ragged (1072, 520) or whole, the shortest k that they take; a second call finds nothing of the first."""
    r = np.random.default_rng(tiles_n)
    rows = np.sort(np.r_[256, 1, r.integers(1, 257, tiles_n - 2)])[::-1]
    experts = 5
    a, w, f = operands(int(rows.sum()) // 2 + 1, N, K, torch.bfloat16, experts, 3)
    n_in = int(rows.sum())
    order = torch.randperm(n_in, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).int()
    first = np.r_[0, np.cumsum(rows)[:-1]]
    tl = torch.zeros(tiles_n + 9, 4, dtype=torch.int32, device="cuda")
    tl[:tiles_n] = torch.tensor([(i % experts, int(s), int(c), 0) for i, (s, c) in enumerate(zip(first, rows))], dtype=torch.int32)
    n = torch.tensor([tiles_n], dtype=torch.int32, device="cuda")
    cols = N // 2 if epi == "SWIGLU" else N
    for _ in range(2):
        out = torch.full((n_in + 1, cols), 7.0, device="cuda").bfloat16()
        d = ti.DenseArgs(w=f.data_ptr(), w_batch=f[0].numel(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=cols, M=len(a), N=N, K=K, batch=1,
                         epi=ti.DE_SWIGLU if epi == "SWIGLU" else ti.DE_T, dtype=ti.DT_BF16, tile_rows=256, max_tiles=len(tl), tiles=tl.data_ptr(),
                         n_tiles=n.data_ptr(), rows_in=order.data_ptr(), rows_out=order.data_ptr(), row_div=2)
        call(ti, d)
        for i in range(tiles_n):
            at = order[int(first[i]) : int(first[i] + rows[i])].long()
            if epi == "SWIGLU":
                check_swiglu(out[at], a[at // 2], w[i % experts], torch.bfloat16)
            else:
                check(out[at], a[at // 2], w[i % experts], torch.bfloat16, True)
        assert (out[n_in] == 7).all()


@pytest.mark.parametrize("M,N,K,act_cols,t_cols,ldo", [
    (1100, 8712, 2048, 4356, 8648, 8656),   # 256 x 256 blocks; an activation and fp32 columns that end inside 64 columns
    (1100, 8712, 2048, 4352, 8704, 8704),   # .. at 64 columns, the last 8 fp32
    (1100, 8712, 2048, 8712, 8712, 8717),   # .. rows that 16 bytes do not fit
    (700, 2304, 2048, 1024, 2304, 2304),    # 128 x 128 in two groups of waves
    (333, 2300, 512, 0, 2236, 2240),
])
@pytest.mark.parametrize("act", ["TANH", "ERF"])
def test_act_blocks(ti, M, N, K, act_cols, t_cols, ldo, act):
    """Bias, activation of the first columns, fp32 columns past the 16-bit ones.  Bound: |gelu'| <= 1.13 times the product's, and the
    roundings of the stored types and of the activation (4e-6 of the value, as test_gelu has it; tanh form 1e-5)."""
    a, w, f = operands(M, N, K, torch.bfloat16, 1, 7)
    bias = torch.randn(N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    out = torch.full((M + 1, ldo), 7.0, device="cuda").bfloat16()
    out2 = torch.full((M + 1, N - t_cols + 4), 7.0, device="cuda")
    call(ti, ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=ldo, M=M, N=N, K=K, batch=1, epi=ti.DE_ACT,
                          dtype=ti.DT_BF16, add=bias.data_ptr(), act=ti.ACT_GELU_TANH if act == "TANH" else ti.ACT_GELU_ERF, act_cols=act_cols,
                          t_cols=t_cols, out2=out2.data_ptr(), ld2=N - t_cols + 4))
    y = a.double() @ w[0].double().T + bias.double()
    tol = 1.13 * (K + 1) * 2.0**-24 * (a.double().abs() @ w[0].double().abs().T + bias.double().abs())
    ref = torch.cat([torch.nn.functional.gelu(y[:, :act_cols], approximate="tanh" if act == "TANH" else "none"), y[:, act_cols:]], 1)
    err = (torch.cat([out[:M, :t_cols].double(), out2[:M, : N - t_cols].double()], 1) - ref).abs()
    assert err[:, :t_cols].le(tol[:, :t_cols] + (2.0**-8 + 1e-5) * ref[:, :t_cols].abs() + 1e-7).all()
    assert err[:, t_cols:].le(tol[:, t_cols:] + 2.0**-23 * ref[:, t_cols:].abs()).all()
    assert (out[M] == 7).all() and (out[:, t_cols:] == 7).all() and (out2[M] == 7).all() and (out2[:, N - t_cols :] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [5, 200])
def test_gelu(ti, dtype, M):
    """GELU (erf form) over both tails and its zeros, from a product with the identity: bf16 half a unit in the last
    place of the exact value plus 4e-6 of it (the erfc fit's tail), fp32 the cancellation of 1 + erf, 2^-23 |z|."""
    N = 512
    z = torch.cat([torch.linspace(-9, 9, M * N - 6, device="cuda"), torch.tensor([0.0, -0.0, 1e-30, -1e-30, 60.0, -60.0], device="cuda")])
    a = z[torch.randperm(M * N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(0))].view(M, N).to(dtype)
    vec = 8 if dtype == torch.bfloat16 else 4
    w = torch.eye(N, device="cuda", dtype=dtype).view(-1, 16, N // (4 * vec), 4, vec).permute(0, 2, 3, 1, 4).contiguous()
    out = torch.empty(M, N, device="cuda", dtype=dtype)
    d = ti.DenseArgs(w=w.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=N, ldo=N, M=M, N=N, K=N, batch=1, epi=ti.DE_ACT, t_cols=N,
                     act=2, act_cols=N, dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    call(ti, d)
    zd = a.double()
    ref = 0.5 * zd * torch.special.erfc(-zd / 2**0.5)
    tol = (2.0**-8 + 4e-6) * ref.abs() + 1e-38 if dtype == torch.bfloat16 else 2.0**-23 * zd.abs() + 2.0**-22 * ref.abs() + 1e-38
    assert (out.double() - ref).abs().le(tol).all()


@pytest.mark.parametrize("lo,hi", [(0.0, 0.3), (-0.3, 0.0), (0.3, 1.5), (-1.0, -0.3), (-3.0, -1.0)])
def test_gelu_roundings(ti, lo, hi):
    """GELU's error before the bf16 store, by how many outputs are not the nearest bf16 of the exact value: an error of e
    (relative, mean) crosses a boundary of the 2^-8 .. 2^-9 steps for about e / 2^-8.5 of the values.  No more than 0.5 z (1
    + erff) gives in fp32 (its roundings: half a unit of 1 + erff, of erff and of the two products), by three standard
    deviations of the count.  z has all its 24 bits: a product of three bf16 parts with three identities."""
    M, N = 4096, 512
    g = torch.Generator(device="cuda").manual_seed(5)
    z = torch.rand(M, N, device="cuda", generator=g) * (hi - lo) + lo
    top = z.bfloat16()
    mid = (z - top.float()).bfloat16()
    a = torch.cat([top, mid, (z - top.float() - mid.float()).bfloat16()], 1)
    z = a.double().view(M, 3, N).sum(1)
    w = torch.eye(N, device="cuda", dtype=torch.bfloat16).repeat(1, 3).view(-1, 16, 3 * N // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()
    out = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    call(ti, ti.DenseArgs(w=w.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=3 * N, ldo=N, M=M, N=N, K=3 * N, batch=1, epi=ti.DE_ACT,
                          t_cols=N, act=2, act_cols=N, dtype=ti.DT_BF16))
    ref = 0.5 * z * torch.special.erfc(-z / 2**0.5)
    zf = z.float()
    assert (zf.double() == z).all()
    fp32 = 0.5 * zf * (1 + torch.erf(zf * 0.70710678118654752))

    def wrong(x):   # 64-bit distance to the stored value against half a step
        step = torch.exp2(torch.floor(torch.log2(ref.abs().clamp_min(1e-30))) - 7)
        return int(((x.double() - ref).abs() > 0.5 * step * (1 + 1e-9)).sum())

    n32 = wrong(fp32.bfloat16())
    assert wrong(out) <= n32 + 3 * (n32 + 1) ** 0.5, (wrong(out), n32)


# Tiles of few rows, their two groups of waves over k, and row tiles of 3/4 of a block: odd numbers of stages, fewer stages
# than the ring holds, ragged last rows and columns.
SPREAD = [
    ((32, 64), 65, 70, 64, torch.bfloat16),        # one stage
    ((32, 64), 97, 1001, 192, torch.bfloat16),     # three; last row tile 1 row
    ((64, 64), 333, 2051, 1088, torch.bfloat16),
    ((64, 128), 700, 2061, 2112, torch.bfloat16),  # 48 rows a tile
    ((64, 128), 250, 6201, 1088, torch.bfloat16),  # 64
    ((128, 128), 650, 4101, 320, torch.bfloat16),  # 96
    ((128, 128), 1300, 2501, 1088, torch.bfloat16),
    ((128, 128), 300, 8201, 320, torch.bfloat16),  # without the groups
    ((128, 256), 2000, 2101, 320, torch.bfloat16),  # 96
    ((32, 64), 97, 1001, 96, torch.float32),
    ((64, 64), 333, 2051, 1056, torch.float32),
    ((128, 128), 650, 4101, 352, torch.float32),
]


@pytest.mark.parametrize("epi", ["f32", "swiglu"])
@pytest.mark.parametrize("shape,M,N,K,dtype", SPREAD)
def test_small_tiles(ti, shape, M, N, K, dtype, epi):
    N += epi == "swiglu" and N % 2
    a, w, f = operands(M, N, K, dtype)
    ldo = N + 5 if epi == "f32" else N // 2
    out = torch.full((M + 1, ldo), 7.0, device="cuda").to(torch.float32 if epi == "f32" else dtype)
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=ldo, M=M, N=N, K=K, batch=1,
                     epi=ti.DE_F32 if epi == "f32" else ti.DE_SWIGLU, dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    assert tile(ti, d) == shape
    call(ti, d)
    if epi == "f32":
        check(out[:M, :N], a, w[0], dtype)
        assert (out[:, N:] == 7).all()
    else:
        check_swiglu(out[:M], a, w[0], dtype)
    assert (out[M] == 7).all()


@pytest.mark.parametrize("M,E,top,tile_rows", [(1, 5, 3, 16), (17, 7, 2, 16), (300, 64, 6, 128), (700, 130, 5, 64), (640, 3, 2, 256), (64, 1, 1, 64)])
def test_route_tiles(ti, M, E, top, tile_rows):
    """Tiles of a given choice: every entry once, in its expert's tile; those of 128 rows and more with the whole ones first,
    then the rests, largest first, smaller ones expert by expert."""
    g = torch.Generator(device="cuda").manual_seed(M)
    skew = torch.rand(M, E, device="cuda", generator=g) ** torch.linspace(1, 4, E, device="cuda")
    idx = skew.topk(top, 1).indices.int().contiguous()
    cap = ti.lib().ti_route_max_tiles(M, E, top, tile_rows)
    wgt = torch.zeros(M, top, device="cuda")
    lst = torch.full((M * top,), -1, dtype=torch.int32, device="cuda")
    tiles = torch.full((cap, 4), -1, dtype=torch.int32, device="cuda")
    n = torch.zeros(1, dtype=torch.int32, device="cuda")
    r = ti.RouteArgs(logits=None, ld=E, M=M, E=E, top=top, idx=idx.data_ptr(), wgt=wgt.data_ptr(), list=lst.data_ptr(),
                     tiles=tiles.data_ptr(), n_tiles=n.data_ptr(), tile_rows=tile_rows)
    torch.cuda.synchronize()
    ti.check(ti.lib().ti_route(C.byref(r), None))
    ti.sync()
    idx, lst, tiles, n = idx.flatten().cpu().numpy(), lst.cpu().numpy(), tiles.cpu().numpy(), int(n)
    counts = np.bincount(idx, minlength=E)
    assert n == (-(-counts // tile_rows)).sum() <= cap and sorted(lst) == list(range(M * top))
    seen = []
    for e, first, rows, _ in tiles[:n]:
        assert (idx[lst[first:first + rows]] == e).all()
        seen += range(first, first + rows)
    assert sorted(seen) == list(range(M * top))
    rows = tiles[:n, 2]
    assert (np.diff(rows if tile_rows >= 128 else -tiles[:n, 1]) <= 0).all() and (rows == tile_rows).sum() == (counts // tile_rows).sum()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [1, 7, 8, 9, 15, 16])
@pytest.mark.parametrize("N,K", [(16, 64), (1, 128), (23, 192), (64, 2048), (2041, 1088), (2048, 8192), (2049, 512)])
def test_few_rows_halves(ti, dtype, M, N, K):
    """Two k-tiles a product (dense_half_kernel, N <= 2048): one pair of them, fewer pairs than waves, ragged columns in
    either half of a column tile, rows of one and of two products; added columns and untouched surroundings."""
    a, w, f = operands(M, N, K, dtype)
    add = torch.randn(N, device="cuda", generator=torch.Generator(device="cuda").manual_seed(5))
    out = torch.full((M + 1, N + 3), 7.0, device="cuda")
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N + 3, M=M, N=N, K=K, batch=1, epi=ti.DE_F32,
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    call(ti, d)
    check(out[:M, :N], a, w[0], dtype)
    plain = out[:M, :N].clone()
    d.add = add.data_ptr()
    call(ti, d)
    assert torch.equal(out[:M, :N], plain + add)
    assert (out[:, N:] == 7).all() and (out[M] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N", [(2, 40), (7, 2048), (16, 1001), (16, 2064), (50, 300), (130, 300)])
def test_shared_rows(ti, dtype, M, N):
    """row_div without row lists: output row m is the product of row m / row_div of a, on the kernels of every row count."""
    K, div = 320, 3
    a, w, f = operands(M, N, K, dtype)
    a = a[: (M - 1) // div + 1].contiguous()
    out = torch.full((M + 1, N), 7.0, device="cuda")
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N, M=M, N=N, K=K, batch=1, epi=ti.DE_F32, row_div=div,
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    call(ti, d)
    check(out[:M], a[torch.arange(M, device="cuda") // div], w[0], dtype)
    assert (out[M] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,per,blocks", [(65, 16, 2), (130, 24, 3), (100, 33, 2), (200, 100, 2), (129, 256, 3)])
def test_lru_gates(ti, dtype, M, per, blocks):
    """Gates of a linear recurrence: whole and ragged 16-byte outputs, odd blocks whose last channel stands alone, rows past a tile.
    Bound: the products' roundings through the logistic functions (slope 1/4), 2^-20 of each function's own, times what the
    coefficients make of them."""
    K = ti.lib().ti_stack_kpad(ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32, per)
    N = 2 * per
    g = torch.Generator("cuda").manual_seed(M)
    u, w, f = operands(M, N, blocks * K, dtype, 1, M)
    _, w, f = operands(M, N, K, dtype, blocks, M + 1)
    bias = torch.randn(blocks, N, device="cuda", generator=g)
    rate = torch.rand(blocks * per, device="cuda", generator=g) * 8 + 0.01
    out = torch.full((M + 1, blocks * per, 2), 7.0, device="cuda")
    d = ti.DenseArgs(w=f.data_ptr(), w_batch=f[0].numel(), a=u.data_ptr(), a_batch=K, out=out.data_ptr(), lda=blocks * K, ldo=2 * blocks * per, M=M, N=N,
                     K=K, batch=blocks, epi=ti.DE_LRU, add=bias.data_ptr(), lru_rate=rate.data_ptr(),
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    call(ti, d)
    for b in range(blocks):
        a = u[:, b * K : (b + 1) * K].double()
        z, e = a @ w[b].double().T + bias[b].double(), K * 2.0**-24 * (a.abs() @ w[b].double().abs().T + bias[b].double().abs())
        r, i, er, ei = z[:, 0::2], z[:, 1::2], e[:, 0::2], e[:, 1::2]
        k = rate[b * per : (b + 1) * per].double()
        la = -torch.sigmoid(r) * k
        da = k * (er / 4 + 2.0**-20)
        s2 = -torch.expm1(2 * la)
        x = a[:, :per]
        ref_b, s = s2.sqrt() * torch.sigmoid(i) * x, s2.sqrt()
        got = out[:M, b * per : (b + 1) * per].double()
        assert (got[..., 0] - la.exp()).abs().le(la.exp() * da + 2.0**-21).all()
        assert (got[..., 1] - ref_b).abs().le(x.abs() * (s * (ei / 4 + 2.0**-19) + torch.exp(2 * la) * da / s.clamp(min=1e-30)) + 1e-12).all()
    assert (out[M] == 7).all()


@pytest.mark.parametrize("dtype,M,N,K,few", [
    (torch.bfloat16, 65, 16, 512, True), (torch.bfloat16, 65, 16, 448, False), (torch.bfloat16, 2048, 64, 1024, True),
    (torch.bfloat16, 2049, 64, 512, False), (torch.bfloat16, 500, 250, 1088, True), (torch.bfloat16, 130, 914, 640, False),
    (torch.float32, 65, 7, 256, True), (torch.float32, 65, 7, 224, False), (torch.float32, 250, 1018, 544, True), (torch.float32, 257, 1018, 544, False)])
def test_few_tiles(ti, dtype, M, N, K, few):
    """Products of more than 64 rows and few tiles of outputs, to either side of the line."""
    a, w, f = operands(M, N, K, dtype)
    out = torch.full((M + 1, N + 3), 7.0, device="cuda")
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N + 3, M=M, N=N, K=K, batch=1, epi=ti.DE_F32,
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    assert (tile(ti, d) == (0, 0)) == few
    call(ti, d)
    check(out[:M, :N], a, w[0], dtype)
    assert (out[M] == 7).all() and (out[:, N:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(65, 64, 2048), (500, 250, 576), (100, 1024, 512)])
def test_few_tiles_swiglu(ti, dtype, M, N, K):
    a, w, f = operands(M, N, K, dtype)
    out = torch.full((M + 1, N // 2), 7.0, device="cuda").to(dtype)
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N // 2, M=M, N=N, K=K, batch=1, epi=ti.DE_SWIGLU,
                     dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    assert tile(ti, d) == (0, 0)
    call(ti, d)
    check_swiglu(out[:M], a, w[0], dtype)
    assert (out[M] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("epi", ["key", "value"])
@pytest.mark.parametrize("M,heads,hw,K", [(1, 2, 64, 64), (65, 8, 64, 256), (129, 3, 32, 320), (500, 16, 128, 512), (641, 13, 128, 128), (1025, 8, 128, 64),
                                          (2049, 9, 128, 64)])
def test_fragments(ti, dtype, epi, M, heads, hw, K):
    """Key and value fragments on either size of block: whole blocks of 128 keys are written, the last key again past the end."""
    N, kt, vec = heads * hw, 32 if dtype == torch.bfloat16 else 16, 8 if dtype == torch.bfloat16 else 4
    a, w, f = operands(M, N, K, dtype)
    rows = -(-M // 128) * 128
    blocks = rows // 16 + 8
    out = torch.full((blocks * 16 * N,), 7.0, device="cuda").to(dtype)
    d = ti.DenseArgs(w=f.data_ptr(), a=a.data_ptr(), out=out.data_ptr(), lda=K, ldo=N, M=M, N=N, K=K, batch=1, head_w=hw, key_blocks=blocks,
                     epi=ti.DE_KFRAG if epi == "key" else ti.DE_VFRAG, dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    call(ti, d)
    m, n = torch.arange(rows, device="cuda")[:, None], torch.arange(N, device="cuda")[None, :]
    h, c = n // hw, n % hw
    if epi == "key":
        at = (((h * blocks + (m >> 4)) * (hw // kt) + c // kt) * 64 + c % kt // vec * 16 + (m & 15)) * vec + c % vec
    else:
        at = (((h * (hw >> 4) + (c >> 4)) * (blocks * 16 // kt) + m // kt) * 64 + ((m & 15) >> 2) * 16 + (c & 15)) * vec + (m % kt >> 4) * 4 + (m & 3)
    got = out[at]
    check(got[:M], a, w[0], dtype, dtype == torch.bfloat16)
    assert (got[M:] == got[M - 1]).all()
    out[at] = 7.0
    assert (out == 7).all()
