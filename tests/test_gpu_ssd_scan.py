"""ti_ssd_scan against the recurrence in float64: states of up to 64, 128 and 256 rows and odd ones, value dimensions that are no multiple
of 16, blocks of 64 tokens whole, one short and one over, a carried state.  Bound: fp32 roundings of the sums -- the state's rows, a
block's tokens, its decays and step sizes (a few units each), the blocks that a state has gone through -- of 2^-24 of the magnitudes'
sum each."""
from __future__ import annotations

import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


class SsdArgs(C.Structure):   # ti_ssd_args (include/ti_stack.h)
    _fields_ = [(n, C.c_void_p) for n in ("a", "dt", "dt_bias", "a_log", "d", "conv_w", "conv_b", "ring", "state", "y", "pos", "slot")] + \
               [(n, C.c_int32) for n in ("M", "heads", "vdim", "state_n", "groups", "taps", "lda", "ldy", "o0", "slot0", "dtype")]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,heads,vdim,n,groups,carry", [
    (1, 2, 16, 128, 1, True), (15, 4, 64, 128, 2, False), (64, 2, 24, 100, 1, True), (65, 2, 64, 68, 2, True), (129, 4, 40, 132, 4, True),
    (200, 2, 64, 256, 1, True), (333, 8, 64, 128, 1, True), (70, 2, 20, 64, 1, True), (130, 2, 16, 12, 2, False), (512, 2, 16, 64, 1, True),
    (577, 2, 20, 40, 1, True)])
def test_ssd_scan(ti, dtype, M, heads, vdim, n, groups, carry):
    g = torch.Generator("cuda").manual_seed(M + n)

    def rand(*s):
        return torch.randn(*s, device="cuda", generator=g)

    kt = 32 if dtype == torch.bfloat16 else 16
    nk, np_, inner = -(-n // kt) * kt, -(-n // 4) * 4, heads * vdim
    lda = inner + 2 * groups * nk
    a = torch.zeros(M, lda, device="cuda", dtype=dtype)
    x, b, c = (torch.nn.functional.silu(rand(*s)).to(dtype) for s in ((M, heads, vdim), (M, groups, n), (M, groups, n)))
    a[:, :inner] = x.reshape(M, inner)
    a[:, inner : inner + groups * nk].view(M, groups, nk)[:, :, :n] = b
    a[:, inner + groups * nk :].view(M, groups, nk)[:, :, :n] = c
    dt, bias, a_log, d = rand(M, heads), rand(heads) - 2, torch.log(1 + 15 * torch.rand(heads, device="cuda", generator=g)), rand(heads)
    state = torch.zeros(2, heads, vdim, np_, device="cuda")   # (slot 1 is another request's)
    state[1] = 3.0
    if carry:
        state[0, :, :, :n] = rand(heads, vdim, n)
    s = state[0, :, :, :n].double()
    mag, y = s.abs(), torch.full((M + 1, inner), 7.0, device="cuda")
    pos = torch.arange(M, device="cuda", dtype=torch.int32) + (50 if carry else 0)
    args = SsdArgs(a=a.data_ptr(), dt=dt.data_ptr(), dt_bias=bias.data_ptr(), a_log=a_log.data_ptr(), d=d.data_ptr(), state=state.data_ptr(),
                   y=y.data_ptr(), pos=pos.data_ptr(), M=M, heads=heads, vdim=vdim, state_n=n, groups=groups, taps=4, lda=lda, ldy=inner, o0=inner,
                   slot0=0, dtype=ti.DT_BF16 if dtype == torch.bfloat16 else ti.DT_F32)
    torch.cuda.synchronize()
    fn = ti.lib().ti_ssd_scan
    fn.argtypes = [C.c_void_p, C.c_void_p]
    ti.check(fn(C.addressof(args), None))
    ti.sync()
    step = torch.nn.functional.softplus(dt.double() + bias.double(), threshold=1e9)
    decay = torch.exp(-torch.exp(a_log.double()) * step)[:, :, None, None]
    x, b, c = x.double(), b.double().repeat_interleave(heads // groups, 1), c.double().repeat_interleave(heads // groups, 1)
    blocks = -(-M // 64)
    unit = (n + 64 + 96 + 8 * blocks) * 2.0**-24
    for t in range(M):
        put = (step[t, :, None] * x[t])[:, :, None] * b[t, :, None, :]
        s, mag = s * decay[t] + put, mag * decay[t] + put.abs()
        ref, size = (s * c[t, :, None, :]).sum(-1), (mag * c[t, :, None, :].abs()).sum(-1)
        ref, size = ref + d.double()[:, None] * x[t], size + (d.double()[:, None] * x[t]).abs()
        assert (y[t].view(heads, vdim).double() - ref).abs().le(unit * size).all(), t
    assert (state[0, :, :, :n].double() - s).abs().le(unit * mag).all()
    assert (y[M] == 7).all() and (state[1] == 3).all() and (state[0, :, :, n:] == 0).all()


@pytest.mark.parametrize("n", [100, 128, 256])
@pytest.mark.parametrize("what", ["c", "x"])
def test_ssd_scan_infinities(ti, what, n):
    """One infinite C (of token 5), or input of a token (70, dimension 3 of every head), beside positive ones: outputs that it takes part in are infinite
    as a sum of whole products has them, the others what they are without it (but for the rows before an infinite input in its block of 64), up to
    the order of fp32 sums of positive values."""
    g = torch.Generator("cuda").manual_seed(n)
    M, heads, vdim = 150, 16, 16
    nk, np_, inner = -(-n // 32) * 32, -(-n // 4) * 4, heads * vdim

    def rand(*s):
        return torch.randn(*s, device="cuda", generator=g).abs() + 0.1

    a = torch.zeros(M, inner + 2 * nk, device="cuda").bfloat16()
    a[:, :inner], a[:, inner : inner + n], a[:, inner + nk : inner + nk + n] = rand(M, inner), rand(M, n), rand(M, n)
    dt, bias, a_log, d = rand(M, heads), rand(heads), torch.full((heads,), -3.0, device="cuda"), rand(heads)
    carry = torch.zeros(heads, vdim, np_, device="cuda")
    carry[:, :, :n] = rand(heads, vdim, n).bfloat16().float()   # (parts of 0)
    pos = torch.arange(M, device="cuda", dtype=torch.int32) + 9
    fn = ti.lib().ti_ssd_scan
    fn.argtypes = [C.c_void_p, C.c_void_p]

    def run():
        state, y = carry.clone(), torch.full((M, inner), 7.0, device="cuda")
        args = SsdArgs(a=a.data_ptr(), dt=dt.data_ptr(), dt_bias=bias.data_ptr(), a_log=a_log.data_ptr(), d=d.data_ptr(), state=state.data_ptr(),
                       y=y.data_ptr(), pos=pos.data_ptr(), M=M, heads=heads, vdim=vdim, state_n=n, groups=1, taps=4, lda=a.shape[1], ldy=inner, o0=inner,
                       slot0=0, dtype=ti.DT_BF16)
        torch.cuda.synchronize()
        ti.check(fn(C.addressof(args), None))
        ti.sync()
        return y.view(M, heads, vdim)

    plain = run()
    assert plain.isfinite().all()
    if what == "c":
        a[5, inner + nk + 7] = float("inf")
        y = run()
        assert (y[5] == float("inf")).all()
        same = torch.arange(M, device="cuda") != 5
        assert ((y - plain)[same].abs() <= 2.0**-19 * plain[same]).all()
    else:
        a[70, 3:inner:vdim] = float("inf")
        y = run()
        # (a state's rows past n are 0 times the input in the blocks behind)
        assert (y[70 : M if n % 64 == 0 else 128, :, 3] == float("inf")).all()
        assert ((y - plain)[:64].abs() <= 2.0**-19 * plain[:64]).all()
        other = torch.arange(vdim, device="cuda") != 3
        assert ((y - plain)[:, :, other].abs() <= 2.0**-19 * plain[:, :, other]).all()
