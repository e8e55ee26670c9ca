"""Prompt attention of the layer-stack models (ti_latent_attn_prefill, ti_gqa_prefill) against float64: 16-bit heads whose keys and
values a workgroup's waves share (64 or 128 dims, 32 or 64 rotated ones), 16 and 32 rows a wave, ragged rows, chunks behind a
prefix, keys past the chunk that hold NaN.  Bound: weights rounded to bf16 (2^-9 each), the output's own rounding, fp32 sums."""
from __future__ import annotations

import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


class Args(C.Structure):
    """ti_latent_prefill_args (include/ti_stack.h)."""
    _fields_ = [(n, C.c_void_p) for n in ("q", "kfrag", "vfrag", "cache", "sink", "gate", "out")] + [("scale", C.c_float)] + \
        [(n, C.c_int32) for n in ("M", "pos0", "heads", "dim_p", "rot_p", "lat_p", "vdim", "vdim_p", "key_blocks", "ldo", "dtype")]


@pytest.mark.parametrize("dim,rot", [(128, 64), (128, 32), (64, 64), (64, 32)])
@pytest.mark.parametrize("M,pos0,heads", [(17, 0, 3), (64, 64, 9), (100, 3, 2), (129, 191, 8), (333, 0, 16), (1401, 70, 24)])
def test_latent_prompt(ti, dim, rot, M, pos0, heads):
    g = torch.Generator(device="cuda").manual_seed(M + dim + rot)
    keys, lat = pos0 + M, 96
    seq = -(-keys // 128) * 128

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g).bfloat16()

    q, k, v, kr = rand(M, heads, dim + rot), rand(heads, seq, dim), rand(heads, seq, dim), rand(seq, rot)
    cache = torch.full((seq, lat + rot), float("nan"), device="cuda").bfloat16()
    cache[:keys, lat:] = kr[:keys]
    # fragments: keys [head][16 keys][32 dims][lane][8], values [head][16 dims][32 keys][lane][8]
    kf = k.view(heads, seq // 16, 16, dim // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).contiguous()
    vf = v.view(heads, seq // 32, 2, 4, 4, dim // 16, 16).permute(0, 5, 1, 3, 6, 2, 4).contiguous()
    sink = torch.randn(heads, device="cuda", generator=g)
    gate = torch.rand(M, heads, device="cuda", generator=g)
    out = torch.full((M + 1, heads * dim), 7.0, device="cuda").bfloat16()
    scale = 2.0 * (dim + rot) ** -0.5
    a = Args(q=q.data_ptr(), kfrag=kf.data_ptr(), vfrag=vf.data_ptr(), cache=cache.data_ptr(), sink=sink.data_ptr(), gate=gate.data_ptr(),
             out=out.data_ptr(), scale=scale, M=M, pos0=pos0, heads=heads, dim_p=dim, rot_p=rot, lat_p=lat, vdim=dim, vdim_p=dim,
             key_blocks=seq // 16, ldo=heads * dim, dtype=ti.DT_BF16)
    torch.cuda.synchronize()
    ti.check(ti.lib().ti_latent_attn_prefill(C.byref(a), None))
    ti.sync()
    assert (out[M] == 7).all()
    mask = torch.arange(keys, device="cuda") > pos0 + torch.arange(M, device="cuda")[:, None]
    for h in range(heads):
        kk = torch.cat([k[h, :keys].double(), kr[:keys].double()], 1)
        sc = (q[:, h].double() @ kk.T * scale).masked_fill(mask, -float("inf"))
        w = torch.softmax(torch.cat([sc, sink[h].double().expand(M, 1)], 1), 1)[:, :-1].contiguous()
        vv, gt = v[h, :keys].double(), gate[:, h, None].double()
        ref, mag = w @ vv * gt, w @ vv.abs() * gt
        err = (out[:M, h * dim : (h + 1) * dim].double() - ref).abs()
        assert err.le(2.0**-8 * mag + 2.0**-8 * ref.abs() + 1e-6).all(), (h, err.max().item())


class GqaArgs(C.Structure):
    """ti_gqa_attn_args (include/ti_stack.h)."""
    _fields_ = [("q", C.c_void_p), ("cache", C.c_void_p), ("slot_stride", C.c_int64)] + \
        [(n, C.c_void_p) for n in ("pos", "slot", "sink", "gate", "out", "part_o", "part_ml")] + [("scale", C.c_float)] + \
        [(n, C.c_int32) for n in ("M", "pos0", "heads", "kv_heads", "dim", "vdim", "seq_p", "splits", "ldg", "ldo", "dtype")]


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("M,pos0,heads,kv,extras", [(17, 0, 6, 3, True), (100, 61, 4, 1, False), (129, 191, 16, 2, True), (300, 0, 12, 4, False),
                                                    (777, 5, 45, 9, True), (1401, 70, 24, 8, True)])
def test_gqa_prompt(ti, dim, M, pos0, heads, kv, extras):
    g = torch.Generator(device="cuda").manual_seed(M + dim)
    keys, rep = pos0 + M, heads // kv
    seq = -(-keys // 64) * 64

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g).bfloat16()

    q, k, v = rand(M, heads, dim), rand(kv, seq, dim), rand(kv, seq, dim)
    k[:, keys:] = float("nan")
    # a block of 64 positions: [4 key tiles][32 dims][lane][8] keys, [16 dims][32 positions][lane][8] values
    kf = k.view(kv, seq // 64, 4, 16, dim // 32, 4, 8).permute(0, 1, 2, 4, 5, 3, 6).reshape(kv, seq // 64, -1)
    vf = v.view(kv, seq // 64, 2, 2, 4, 4, dim // 16, 16).permute(0, 1, 6, 2, 4, 7, 3, 5).reshape(kv, seq // 64, -1)
    cache = torch.cat([kf, vf], -1).contiguous()
    assert cache[0, 0].numel() == ti.lib().ti_gqa_block_elems(ti.DT_BF16, dim, dim)
    sink = torch.randn(heads, device="cuda", generator=g)
    gate = torch.randn(M, heads * dim + 4, device="cuda", generator=g)
    out = torch.full((M + 1, heads * dim), 7.0, device="cuda").bfloat16()
    scale = 2.0 * dim**-0.5
    a = GqaArgs(q=q.data_ptr(), cache=cache.data_ptr(), sink=sink.data_ptr() if extras else None, gate=gate.data_ptr() if extras else None,
                out=out.data_ptr(), scale=scale, M=M, pos0=pos0, heads=heads, kv_heads=kv, dim=dim, vdim=dim, seq_p=seq, ldg=heads * dim + 4,
                ldo=heads * dim, dtype=ti.DT_BF16)
    torch.cuda.synchronize()
    ti.check(ti.lib().ti_gqa_prefill(C.byref(a), None))
    ti.sync()
    assert (out[M] == 7).all()
    mask = torch.arange(keys, device="cuda") > pos0 + torch.arange(M, device="cuda")[:, None]
    for h in range(heads):
        sc = (q[:, h].double() @ k[h // rep, :keys].double().T * scale).masked_fill(mask, -float("inf"))
        s0 = sink[h].double().expand(M, 1) if extras else sc.new_full((M, 1), -float("inf"))
        w = torch.softmax(torch.cat([sc, s0], 1), 1)[:, :-1].contiguous()
        gt = torch.sigmoid(gate[:, h * dim : (h + 1) * dim].double()) if extras else 1.0
        vv = v[h // rep, :keys].double()
        ref, mag = w @ vv * gt, w @ vv.abs() * gt
        err = (out[:M, h * dim : (h + 1) * dim].double() - ref).abs()
        assert err.le(2.0**-8 * mag + 2.0**-8 * ref.abs() + 1e-6).all(), (h, err.max().item())


def latent_prompt(ti, q, k, v, kr, sink, scale, pos0):
    """Outputs [row][head][dim] of keys k, values v [head][key][dim] and rotated parts kr [key][rot], without a gate."""
    (M, heads, width), (_, seq, dim) = q.shape, k.shape
    kf = k.view(heads, seq // 16, 16, dim // 32, 4, 8).permute(0, 1, 3, 4, 2, 5).contiguous()
    vf = v.view(heads, seq // 32, 2, 4, 4, dim // 16, 16).permute(0, 5, 1, 3, 6, 2, 4).contiguous()
    cache, gate, out = torch.cat([kr, kr], 1).contiguous(), torch.ones(M, heads, device="cuda"), torch.empty(M, heads, dim, device="cuda").bfloat16()
    a = Args(q=q.data_ptr(), kfrag=kf.data_ptr(), vfrag=vf.data_ptr(), cache=cache.data_ptr(), sink=sink.data_ptr(), gate=gate.data_ptr(),
             out=out.data_ptr(), scale=scale, M=M, pos0=pos0, heads=heads, dim_p=dim, rot_p=width - dim, lat_p=width - dim, vdim=dim, vdim_p=dim,
             key_blocks=seq // 16, ldo=heads * dim, dtype=ti.DT_BF16)
    torch.cuda.synchronize()
    ti.check(ti.lib().ti_latent_attn_prefill(C.byref(a), None))
    ti.sync()
    return out


def gqa_prompt(ti, q, k, v, sink, scale, pos0):
    """Outputs [row][head][dim] of keys and values [kv-head][key][dim]."""
    (M, heads, dim), (kv, seq, _) = q.shape, k.shape
    kf = k.view(kv, seq // 64, 4, 16, dim // 32, 4, 8).permute(0, 1, 2, 4, 5, 3, 6).reshape(kv, seq // 64, -1)
    vf = v.view(kv, seq // 64, 2, 2, 4, 4, dim // 16, 16).permute(0, 1, 6, 2, 4, 7, 3, 5).reshape(kv, seq // 64, -1)
    cache, out = torch.cat([kf, vf], -1).contiguous(), torch.empty(M, heads, dim, device="cuda").bfloat16()
    a = GqaArgs(q=q.data_ptr(), cache=cache.data_ptr(), sink=None if sink is None else sink.data_ptr(), out=out.data_ptr(), scale=scale, M=M,
                pos0=pos0, heads=heads, kv_heads=kv, dim=dim, vdim=dim, seq_p=seq, ldo=heads * dim, dtype=ti.DT_BF16)
    torch.cuda.synchronize()
    ti.check(ti.lib().ti_gqa_prefill(C.byref(a), None))
    ti.sync()
    return out


def prompt(ti, kind, dim, M, pos0, heads, sharp, sink, rot=32, group=2):
    """A call's outputs and, in float64, its weights [head][row][key] and values [head][key][dim]."""
    g = torch.Generator(device="cuda").manual_seed(M + dim)
    keys, rot = pos0 + M, rot if kind == "latent" else 0
    kv = heads if kind == "latent" else heads // group
    seq = -(-keys // 128) * 128

    def rand(*shape):
        return torch.randn(*shape, device="cuda", generator=g).bfloat16()

    q, k, v, kr = rand(M, heads, dim + rot), rand(kv, seq, dim), rand(kv, seq, dim), rand(seq, rot)
    scale = sharp * (dim + rot) ** -0.5
    out = latent_prompt(ti, q, k, v, kr, sink, scale, pos0) if kind == "latent" else gqa_prompt(ti, q, k, v, sink, scale, pos0)
    kk = torch.cat([k[:, :keys].double(), kr[:keys].double().expand(kv, keys, rot)], 2).repeat_interleave(heads // kv, 0)
    sc = (q.double().transpose(0, 1) @ kk.transpose(1, 2).contiguous()) * scale
    sc = sc.masked_fill(torch.arange(keys, device="cuda") > pos0 + torch.arange(M, device="cuda")[:, None], -float("inf"))
    w = torch.softmax(torch.cat([sc, sink.double().view(heads, 1, 1).expand(heads, M, 1)], 2), 2)[:, :, :-1].contiguous()
    return out, w, v[:, :keys].double().repeat_interleave(heads // kv, 0)


@pytest.mark.parametrize("kind", ["latent", "gqa"])
@pytest.mark.parametrize("dim,M,pos0,heads", [(128, 100, 3, 4), (128, 700, 0, 16), (128, 1401, 70, 24), (64, 300, 64, 8), (64, 1401, 5, 24)])
def test_largest_weight_is_not_rounded(ti, kind, dim, M, pos0, heads):
    """Sharp rows, one weight near 1: a block's largest weight is a power of 2 before the row's sum divides it, so bf16 rounds only the
    others (2^-8 of each) and the output."""
    out, w, v = prompt(ti, kind, dim, M, pos0, heads, 6.0, torch.full((heads,), -60.0, device="cuda"))
    top, at = w.max(2)
    ref, mag = w @ v, w @ v.abs() - top[:, :, None] * torch.gather(v.abs(), 1, at[:, :, None].expand(-1, -1, dim))
    err = (out.transpose(0, 1).double() - ref).abs()
    assert err.le(2.0**-8 * mag + 2.0**-8 * ref.abs() + 1e-5).all()


@pytest.mark.parametrize("kind", ["latent", "gqa"])
@pytest.mark.parametrize("dim,M,pos0,heads", [(128, 100, 3, 4), (128, 1401, 16, 24), (64, 300, 41, 8), (64, 1401, 5, 40), (96, 200, 9, 6)])
def test_sinks_of_minus_infinity(ti, kind, dim, M, pos0, heads):
    """Heads without a sink beside ones with it; blocks whose keys a row does not see come before its first (positions that start inside
    64).  Bound as above."""
    sink = torch.randn(heads, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    sink[::2] = -float("inf")
    out, w, v = prompt(ti, kind, dim, M, pos0, heads, 2.0, sink)
    ref = w @ v
    assert (out.transpose(0, 1).double() - ref).abs().le(2.0**-8 * (w @ v.abs()) + 2.0**-8 * ref.abs() + 1e-6).all()


@pytest.mark.parametrize("kind,dim,rot,M,pos0,heads,group", [   # one of every kernel, by attn_plan.hpp
    ("latent", 128, 64, 700, 0, 4, 1), ("latent", 128, 64, 1024, 5, 16, 1), ("latent", 128, 64, 2041, 0, 16, 1), ("latent", 128, 64, 1301, 0, 24, 1),
    ("latent", 128, 32, 1024, 5, 16, 1), ("latent", 128, 32, 2041, 70, 16, 1), ("latent", 128, 32, 1301, 0, 24, 1),
    ("latent", 64, 64, 1000, 0, 16, 1), ("latent", 64, 64, 2041, 0, 16, 1), ("latent", 64, 64, 1301, 0, 24, 1),
    ("latent", 64, 32, 700, 0, 4, 1), ("latent", 64, 32, 2041, 0, 24, 1),
    ("gqa", 128, 0, 1000, 0, 16, 4), ("gqa", 128, 0, 2041, 0, 16, 4), ("gqa", 128, 0, 100, 20, 8, 4),
    ("gqa", 64, 0, 500, 0, 8, 4), ("gqa", 64, 0, 1999, 0, 16, 4), ("gqa", 64, 0, 1601, 0, 32, 4), ("gqa", 64, 0, 100, 20, 8, 4)])
def test_prompt_kernels(ti, kind, dim, rot, M, pos0, heads, group):
    """Bound as above."""
    sink = torch.randn(heads, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    out, w, v = prompt(ti, kind, dim, M, pos0, heads, 2.0, sink, rot, group)
    ref = w @ v
    assert (out.transpose(0, 1).double() - ref).abs().le(2.0**-8 * (w @ v.abs()) + 2.0**-8 * ref.abs() + 1e-6).all()
