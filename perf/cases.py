"""Workloads of the framework, measured through its public entry points.

A case is one pass of a user's program over an engine that it keeps:

* "prompt": the tokens of a prompt go into a stream slot (behind `prefix` tokens already in its cache)
  and the last one's logits come back: what a serving program waits for before the first token.
* "step": one decode step of every stream at its own length, logits back to the program's own sampler.
* "run": requests decoded token by token from an empty state, logits of every step back: how a
  recurrent model is stepped (its state cannot go back, so a pass starts anew).

Models are the ones that the benchmark names (synthetic weights of the architecture), plus a small one
of the test suite's sizes.  Weight formats: int4 / int8 per group of 128, fp16, and blocks of 32 (GGUF
Q4_0 / Q8_0); layer-stack models in bf16 or fp32.
"""
import math

import numpy as np
import torch

import turboinfer_amd as T

# name: (vocab, hidden, layers, heads, kv_heads, head_dim, inter, rope_theta)
LLAMAS = {
    "llama2-7b": (32000, 4096, 32, 32, 32, 128, 11008, 10000.0),
    "tinyllama-1.1b": (32000, 2048, 22, 32, 4, 64, 5632, 10000.0),
    "llama3-8b": (128256, 4096, 32, 32, 8, 128, 14336, 500000.0),
    "small": (512, 256, 2, 4, 2, 64, 512, 10000.0),
    "medium": (4096, 1024, 4, 8, 2, 128, 2816, 10000.0),
}
# name: (vocab, width, layers, loop, mixer, experts, top, ff)
STACKS = {
    "gegepel-2k": (32000, 2048, 6, (2, 5, 2), dict(heads=16, dim=128, rot_dim=64, vdim=128, q_rank=1536, kv_rank=512), 64, 6, 1408),
    "gegepel-1k": (32000, 1024, 8, (2, 6, 2), dict(heads=8, dim=64, rot_dim=32, vdim=64, q_rank=512, kv_rank=256), 32, 4, 768),
}
# name: (vocab, width, ff, attention, mamba2, rglru)
HYBRIDS = {
    "nogitar-1k": (32000, 1024, 4096, dict(heads=8, kv_heads=2, dim=128, vdim=128),
                   dict(heads=32, vdim=64, state=128, groups=1, norm_groups=1, conv=4), dict(width=1280, blocks=10, conv=4)),
    "nogitar-2k": (32000, 2048, 8192, dict(heads=16, kv_heads=4, dim=128, vdim=128),
                   dict(heads=64, vdim=64, state=128, groups=1, norm_groups=1, conv=4), dict(width=2560, blocks=10, conv=4)),
}
EPS, JITTER = 1e-5, 0.1
G32 = T.BITS_G32


def listed():
    return [
        # one user of a small quantized model: the shortest launches, latency first
        dict(name="tinyllama int8 step x1", kind="step", model="tinyllama-1.1b", bits=8, streams=1, length=2048, spread=0),
        # the benchmark's headline: one user, 2048 tokens of context
        dict(name="7b int4 step x1", kind="step", model="llama2-7b", bits=4, streams=1, length=2048, spread=0),
        # a full server of 7B requests: attention over 64 caches beside 64-row products
        dict(name="7b int4 step x64", kind="step", model="llama2-7b", bits=4, streams=64, length=2048, spread=0),
        # long contexts under grouped queries, requests of different age
        dict(name="llama3-8b int4 step x32 long", kind="step", model="llama3-8b", bits=4, streams=32, length=8192, spread=4096),
        # a batch of a quantized model that is no multiple of a tile, ragged lengths
        dict(name="tinyllama int8 step x24", kind="step", model="tinyllama-1.1b", bits=8, streams=24, length=1400, spread=700),
        # time to the first token of an ordinary prompt
        dict(name="7b int4 prompt 512", kind="prompt", model="llama2-7b", bits=4, length=512, prefix=0),
        # an odd prompt length on int8 weights
        dict(name="tinyllama int8 prompt 1000", kind="prompt", model="tinyllama-1.1b", bits=8, length=1000, prefix=0),
        # an unquantized checkpoint (the C++ API's default for floating weights): a chat turn behind a cached prefix
        dict(name="tinyllama fp16 prompt 333", kind="prompt", model="tinyllama-1.1b", bits=16, length=333, prefix=600),
        # layer-stack models: a long prompt and a batch step with routed experts
        dict(name="gegepel-2k prompt 2048", kind="prompt", model="gegepel-2k", dtype="bfloat16", length=2048, prefix=0),
        dict(name="gegepel-2k step x16", kind="step", model="gegepel-2k", dtype="bfloat16", streams=16, length=512, spread=200),
        # recurrent layers: an odd prompt and short requests stepped from an empty state
        dict(name="nogitar-2k prompt 1500", kind="prompt", model="nogitar-2k", dtype="bfloat16", length=1500, prefix=0),
        dict(name="nogitar-2k run x8", kind="run", model="nogitar-2k", dtype="bfloat16", streams=8, length=8),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: every model, format and direction; sizes log-uniform, rarely round."""
    what = rng.choice(["llama", "llama", "llama", "stack", "stack", "blocks"])
    if what == "llama":
        model = rng.choice(["small", "medium", "tinyllama-1.1b", "tinyllama-1.1b", "llama2-7b", "llama3-8b"])
        c = dict(model=model, bits=4 if model == "llama3-8b" else rng.choice([4, 8, 16]))
        big = model.startswith("llama")
        if rng.random() < 0.5:
            return dict(c, kind="prompt", length=_spread(rng, 2, 440 if big else 1500), prefix=rng.choice([0, 0, _spread(rng, 1, 500)]))
        n = _spread(rng, 1, 64)
        length = _spread(rng, 8, 2048)
        return dict(c, kind="step", streams=n, length=length, spread=rng.choice([0, length // 2]))
    if what == "blocks":
        c = dict(model="medium", bits=rng.choice([4, 8]) | G32)
        if rng.random() < 0.5:
            return dict(c, kind="prompt", length=_spread(rng, 2, 1500), prefix=0)
        return dict(c, kind="step", streams=_spread(rng, 1, 64), length=_spread(rng, 8, 2048), spread=0)
    if rng.random() < 0.5:
        c = dict(model=rng.choice(["gegepel-1k", "gegepel-2k"]), dtype=rng.choice(["bfloat16", "bfloat16", "float32"]))
        if rng.random() < 0.5:
            return dict(c, kind="step", streams=_spread(rng, 1, 32), length=_spread(rng, 8, 500), spread=0)
    else:
        c = dict(model=rng.choice(["nogitar-1k", "nogitar-2k"]), dtype=rng.choice(["bfloat16", "bfloat16", "float32"]))
        if rng.random() < 0.5:
            return dict(c, kind="run", streams=_spread(rng, 1, 32), length=_spread(rng, 2, 8))
    return dict(c, kind="prompt", length=_spread(rng, 2, 2048 if c["dtype"] == "bfloat16" else 700), prefix=0)


# ------------------------------------------------------------------ inputs
def stack_config(name):
    if name in HYBRIDS:
        V, W, ff, at, ma, rg = HYBRIDS[name]
        at = dict(at, scale=at["dim"] ** -0.5, q_temp=dict(coef=0.1, every=1024))
        mlp = dict(kind="dense", ff=ff)
        layers = []
        for i in range(3):
            layers += [dict(type="rglru", mixer=rg, mlp=mlp), dict(type="mamba2", mixer=ma, mlp=None),
                       dict(type="attention", mixer=dict(at, kv_from=2) if i == 1 else at, mlp=mlp)]
        return dict(architecture="Nogitar", vocab=V, width=W, norm=dict(eps=EPS), layers=layers,
                    embedding=dict(scale=1.0, bigram=dict(buckets=65521, mul_prev=31337, mul_cur=1009)))
    V, W, n, (l0, l1, t), mx, E, top, ff = STACKS[name]
    mixer = dict(mx, rot=dict(base=10000.0, dims=mx["rot_dim"]), scale=(mx["dim"] + mx["rot_dim"]) ** -0.5)
    layer = dict(type="latent_attention", mixer=mixer, mlp=dict(kind="moe", expert=dict(ff=ff), router=dict(experts=E, top=top)))
    return dict(architecture="Gegepel", vocab=V, width=W, embedding=dict(scale=1.0), norm=dict(eps=EPS), layers=[layer] * n,
                loop=dict(start=l0, stop=l1, times=t))


def _sizes(case):
    """Vocabulary, streams, tokens of a pass and each stream's tokens in the cache before it."""
    model = case["model"]
    vocab = (LLAMAS.get(model) or STACKS.get(model) or HYBRIDS.get(model))[0]
    if case["kind"] == "prompt":
        return vocab, 1, case["length"], [case["prefix"]]
    if case["kind"] == "run":
        return vocab, case["streams"], case["length"], [0] * case["streams"]
    before = [max(0, case["length"] - 1 - (s * 389) % (case["spread"] + 1)) for s in range(case["streams"])]
    return vocab, case["streams"], 1, before


def _tokens(case, seed):
    """(tokens of the pass [streams][n], tokens that a layer-stack model has in its cache before it)."""
    vocab, streams, n, before = _sizes(case)
    r = np.random.RandomState((seed * 7919 + 17) % (1 << 31))
    now = r.randint(0, vocab, (streams, n)).astype(np.int32)
    return now, [r.randint(0, vocab, b).astype(np.int32) for b in before]


def _blocks(case, seed):
    """Group-32 weights as a GGUF file holds them: (slot, layer, q int8 [K][N], d fp16 [K/32][N]) of every product."""
    V, H, layers, heads, kv, hd, inter, _ = LLAMAS[case["model"]]
    r = np.random.default_rng(seed + 5)
    top = 7 if case["bits"] & 15 == 4 else 127
    shapes = [(T.W_Q, H, heads * hd), (T.W_K, H, kv * hd), (T.W_V, H, kv * hd), (T.W_O, heads * hd, H), (T.W_GATE, H, inter),
              (T.W_UP, H, inter), (T.W_DOWN, inter, H)]
    for i in range(layers + 1):
        for slot, K, N in shapes if i < layers else [(T.W_LM_HEAD, H, V)]:
            q = r.integers(-top, top + 1, (K, N), dtype=np.int8)
            d = (math.sqrt(3.0 / K) / top * r.uniform(0.5, 1.5, (K // 32, N))).astype(np.float16)
            yield slot, i if i < layers else 0, q, d


def _vectors(case, seed):
    """Norms and embedding of a group-32 model, which comes without the synthetic generator."""
    V, H, layers = LLAMAS[case["model"]][:3]
    r = np.random.default_rng(seed + 6)
    norms = (1 + JITTER * r.uniform(-1, 1, (2 * layers + 1, H))).astype(np.float32)
    return norms, r.uniform(-0.02, 0.02, (V, H)).astype(np.float16).astype(np.float32)


ROUTER, GAIN = 3.0, 0.1


def _trained(name, seed, rows, cols):
    """Tensors of a mixture-of-experts model that random values of unit scale would misstate, or None: a trained
    router's scores are peaked, and post-norm gains are small in deep models (a layer refines the residual, it
    does not replace it).  So a token whose last chosen expert ties with the next one is hardly changed by the
    choice."""
    if not name.endswith((".norm1b", ".norm2b", ".router")):
        return None
    r = np.random.RandomState((seed * 31 + sum(map(ord, name)) + 64 * int(name[1 : name.index(".")])) % (1 << 31))
    if cols > 1:
        return (r.uniform(-1, 1, (rows, cols)) * ROUTER * math.sqrt(3.0 / cols)).astype(np.float32)
    return (GAIN * r.uniform(0.5, 1.5, rows)).astype(np.float32)


def prepare(case, seed):
    _, streams, n, before = _sizes(case)
    now, past = _tokens(case, seed)
    seq = max(before) + n
    seq += -seq % 128
    if case["model"] in LLAMAS:
        V, H, layers, heads, kv, hd, inter, theta = LLAMAS[case["model"]]
        e = T.Engine(V, H, layers, heads, kv, hd, inter, bits=case["bits"], max_seq=seq, max_batch=streams, rope_theta=theta, eps=EPS)
        if case["bits"] & G32:
            for slot, layer, q, d in _blocks(case, seed):
                e.set_tensor_q(slot, layer, q, d)
            norms, emb = _vectors(case, seed)
            for i in range(layers):
                e.set_tensor(T.V_ATTN_NORM, i, norms[2 * i])
                e.set_tensor(T.V_FFN_NORM, i, norms[2 * i + 1])
            e.set_tensor(T.V_OUT_NORM, 0, norms[2 * layers])
            e.set_tensor(T.E_EMBED, 0, emb)
        else:
            e.synth(seed, JITTER)
        for s, b in enumerate(before):
            if b:
                e.fill_kv(s, b, seed + 1000 + s)
    else:
        e = T.Engine.stack(stack_config(case["model"]), case["dtype"], max_seq=seq, max_batch=streams)
        e.synth(seed, JITTER)
        for name, rows, cols in e.weights():
            w = _trained(name, seed, rows, cols)
            if w is not None:
                e.set_weight(name, w)
        for s, t in enumerate(past):
            if t.size:
                e.prefill(s, t)
    return dict(kind=case["kind"], engine=e, tokens=now, pos=np.asarray(before, np.int32))


def run(state):
    e, tok, pos = state["engine"], state["tokens"], state["pos"]
    if state["kind"] == "prompt":
        return e.prefill(0, tok[0], pos0=int(pos[0]))
    return [e.step(np.ascontiguousarray(tok[:, i]), pos + i) for i in range(tok.shape[1])]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    V, streams, n, before = _sizes(case)
    rows = streams * n
    es = 2 if case.get("dtype", "bfloat16") == "bfloat16" else 4
    kv_bytes = flops = 0
    steps = 1 if case["kind"] != "run" else n   # times the weights are read
    heads_rows = rows if case["kind"] != "prompt" else 1
    keys = sum(b * n + n * (n + 1) / 2 for b in before)   # (query, key) pairs of one head
    if case["model"] in LLAMAS:
        _, H, L, nh, nkv, hd, I, _ = LLAMAS[case["model"]]
        bits = case["bits"] & 31 if not case["bits"] & G32 else case["bits"] & 15
        per = H * (2 * nh + 2 * nkv) * hd + 3 * H * I
        group = 32 if case["bits"] & G32 else 128
        weights = (L * per + H * V) * (bits / 8 + (2 / group if bits < 16 else 0))
        kv_bytes = L * 4 * nkv * hd * (sum(before) + rows)
        flops = 2 * rows * L * per + 2 * heads_rows * H * V + 4 * L * nh * hd * keys
    elif case["model"] in STACKS:
        _, W, n_l, (l0, l1, t), mx, E, top, ff = STACKS[case["model"]]
        runs = n_l + (t - 1) * (l1 - l0)
        qd = mx["heads"] * (mx["dim"] + mx["rot_dim"])
        mix = W * (mx["q_rank"] + mx["kv_rank"] + mx["rot_dim"] + mx["heads"] * (mx["vdim"] + 1)) + mx["q_rank"] * qd + \
            mx["kv_rank"] * mx["heads"] * (mx["dim"] + mx["vdim"])
        used = E * (1 - (1 - top / E) ** (rows / steps))   # experts that the rows of a step reach
        weights = es * (runs * (mix + E * W + used * 3 * W * ff) + W * V + 2 * W * W * t)
        kv_bytes = runs * es * (mx["kv_rank"] + mx["rot_dim"]) * (sum(before) + rows)
        flops = 2 * rows * (runs * (mix + E * W + top * 3 * W * ff) + 2 * W * W * t) + 2 * heads_rows * W * V + \
            2 * runs * mx["heads"] * (mx["dim"] + mx["rot_dim"] + mx["vdim"]) * keys
    else:
        _, W, ff, at, ma, rg = HYBRIDS[case["model"]]
        inner, w = ma["heads"] * ma["vdim"], rg["width"]
        cin = inner + 2 * ma["groups"] * ma["state"]
        kvd = at["kv_heads"] * (at["dim"] + at["vdim"])
        hq = at["heads"] * at["dim"]
        per = 3 * (W * (inner + cin + ma["heads"]) + W * inner + 3 * W * w + 2 * w * w / rg["blocks"] + 4 * W * ff + 3 * W * hq) + 2 * W * kvd
        weights = es * (per + W * V)
        state = 3 * 4 * (inner * ma["state"] + w)
        kv_bytes = 2 * streams * steps * state + 3 * es * kvd * keys / max(1, n if steps == 1 else 1)
        flops = 2 * rows * per + 2 * heads_rows * W * V + 3 * 2 * at["heads"] * (at["dim"] + at["vdim"]) * keys + \
            3 * 6 * rows * inner * ma["state"]
    return {"bytes": steps * weights + kv_bytes + 4 * heads_rows * V + 4 * rows, "flops": flops}


def tolerance(case):
    # logits behind 16-bit activations and products.  Measured against exact(): llama models 1e-3 (prompts) to
    # 3e-3 (steps over a random cache); bf16 3e-3 (gegepel) to 8e-3 (nogitar); fp32 1e-6 to 1.3e-5.  Between the
    # prompt's and the steps' kernels as much.  A routed expert that ties to rounding and falls the other way
    # moves a token's logits by up to 2e-2.
    if case.get("dtype") == "float32":
        return {"rel": 5e-5}
    return {"rel": 1e-2 if case["model"] in LLAMAS else 3e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _signed(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _mix(x):
    def down(v, n):
        return (v >> n) & ((1 << (64 - n)) - 1)
    z = x + _signed(0x9E3779B97F4A7C15)
    z = (z ^ down(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ down(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ down(z, 31)


def _unit(seed, tid, shape):
    """The synthetic generator's values in [-1, 1) of tensor `tid`, fp32 (24 random bits, exact)."""
    n = int(np.prod(shape))
    stream = _mix(torch.tensor(_signed(seed ^ (tid * 0xD1B54A32D192ED03)), dtype=torch.int64, device=_dev()))
    h = _mix(torch.arange(n, dtype=torch.int64, device=_dev()) + stream)
    return ((((h >> 40) & 0xFFFFFF) * 2 - (1 << 24)).to(torch.float32) * (1.0 / (1 << 24))).reshape(shape)


def _quantized(w, bits):
    """w fp32 [K][N] as its format holds it, fp64: symmetric per group of 128 along K with fp16 scales, or fp16."""
    if bits == 16:
        return w.half().double()
    K, N = w.shape
    g = w.reshape(K // 128, 128, N)
    s = g.abs().amax(1, keepdim=True) / (7.0 if bits == 4 else 127.0)
    v = (g / s).double()
    q = torch.copysign(torch.floor(v.abs() + 0.5), v).clamp(-7 if bits == 4 else -128, 7 if bits == 4 else 127)
    return (q * s.half().double()).reshape(K, N)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _exact_llama(case, seed):
    V, H, layers, heads, kvh, hd, inter, theta = LLAMAS[case["model"]]
    _, streams, n, before = _sizes(case)
    now = torch.from_numpy(_tokens(case, seed)[0].astype(np.int64)).to(_dev())
    bits, group = case["bits"], heads // kvh
    if bits & G32:
        held = {(s, i): (q, d) for s, i, q, d in _blocks(case, seed)}
        norms, emb = (torch.from_numpy(v).to(_dev()).double() for v in _vectors(case, seed))

        def weight(slot, i, K, N):
            q, d = (torch.from_numpy(v).to(_dev()).double() for v in held[slot, i])
            return (q.reshape(K // 32, 32, N) * d[:, None]).reshape(K, N)

        def norm(i):
            return norms[i]
    else:
        tid = {T.W_Q: 2, T.W_K: 3, T.W_V: 4, T.W_O: 5, T.W_GATE: 6, T.W_UP: 7, T.W_DOWN: 8}
        emb = (_unit(seed, 1, (V, H)) * np.float32(0.02).item()).half().double()

        def weight(slot, i, K, N):
            amp = (np.sqrt(np.float32(3.0)) / np.sqrt(np.float32(K))).item()
            return _quantized(_unit(seed, 3 if slot == T.W_LM_HEAD else 16 + 16 * i + tid[slot], (K, N)) * amp, bits)

        def norm(i):
            return (1.0 + np.float32(JITTER).item() * _unit(seed, 2 if i == 2 * layers else 16 + 16 * (i // 2) + i % 2, (H,))).double()

    freq = theta ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64, device=_dev()) / hd)
    pos = torch.tensor(before, dtype=torch.float64, device=_dev())[:, None] + torch.arange(n, device=_dev())
    ang = (pos[:, :, None] * freq).reshape(-1, 1, hd // 2)

    def rope(v, h):
        v = v.reshape(-1, h, hd // 2, 2)
        a, b = v[..., 0], v[..., 1]
        return torch.stack([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1).reshape(streams, n, h, hd)

    x = emb[now.reshape(-1)]
    for i in range(layers):
        y = _rms(x, norm(2 * i))
        q = rope(y @ weight(T.W_Q, i, H, heads * hd), heads)
        k = rope(y @ weight(T.W_K, i, H, kvh * hd), kvh)
        v = (y @ weight(T.W_V, i, H, kvh * hd)).reshape(streams, n, kvh, hd)
        att = torch.empty(streams, n, heads * hd, dtype=torch.float64, device=_dev())
        for s, b in enumerate(before):
            ks, vs = k[s], v[s]
            if b:
                ks, vs = (torch.cat([_unit(seed + 1000 + s, 0x100000 + 2 * i + j, (b, kvh, hd)).half().double(), c]) for j, c in enumerate((ks, vs)))
            qs = q[s].reshape(n, kvh, group, hd).permute(1, 2, 0, 3).reshape(kvh, group * n, hd)
            sc = (qs @ ks.permute(1, 2, 0).contiguous() / math.sqrt(hd)).reshape(kvh, group, n, b + n)
            if n > 1:
                sc = sc.masked_fill(torch.ones(n, b + n, dtype=torch.bool, device=_dev()).triu(b + 1), -math.inf)
            o = torch.softmax(sc, -1).reshape(kvh, group * n, b + n) @ vs.permute(1, 0, 2).contiguous()
            att[s] = o.reshape(kvh, group, n, hd).permute(2, 0, 1, 3).reshape(n, heads * hd)
        x = x + att.reshape(-1, heads * hd) @ weight(T.W_O, i, heads * hd, H)
        y = _rms(x, norm(2 * i + 1))
        y = torch.nn.functional.silu(y @ weight(T.W_GATE, i, H, inter)) * (y @ weight(T.W_UP, i, H, inter))
        x = x + y @ weight(T.W_DOWN, i, inter, H)
    x = x.reshape(streams, n, H)[:, -1]
    return _rms(x, norm(2 * layers)) @ weight(T.W_LM_HEAD, 0, H, V)


def _stack_names(cfg):
    """[(name, rows, columns)] in the order in which the synthetic generator counts the tensors."""
    W, sandwich = cfg["width"], cfg["architecture"] == "Gegepel"
    out = [("embed", cfg["vocab"], W)]
    if not sandwich:
        out.append(("bigram", cfg["embedding"]["bigram"]["buckets"] + 1, W))
    if cfg.get("loop"):
        out += [("loop.in", W, 2 * W), ("loop.step", cfg["loop"]["times"], W)]
    for i, l in enumerate(cfg["layers"]):
        p, mx = "l%d." % i, l["mixer"]
        for nm in ("norm1", "norm1b", "norm2", "norm2b") if sandwich else ("norm1", "norm2"):
            if l["mlp"] or nm[4] == "1":
                out += [(p + nm, W, 1)] + ([(p + nm + ".b", W, 1)] if sandwich else [])
        m = p + "mix."
        if l["type"] == "latent_attention":
            h, d, r, qr, kr = mx["heads"], mx["dim"], mx["rot_dim"], mx["q_rank"], mx["kv_rank"]
            out += [(m + "dq", qr, W), (m + "dq.norm", qr, 1), (m + "uq", h * (d + r), qr), (m + "dkv", kr + r, W), (m + "dkv.norm", kr, 1),
                    (m + "uk", h * d, kr), (m + "uv", h * mx["vdim"], kr), (m + "sink", h, 1), (m + "g", h, W), (m + "o", W, h * mx["vdim"])]
        elif l["type"] == "attention":
            h, g, d, dv = mx["heads"], mx["kv_heads"], mx["dim"], mx["vdim"]
            out += [(m + "q", h * d, W), (m + "q.norm", h * d, 1)]
            if "kv_from" not in mx:
                out += [(m + "k", g * d, W), (m + "k.norm", g * d, 1), (m + "v", g * dv, W)]
            out += [(m + "g", h * dv, W), (m + "o", W, h * dv)]
        elif l["type"] == "mamba2":
            h, inner = mx["heads"], mx["heads"] * mx["vdim"]
            cin = inner + 2 * mx["groups"] * mx["state"]
            out += [(m + "in", inner + cin + h, W), (m + "conv", cin, mx["conv"]), (m + "conv.b", cin, 1), (m + "dt_bias", h, 1),
                    (m + "A_log", h, 1), (m + "D", h, 1), (m + "norm", inner, 1), (m + "o", W, inner)]
        else:
            w, bw = mx["width"], mx["width"] // mx["blocks"]
            out += [(m + "y", w, W), (m + "y.b", w, 1), (m + "x", w, W), (m + "x.b", w, 1), (m + "conv", w, mx["conv"]), (m + "conv.b", w, 1),
                    (m + "ra", w, bw), (m + "ra.b", mx["blocks"], bw), (m + "ri", w, bw), (m + "ri.b", mx["blocks"], bw), (m + "lam", w, 1),
                    (m + "o", W, w)]
        if l["mlp"] and l["mlp"]["kind"] == "dense":
            out += [(p + "mlp.up", l["mlp"]["ff"], W), (p + "mlp.down", W, l["mlp"]["ff"])]
        elif l["mlp"]:
            out.append((p + "mlp.router", l["mlp"]["router"]["experts"], W))
            for e in range(l["mlp"]["router"]["experts"]):
                ff = l["mlp"]["expert"]["ff"]
                out += [("%smlp.e%d.%s" % (p, e, t), *s) for t, s in (("gate", (ff, W)), ("up", (ff, W)), ("down", (W, ff)))]
    return out + [("final.norm", W, 1)] + ([("final.norm.b", W, 1)] if sandwich else []) + [("head", cfg["vocab"], W)]


def _stack_weights(cfg, seed, dtype):
    """name -> fp64 tensor as the engine holds it, made when asked for."""
    order = {n: (i, r, c) for i, (n, r, c) in enumerate(_stack_names(cfg))}

    def get(name):
        i, r, c = order[name]
        w = _trained(name, seed, r, c)
        if w is not None:
            w = torch.from_numpy(w).to(_dev())
            return (w if dtype == "float32" or c == 1 else w.bfloat16()).double()
        u = _unit(seed, 1000 + i, (r, c))
        if c == 1:
            add = 0.0 if name.endswith(".b") or name.endswith(".sink") else 1.0
            return (add + np.float32(JITTER).item() * u).double().reshape(r)
        s = 1.7320508 if name == "embed" else 0.1 if name == "loop.step" else math.sqrt(3.0 / c)
        w = u * np.float32(s).item()
        kept = name == "loop.step" or name.endswith(".conv") or name.endswith(".b")
        return (w if dtype == "float32" or kept else w.bfloat16()).double()
    return get


def _sequences(case, seed):
    now, past = _tokens(case, seed)
    return [torch.from_numpy(np.concatenate([p, t]).astype(np.int64)).to(_dev()) for p, t in zip(past, now)]


def _each(seqs, x, f):
    """f over each sequence's rows of x."""
    return torch.cat([f(v) for v in x.split([len(s) for s in seqs])])


def _exact_gegepel(case, seed):
    cfg = stack_config(case["model"])
    get, mx, ml = _stack_weights(cfg, seed, case["dtype"]), cfg["layers"][0]["mixer"], cfg["layers"][0]["mlp"]
    H, d, r, dv, kr, top = mx["heads"], mx["dim"], mx["rot_dim"], mx["vdim"], mx["kv_rank"], ml["router"]["top"]
    seqs = _sequences(case, seed)
    pos = torch.cat([torch.arange(len(s), device=_dev()) for s in seqs])
    half = mx["rot"]["dims"] // 2
    ang = pos[:, None].double() * mx["rot"]["base"] ** (-torch.arange(half, dtype=torch.float64, device=_dev()) / half)

    def layer_norm(x, n):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], get(n), get(n + ".b"), EPS)

    def turn(v):
        a, b = v[..., :half], v[..., half:]
        c, s = (f(ang).reshape(-1, *[1] * (v.dim() - 2), half) for f in (torch.cos, torch.sin))
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    def attention(h, p):
        q = (_rms(h @ get(p + "dq").T, get(p + "dq.norm")) @ get(p + "uq").T).reshape(-1, H, d + r)
        kv = h @ get(p + "dkv").T
        c = _rms(kv[:, :kr], get(p + "dkv.norm"))
        q = torch.cat([q[..., :d], turn(q[..., d:])], -1)
        k = torch.cat([(c @ get(p + "uk").T).reshape(-1, H, d), turn(kv[:, kr:])[:, None].expand(-1, H, -1)], -1)
        v = (c @ get(p + "uv").T).reshape(-1, H, dv)
        sink, at = get(p + "sink"), 0
        outs = []
        for s in seqs:
            t = len(s)
            qs, ks, vs = (z[at : at + t].permute(1, 0, 2).contiguous() for z in (q, k, v))
            sc = (qs @ ks.transpose(1, 2).contiguous()) * mx["scale"]
            sc = sc.masked_fill(torch.ones(t, t, dtype=torch.bool, device=_dev()).triu(1), -math.inf)
            pr = torch.softmax(torch.cat([sc, sink[:, None, None].expand(H, t, 1)], -1), -1)[..., :-1]
            outs.append((pr.contiguous() @ vs).permute(1, 0, 2))
            at += t
        o = torch.cat(outs) * torch.sigmoid(h @ get(p + "g").T)[:, :, None]
        return o.reshape(-1, H * dv) @ get(p + "o").T

    def moe(h, p):
        sc, idx = torch.softmax(h @ get(p + "router").T, -1).topk(top, -1)
        out = torch.zeros_like(h)
        for e in range(ml["router"]["experts"]):
            t, k = torch.nonzero(idx == e, as_tuple=True)
            if t.numel():
                y = torch.nn.functional.silu(h[t] @ get("%se%d.gate" % (p, e)).T) * (h[t] @ get("%se%d.up" % (p, e)).T)
                out.index_add_(0, t, sc[t, k][:, None] * (y @ get("%se%d.down" % (p, e)).T))
        return out

    lp, n = cfg["loop"], len(cfg["layers"])
    order = [(i, None) for i in range(lp["start"])]
    for t in range(lp["times"]):
        order += [(i, t if i == lp["start"] else None) for i in range(lp["start"], lp["stop"])]
    x = x0 = get("embed")[torch.cat(seqs)] * cfg["embedding"]["scale"]
    for i, t in order + [(i, None) for i in range(lp["stop"], n)]:
        if t is not None:
            x = torch.cat([x, x0], -1) @ get("loop.in").T + get("loop.step")[t]
        p = "l%d." % i
        x = x + layer_norm(attention(layer_norm(x, p + "norm1"), p + "mix."), p + "norm1b")
        x = x + layer_norm(moe(layer_norm(x, p + "norm2"), p + "mlp."), p + "norm2b")
    last = torch.cumsum(torch.tensor([len(s) for s in seqs]), 0) - 1
    return layer_norm(x[last.to(_dev())], "final.norm") @ get("head").T


def _exact_nogitar(case, seed):
    cfg = stack_config(case["model"])
    get, W, seqs = _stack_weights(cfg, seed, case["dtype"]), cfg["width"], _sequences(case, seed)
    S, t = len(seqs), len(seqs[0])   # (the cases step or prompt all requests from the start: one length)
    bg = cfg["embedding"]["bigram"]
    tok = torch.stack(seqs)
    pair = (tok[:, :-1] * bg["mul_prev"] + tok[:, 1:] * bg["mul_cur"]) % bg["buckets"]
    pair = torch.cat([torch.full((S, 1), bg["buckets"], dtype=torch.int64, device=_dev()), pair], 1)
    e = torch.arange(W, device=_dev())
    ang = torch.arange(t, dtype=torch.float64, device=_dev())[:, None] * 10000.0 ** (-2.0 * (e // 2).double() / W)
    x = get("embed")[tok] * cfg["embedding"]["scale"] + get("bigram")[pair] + torch.where(e % 2 == 1, ang.cos(), ang.sin())
    zero = torch.zeros(W, dtype=torch.float64, device=_dev())
    sigmoid, silu, softplus = torch.sigmoid, torch.nn.functional.silu, torch.nn.functional.softplus

    def conv(v, p):
        w, taps = get(p + "conv"), cfg["layers"][0]["mixer"]["conv"]
        v = torch.cat([v.new_zeros(S, taps - 1, v.shape[-1]), v], 1)
        return sum(w[:, j] * v[:, j : j + t] for j in range(taps)) + get(p + "conv.b")

    def attention(h, p, mx, kv):
        H, G = mx["heads"], mx["kv_heads"]
        q = _rms(h @ get(p + "q").T, get(p + "q.norm"))
        at = torch.arange(t, dtype=torch.float64, device=_dev())
        q = q * (1 + mx["q_temp"]["coef"] * torch.log(torch.floor((at + 1) / mx["q_temp"]["every"]) + 1))[:, None]
        q = q.reshape(S, t, H, -1).transpose(1, 2).contiguous()
        k, v = (z.reshape(S, t, G, -1).transpose(1, 2).repeat_interleave(H // G, 1) for z in kv)
        sc = (q @ k.transpose(2, 3).contiguous()) * mx["scale"]
        sc = sc.masked_fill(torch.ones(t, t, dtype=torch.bool, device=_dev()).triu(1), -math.inf)
        pr = torch.softmax(torch.cat([sc, sc.new_zeros(S, H, t, 1)], -1), -1)[..., :-1]
        o = (pr.contiguous() @ v.contiguous()).transpose(1, 2).reshape(S, t, -1) * sigmoid(h @ get(p + "g").T)
        return o @ get(p + "o").T

    def mamba2(h, p, mx):
        H, P, N, G = mx["heads"], mx["vdim"], mx["state"], mx["groups"]
        inner = H * P
        z, xbc, dt = (h @ get(p + "in").T).split([inner, inner + 2 * G * N, H], -1)
        xs, B, C = silu(conv(xbc, p)).split([inner, G * N, G * N], -1)
        xs = xs.reshape(S, t, H, P)
        B, C = (v.reshape(S, t, G, N).repeat_interleave(H // G, 2) for v in (B, C))
        dt = softplus(dt + get(p + "dt_bias"), threshold=1e9)
        a, D = torch.exp(-get(p + "A_log").exp() * dt), get(p + "D")
        st, ys = x.new_zeros(S, H, N, P), []
        for i in range(t):
            st = a[:, i, :, None, None] * st + (dt[:, i, :, None] * B[:, i])[..., None] * xs[:, i, :, None]
            ys.append((st * C[:, i, :, :, None]).sum(2) + D[:, None] * xs[:, i])
        y = (torch.stack(ys, 1).reshape(S, t, inner) * silu(z)).reshape(S, t, mx["norm_groups"], -1)
        return (_rms(y, 1.0).reshape(S, t, inner) * get(p + "norm")) @ get(p + "o").T

    def rglru(h, p, mx):
        y = torch.nn.functional.gelu(h @ get(p + "y").T + get(p + "y.b"), approximate="tanh")
        u = conv(h @ get(p + "x").T + get(p + "x.b"), p)
        b, bw = mx["blocks"], mx["width"] // mx["blocks"]
        ub = u.reshape(S * t, b, bw).transpose(0, 1).contiguous()
        r, g = (sigmoid(ub @ get(p + n).reshape(b, bw, bw).transpose(1, 2).contiguous() + get(p + n + ".b")[:, None]).transpose(0, 1).reshape(u.shape)
                for n in ("ra", "ri"))
        la = -8.0 * r * softplus(get(p + "lam"), threshold=1e9)
        a, add = torch.exp(la), torch.sqrt(-torch.expm1(2 * la)) * g * u
        st, out = x.new_zeros(S, u.shape[-1]), []
        for i in range(t):
            st = a[:, i] * st + add[:, i]
            out.append(st)
        return (torch.stack(out, 1) * y) @ get(p + "o").T

    kvs = {}
    for i, l in enumerate(cfg["layers"]):
        p, mx = "l%d." % i, l["mixer"]
        if l["type"] == "attention":
            if "kv_from" not in mx:
                kvs[i] = _rms(x @ get(p + "mix.k").T, get(p + "mix.k.norm")), x @ get(p + "mix.v").T
            y = attention(x, p + "mix.", mx, kvs[mx.get("kv_from", i)])
        else:
            y = (mamba2 if l["type"] == "mamba2" else rglru)(x, p + "mix.", mx)
        x = x + _rms(y, get(p + "norm1"))
        if l["mlp"]:
            y = torch.nn.functional.gelu(x @ get(p + "mlp.up").T) @ get(p + "mlp.down").T
            x = x + _rms(y, get(p + "norm2"))
    x = _rms(x[:, -1:] if case["kind"] == "prompt" else x, get("final.norm") + zero) @ get("head").T
    return [x[:, i] for i in range(x.shape[1])]


def exact(case, seed):
    with torch.no_grad():
        if case["model"] in LLAMAS:
            out = [_exact_llama(case, seed)]
        else:
            out = [_exact_gegepel(case, seed)] if case["model"] in STACKS else _exact_nogitar(case, seed)
        return out[0] if case["kind"] == "prompt" else out
