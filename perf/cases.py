"""The work whose speed this backend is judged by, as cases that can be timed and compared.

Every case is one call (or the two calls of a feed-forward block) that ts5's token loop makes of the
backend, through the entry points of tokenstation5_amd.ts5hip: the feed-forward block of one token, of
a speculative-decoding verify batch and of a prompt chunk; decode attention of one sequence and of a
batch of sequences; a verify batch's attention; a prompt chunk's attention; the output head with its
pick; and whole forward calls of a model. Widths are those of the models in tokenstation5_amd/synth.py
(the 8B, the 48x5120 target, the 0.5B draft) and, in drawn cases, other multiples of the block sizes.

Weights are random GGUF blocks whose values have mean 0 and a standard deviation near 0.02, as trained
matrices have; hidden states, queries and cached keys and values are normally distributed.
`exact` computes the same outputs in float64 with torch alone.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from tokenstation5_amd import synth, ts5hip

Q8_0, Q4_K, Q6_K = synth.Q8_0, synth.Q4_K, synth.Q6_K
TYPES = {"q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
MODELS = {"llama_8b": synth.LLAMA_8B, "target_14b": synth.TARGET_14B, "draft_0p5b": synth.DRAFT_0P5B}
EPS = 1e-5


def listed():
    return [
        # The draft model's feed-forward block of one token: the smallest calls of speculative decoding.
        dict(name="ffn_draft_1", kind="ffn", n_embd=896, n_ff=4864, wtype="q8_0", dtype="q4_k", ntok=1),
        # The 8B's feed-forward block of one token: most of a decode step's bytes.
        dict(name="ffn_8b_1", kind="ffn", n_embd=4096, n_ff=14336, wtype="q4_k", dtype="q4_k", ntok=1),
        # The same for a verify batch: the pending token and four drafts.
        dict(name="ffn_8b_5", kind="ffn", n_embd=4096, n_ff=14336, wtype="q4_k", dtype="q4_k", ntok=5),
        # A short message, or the ragged end of a prompt, on the 48x5120 target.
        dict(name="ffn_14b_37", kind="ffn", n_embd=5120, n_ff=13824, wtype="q4_k", dtype="q4_k", ntok=37),
        # A whole prompt chunk on the 8B.
        dict(name="ffn_8b_256", kind="ffn", n_embd=4096, n_ff=14336, wtype="q4_k", dtype="q4_k", ntok=256),
        # The 8B's output head and greedy pick.
        dict(name="head_8b", kind="head", n_embd=4096, n_vocab=128256, wtype="q6_k", pick="greedy"),
        # One layer's decode attention of one 4k conversation.
        dict(name="attn_1x4097_q8", kind="attn", n_head=32, n_head_kv=8, head_dim=128, batch=1, keys=4097, kv="q8"),
        # The largest decode attention: 16 sequences of up to 32k keys.
        dict(name="attn_16x32768_q8", kind="attn", n_head=32, n_head_kv=8, head_dim=128, batch=16, keys=32768,
             kv="q8"),
        # One layer's attention of a five-token verify batch at 4k keys.
        dict(name="verify_5x4101_q8", kind="verify", n_head=32, n_head_kv=8, head_dim=128, batch=5, keys=4101,
             kv="q8"),
        # One layer's attention of the last chunk of a 4096-token prompt, over the f16 cache that the
        # loader picks where the training context fits.
        dict(name="prompt_256x4096_f16", kind="prompt", n_head=32, n_head_kv=8, head_dim=128, batch=256, keys=4096,
             kv="f16"),
        # A decode step of the 8B in a 4k conversation, logits to the host.
        dict(name="step_8b_4096", kind="model", model="llama_8b", ntok=1, pos=4096, kv="q8"),
        # A new 512-token turn of an 8B conversation whose 3584 earlier tokens are cached.
        dict(name="turn_8b_512", kind="model", model="llama_8b", ntok=512, pos=3584, kv="q8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ffn", "ffn", "ffn", "attn", "attn", "verify", "prompt", "head", "model"])
    if kind == "ffn":
        ntok = rng.choice([1, 1, _log(rng, 2, 16), _log(rng, 17, 256)])
        if rng.random() < 0.25:  # rows that are no whole 256-value blocks are kept in Q8_0
            return dict(kind=kind, n_embd=32 * rng.randint(16, 48), n_ff=256 * rng.randint(6, 24), wtype="q8_0",
                        dtype="q4_k", ntok=ntok)
        n_embd = rng.choice([4096, 5120, 256 * rng.randint(6, 20)])
        return dict(kind=kind, n_embd=n_embd, n_ff=256 * rng.randint(2 * n_embd // 256, 56), wtype="q4_k",
                    dtype="q4_k", ntok=ntok)
    if kind == "head":
        n_embd, wtype = rng.choice([(4096, "q6_k"), (5120, "q6_k"), (896, "q8_0"), (256 * rng.randint(6, 20), "q6_k")])
        return dict(kind=kind, n_embd=n_embd, n_vocab=_log(rng, 32000, 151936 if n_embd < 4096 else 128256),
                    wtype=wtype, pick=rng.choice(["greedy", "top40"]))
    if kind == "model":
        kv = rng.choice(["q8", "f16"])
        if rng.random() < 0.5:
            return dict(kind=kind, model="draft_0p5b", ntok=rng.choice([1, rng.randint(2, 8), _log(rng, 9, 512)]),
                        pos=_log(rng, 16, 3584), kv=kv)
        if rng.random() < 0.5:
            return dict(kind=kind, model="llama_8b", ntok=1, pos=rng.randint(2048, 4096), kv=kv)
        return dict(kind=kind, model="llama_8b", ntok=rng.randint(128, 512), pos=rng.randint(1024, 3584), kv=kv)
    n_head, n_head_kv, head_dim = rng.choice([(32, 8, 128), (32, 8, 128), (40, 8, 128), (14, 2, 64)])
    kv = rng.choice(["q8", "f16"])
    if kind == "attn":
        batch = rng.choice([1, 1, rng.randint(2, 16)])
        keys = _log(rng, 64, 32768 if kv == "q8" or batch < 8 else 16384)
        if n_head == 40 and batch == 1:  # the 48x5120 target speaks in contexts of a 2048-token prompt
            keys = _log(rng, 64, 3840)
    elif kind == "verify":
        batch, keys = rng.randint(2, 16), _log(rng, 64, 16384)
    else:
        batch = _log(rng, 17, 256)
        keys = batch + _log(rng, 16, 8192)
    return dict(kind=kind, n_head=n_head, n_head_kv=n_head_kv, head_dim=head_dim, batch=batch, keys=keys, kv=kv)


# ---- inputs --------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _ctx():
    """The program's context: one stream on the GPU."""
    return ts5hip.Context(0)


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + salt) % (1 << 62))
    return g


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _blocks(t, n, g):
    """n GGUF blocks of type t on the GPU, [n][block bytes], of values with mean 0 and deviation near 0.02."""
    out = torch.randint(0, 256, (n, synth.BLOCK[t][1]), generator=g, device="cuda", dtype=torch.uint8)
    d = 0.5 + torch.rand(n, generator=g, device="cuda")
    if t == Q4_K:  # d * sc * q - 8 d * m with m near 7.5 sc / 8
        d = (d * 1.2e-4).to(torch.float16)
        sc = torch.randint(8, 64, (n, 8), generator=g, device="cuda", dtype=torch.int32)
        m = (sc * 15 + 8) // 16
        out[:, 0:2] = _half_bytes(d)
        out[:, 2:4] = _half_bytes(d.float() * 8)
        out[:, 4:8] = ((sc[:, 0:4] & 63) | ((sc[:, 4:8] >> 4) << 6)).to(torch.uint8)
        out[:, 8:12] = ((m[:, 0:4] & 63) | ((m[:, 4:8] >> 4) << 6)).to(torch.uint8)
        out[:, 12:16] = ((sc[:, 4:8] & 15) | ((m[:, 4:8] & 15) << 4)).to(torch.uint8)
    elif t == Q6_K:  # d * sc * (q - 32)
        out[:, 208:210] = _half_bytes(d * 1.5e-5)
    else:  # d * q
        out[:, 0:2] = _half_bytes(d * 2.7e-4)
    return out


def _weight(t, ne0, ne1, g):
    return _ctx().weight(t, ne0, ne1, _blocks(t, ne0 // synth.BLOCK[t][0] * ne1, g).cpu().numpy())


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std + mean


def _round_q8(x):
    """x [..., 32k] as the q8 cache keeps it: int8 values and an f16 scale per 32 (max / 127, to even)."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    sc = (b.abs().amax(-1) / 127).to(torch.float16)
    s = sc.to(x.dtype).unsqueeze(-1)
    q = torch.where(s > 0, torch.round(b / s), torch.zeros_like(b)).clamp_(-127, 127)
    return q.to(torch.int8).reshape(x.shape), sc


def _cache(case, seed, b, salt):
    """K (salt 0) or V (salt 1) of sequence b: (values, scales) with scales None for f16."""
    shape = (case["n_head_kv"], _slots(case), case["head_dim"])
    x = torch.randn(*shape, generator=_gen(seed, 1000 + 2 * b + salt), device="cuda")
    return _round_q8(x) if case["kv"] == "q8" else (x.to(torch.float16), None)


def _slots(case):
    return -(-case["keys"] // 256) * 256


def _lengths(case):
    """Keys of each sequence: the first has them all, the others end earlier, up to a quarter."""
    return [case["keys"] - b * case["keys"] // (4 * case["batch"]) for b in range(case["batch"])]


def _attn_inputs(case, seed):
    seqs = case["batch"] if case["kind"] == "attn" else 1
    q = _normal(_gen(seed, 1), case["batch"], case["n_head"] * case["head_dim"])
    kv = [[_cache(case, seed, b, salt) for b in range(seqs)] for salt in (0, 1)]
    return q, kv


# A model's matrices are slices of one pool of blocks per type, each from an offset of its own.
POOL_BLOCKS = {Q4_K: 2200000, Q6_K: 2100000, Q8_0: 4400000}


def _tensor_slices(hp):
    """(name, type, ne0, ne1, first block in its pool or None for a norm weight)."""
    for i, (name, t, ne0, ne1) in enumerate(synth.tensor_specs(hp)):
        if t not in POOL_BLOCKS:
            yield name, t, ne0, ne1, None
        else:
            n = ne0 // synth.BLOCK[t][0] * ne1
            yield name, t, ne0, ne1, i * 104729 % (POOL_BLOCKS[t] - n + 1)


def _pools(hp, seed):
    types = {t for _, t, _, _ in synth.tensor_specs(hp)} & set(POOL_BLOCKS)
    return {t: _blocks(t, POOL_BLOCKS[t], _gen(seed, 10 + t)) for t in sorted(types)}


def _norms(hp, seed):
    """Norm weights by name, float32 on the CPU."""
    names = [(name, ne0) for name, _, ne0, _, at in _tensor_slices(hp) if at is None]
    all_ = torch.cat([_normal(_gen(seed, 5000 + i), n, mean=1.0, std=0.02) for i, (_, n) in enumerate(names)]).cpu()
    out, at = {}, 0
    for name, n in names:
        out[name] = all_[at:at + n]
        at += n
    return out


def _model_kv(hp, case, seed, layer, which):
    """A layer's cached K (which 0) or V (1) before the call: [pos][n_head_kv * head_dim]."""
    g = _gen(seed, 9000 + 2 * layer + which)
    return _normal(g, case["pos"], hp["n_head_kv"] * hp["head_dim"])


def _tokens(hp, case, seed):
    return np.random.default_rng([int(seed), 77]).integers(0, hp["n_vocab"], case["ntok"]).astype(np.int32)


def _all_logits(case):
    return 1 < case["ntok"] <= 16  # a verify batch needs every position's


def prepare(case, seed):
    c = _ctx()
    kind = case["kind"]
    s = dict(case, ctx=c)
    if kind == "ffn":
        E, F, n = case["n_embd"], case["n_ff"], case["ntok"]
        s["t"], s["dt"] = TYPES[case["wtype"]], TYPES[case["dtype"]]
        s["gate"], s["up"] = (_weight(s["t"], E, F, _gen(seed, 2 + i)) for i in (0, 1))
        s["down"] = _weight(s["dt"], F, E, _gen(seed, 4))
        s["x"] = _normal(_gen(seed, 1), n, E)
        s["norm"] = _normal(_gen(seed, 5), E, mean=1.0, std=0.02)
        s["h"] = torch.empty(n, F, device="cuda")
        s["y"] = torch.empty(n, E, device="cuda")
    elif kind == "head":
        E, V = case["n_embd"], case["n_vocab"]
        s["t"] = TYPES[case["wtype"]]
        s["w"] = _weight(s["t"], E, V, _gen(seed, 2))
        s["x"] = _normal(_gen(seed, 1), E)
        s["norm"] = _normal(_gen(seed, 5), E, mean=1.0, std=0.02)
        s["y"] = torch.empty(V, device="cuda")
        s["id"] = torch.empty(1, device="cuda", dtype=torch.int32)
        s["vals"] = torch.empty(40, device="cuda")
        s["ids"] = torch.empty(40, device="cuda", dtype=torch.int32)
    elif kind == "model":
        hp = MODELS[case["model"]]
        n_ctx = -(-(case["pos"] + case["ntok"]) // 256) * 256
        m = ts5hip.Model(c, hp, n_ctx, ts5hip.KV_Q8 if case["kv"] == "q8" else ts5hip.KV_F16)
        pools = {t: p.cpu().numpy() for t, p in _pools(hp, seed).items()}
        norms = _norms(hp, seed)
        for name, t, ne0, ne1, at in _tensor_slices(hp):
            if at is None:
                data = norms[name].numpy().view(np.uint8)
            else:
                data = pools[t][at:at + ne0 // synth.BLOCK[t][0] * ne1]
            m.set_tensors({name: (t, ne0, ne1, data)})
        for layer in range(hp["n_layer"]):
            for which in (0, 1):
                m.kv_write(layer, which, 0, _model_kv(hp, case, seed, layer, which).cpu().numpy())
        s["m"], s["tokens"] = m, _tokens(hp, case, seed)
    else:
        q, kv = _attn_inputs(case, seed)
        s["q"], s["out"] = q, torch.empty_like(q)
        for name, seqs in zip("kv", kv):
            s[name] = torch.stack([v for v, _ in seqs])
            s[name + "s"] = torch.stack([sc for _, sc in seqs]) if case["kv"] == "q8" else None
        s["n_ctx"] = _slots(case)
        s["scale"] = 1.0 / math.sqrt(case["head_dim"])
        n = _lengths(case) if kind == "attn" else [case["keys"] - case["batch"]]
        s["n_keys"] = torch.tensor(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    c.sync()
    return s


# ---- one pass ------------------------------------------------------------------------------------

def run(s):
    c, kind = s["ctx"], s["kind"]
    if kind == "ffn":
        E, F, n = s["n_embd"], s["n_ff"], s["ntok"]
        x, h, y, norm = (s[k].data_ptr() for k in ("x", "h", "y", "norm"))
        if n == 1:
            c.matvec_glu(s["t"], s["gate"], s["up"], E, F, x, h, norm, EPS)
            c.matvec(s["dt"], s["down"], F, E, h, y)
        else:
            c.matmul_glu(s["t"], s["gate"], s["up"], E, F, x, n, h, norm, EPS)
            c.matmul(s["dt"], s["down"], F, E, h, n, y)
        return s["h"], s["y"]
    if kind == "head":
        x, y, norm = (s[k].data_ptr() for k in ("x", "y", "norm"))
        if s["pick"] == "greedy":
            c.matvec_argmax(s["t"], s["w"], s["n_embd"], s["n_vocab"], x, y, s["id"].data_ptr(), norm, EPS)
            return s["y"], s["id"]
        c.matvec(s["t"], s["w"], s["n_embd"], s["n_vocab"], x, y, norm, EPS)
        c.topk(y, s["n_vocab"], 40, s["vals"].data_ptr(), s["ids"].data_ptr())
        return s["y"], s["vals"], s["ids"]
    if kind == "model":
        return s["m"].forward(s["tokens"], s["pos"], all_logits=_all_logits(s))
    q, out, k, v = (s[n].data_ptr() for n in ("q", "out", "k", "v"))
    heads = s["n_head"], s["n_head_kv"], s["head_dim"]
    q8 = s["kv"] == "q8"
    ks, vs = (s["ks"].data_ptr(), s["vs"].data_ptr()) if q8 else (None, None)
    if kind == "prompt":
        pos0 = s["keys"] - s["batch"]
        if q8:
            c.attn_prompt(q, s["batch"], *heads, k, ks, v, vs, s["n_ctx"], pos0, s["scale"], out)
        else:
            c.attn_prompt_f16(q, s["batch"], *heads, k, v, s["n_ctx"], pos0, s["scale"], out)
    else:
        per, n = kind == "attn", s["n_keys"].data_ptr()
        if q8:
            c.attn_decode(q, s["batch"], *heads, k, ks, v, vs, s["n_ctx"], n, per, s["scale"], out)
        else:
            c.attn_decode_f16(q, s["batch"], *heads, k, v, s["n_ctx"], n, per, s["scale"], out)
    return s["out"]


# ---- what a pass cannot do without ---------------------------------------------------------------

def _pairs(case):
    """(query, key) pairs of an attention case."""
    if case["kind"] == "attn":
        return sum(_lengths(case))
    return sum(case["keys"] - case["batch"] + t + 1 for t in range(case["batch"]))


def _kv_bytes(n_head_kv, head_dim, kv):
    """Bytes of one key and its value over all KV heads."""
    return n_head_kv * (2 * head_dim + 4 * head_dim // 32 if kv == "q8" else 4 * head_dim)


def work(case):
    kind = case["kind"]
    if kind == "ffn":
        E, F, n = case["n_embd"], case["n_ff"], case["ntok"]
        w = 2 * F * synth.row_bytes(TYPES[case["wtype"]], E) + E * synth.row_bytes(TYPES[case["dtype"]], F)
        return dict(bytes=w + 4 * E + 4 * n * (2 * E + F), flops=6 * n * E * F)
    if kind == "head":
        E, V = case["n_embd"], case["n_vocab"]
        return dict(bytes=V * synth.row_bytes(TYPES[case["wtype"]], E) + 8 * E + 4 * V, flops=2 * E * V)
    if kind == "model":
        hp, n = MODELS[case["model"]], case["ntok"]
        wb, rows = synth.weight_bytes(hp), n if _all_logits(case) else 1
        keys = case["pos"] + n
        E, F, H, HKV, HD, V = (hp[k] for k in ("n_embd", "n_ff", "n_head", "n_head_kv", "head_dim", "n_vocab"))
        values = hp["n_layer"] * E * (2 * H * HD + 2 * HKV * HD + 3 * F)
        pairs = sum(case["pos"] + t + 1 for t in range(n))
        return dict(bytes=wb["layers"] + wb["head"] + wb["norms"] + n * wb["embd_row"] + 4 * rows * V
                    + hp["n_layer"] * keys * _kv_bytes(HKV, HD, case["kv"]),
                    flops=2 * n * values + 2 * rows * E * V + 4 * hp["n_layer"] * pairs * H * HD)
    keys = _pairs(case) if kind == "attn" else case["keys"]
    q = case["batch"] * case["n_head"] * case["head_dim"]
    return dict(bytes=keys * _kv_bytes(case["n_head_kv"], case["head_dim"], case["kv"]) + 8 * q,
                flops=4 * _pairs(case) * case["n_head"] * case["head_dim"])


# Inputs are rounded to 22 or 23 bits and sums run in 32: single blocks are 2e-7 to 8e-7 from float64.
# In a whole model a last-bit difference can also land a new key or value on the other side of a
# rounding step of the cache: one step of one new key among thousands hardly shows (3e-6 to 7e-6 seen),
# a chunk's keys see each other through such steps in every layer (8B: q8 1e-3 to 2e-3, f16 1.5e-4;
# draft: q8 2e-5 to 2e-4, f16 6e-6 to 3e-5).
def tolerance(case):
    if case["kind"] != "model":
        return {"rel": 1e-5}
    if case["ntok"] == 1:
        return {"rel": 1e-4}
    if case["model"] == "llama_8b":
        return {"rel": 8e-3 if case["kv"] == "q8" else 1e-3}
    return {"rel": 1e-3 if case["kv"] == "q8" else 2e-4}


# ---- float64 -------------------------------------------------------------------------------------

def _values(t, b):
    """The float64 values of GGUF blocks b [..., block bytes], [..., values]."""
    def half(at):
        return b[..., at:at + 2].contiguous().view(torch.float16).double()
    if t == Q4_K:
        d, dmin, s = half(0), half(2), b[..., 4:16].int()
        lo, mid, hi = s[..., 0:4], s[..., 4:8], s[..., 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1)
        m = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1)
        n = b[..., 16:144].reshape(*b.shape[:-1], 4, 1, 32)
        q = torch.cat([n & 15, n >> 4], -2).reshape(*b.shape[:-1], 8, 32).double()
        return ((d * sc).unsqueeze(-1) * q - (dmin * m).unsqueeze(-1)).reshape(*b.shape[:-1], 256)
    if t == Q6_K:
        ql = b[..., 0:128].reshape(*b.shape[:-1], 2, 2, 32).int()  # half, low or high 32, byte
        qh = b[..., 128:192].reshape(*b.shape[:-1], 2, 32).int()
        q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | ((qh >> 2 & 3) << 4),
                         (ql[..., 0, :] >> 4) | ((qh >> 4 & 3) << 4), (ql[..., 1, :] >> 4) | ((qh >> 6) << 4)], -2)
        q = (q - 32).reshape(*b.shape[:-1], 16, 16).double()
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        return ((half(208) * sc).unsqueeze(-1) * q).reshape(*b.shape[:-1], 256)
    return half(0) * b[..., 2:34].contiguous().view(torch.int8).double()


def _product(t, blocks, ne0, x):
    """x [n][ne0] times the rows of GGUF blocks [rows * blocks a row][bytes], in float64."""
    per = ne0 // synth.BLOCK[t][0]
    rows = blocks.shape[0] // per
    out = torch.empty(x.shape[0], rows, dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // ne0)
    for r in range(0, rows, step):
        e = min(rows, r + step)
        w = _values(t, blocks[r * per:e * per]).reshape(e - r, ne0)
        out[:, r:e] = x @ w.t().contiguous()
    return out


def _rmsnorm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _cache_values(values, scales):
    if scales is None:
        return values.double()
    return (values.double().reshape(*scales.shape, 32) * scales.double().unsqueeze(-1)).reshape(values.shape)


def _attention(q, k, v, first, scale):
    """q [n][H][HD] over k, v [HKV][keys][HD]; query t sees the first `first` + t + 1 keys."""
    n, H, HD = q.shape
    HKV = k.shape[0]
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[1], device="cuda")[None, :] <= first + torch.arange(n, device="cuda")[:, None]
    for h in range(H):
        kh = h // (H // HKV)
        p = (q[:, h] @ k[kh].t().contiguous()) * scale
        out[:, h] = torch.softmax(p.masked_fill(~seen, -math.inf), -1) @ v[kh]
    return out


def _rope(x, hp, pos):
    """x [n][heads][HD] at positions pos..; angles are float32 products, as the models define them."""
    half = hp["head_dim"] // 2
    e = np.float32(-2) * np.arange(half, dtype=np.float32) / np.float32(hp["head_dim"])
    inv = np.power(float(hp["rope_base"]), e.astype(np.float64)).astype(np.float32)  # float32, correctly rounded
    a = np.arange(pos, pos + x.shape[0], dtype=np.float32)[:, None] * inv[None, :]
    a = torch.from_numpy(a).cuda().double().unsqueeze(1)
    c, s = torch.cos(a), torch.sin(a)
    neox = hp["arch"] == "qwen2"
    u, v = (x[..., :half], x[..., half:]) if neox else (x[..., 0::2], x[..., 1::2])
    u, v = u * c - v * s, u * s + v * c
    return torch.cat([u, v], -1) if neox else torch.stack([u, v], -1).flatten(-2)


def _kept(x, kv):
    """x [..., 32k] as the cache keeps it, back in float64."""
    if kv == "f16":
        return x.float().to(torch.float16).double()
    q, sc = _round_q8(x.float())
    return _cache_values(q, sc)


def _exact_model(case, seed):
    hp = MODELS[case["model"]]
    H, HKV, HD, pos, n = hp["n_head"], hp["n_head_kv"], hp["head_dim"], case["pos"], case["ntok"]
    pools, norms = _pools(hp, seed), _norms(hp, seed)
    spec = {name: (t, ne0, ne1, at) for name, t, ne0, ne1, at in _tensor_slices(hp)}

    def blocks(name):
        t, ne0, ne1, at = spec[name]
        return pools[t][at:at + ne0 // synth.BLOCK[t][0] * ne1]

    def product(name, x):
        return _product(spec[name][0], blocks(name), spec[name][1], x)

    def norm(name, x):
        return _rmsnorm(x, norms[name].cuda(), hp["rms_eps"])

    t, ne0, ne1, _ = spec["token_embd.weight"]
    rows = blocks("token_embd.weight").reshape(ne1, -1, synth.BLOCK[t][1])
    x = _values(t, rows[torch.from_numpy(_tokens(hp, case, seed)).long().cuda()]).reshape(n, ne0)
    for layer in range(hp["n_layer"]):
        p = "blk.%d." % layer
        a = norm(p + "attn_norm.weight", x)
        q = _rope(product(p + "attn_q.weight", a).reshape(n, H, HD), hp, pos)
        k = _kept(_rope(product(p + "attn_k.weight", a).reshape(n, HKV, HD), hp, pos), case["kv"])
        v = _kept(product(p + "attn_v.weight", a).reshape(n, HKV, HD), case["kv"])
        old = [_kept(_model_kv(hp, case, seed, layer, w).reshape(pos, HKV, HD), case["kv"]) for w in (0, 1)]
        k, v = (torch.cat([o, e]).transpose(0, 1).contiguous() for o, e in zip(old, (k, v)))
        o = _attention(q, k, v, pos, 1.0 / math.sqrt(HD))
        x = x + product(p + "attn_output.weight", o.reshape(n, H * HD))
        a = norm(p + "ffn_norm.weight", x)
        g = product(p + "ffn_gate.weight", a)
        x = x + product(p + "ffn_down.weight", g * torch.sigmoid(g) * product(p + "ffn_up.weight", a))
    x = x if _all_logits(case) else x[-1:]
    return product("output.weight" if "output.weight" in spec else "token_embd.weight", norm("output_norm.weight", x))


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _exact_model(case, seed).cpu().numpy()
    if kind == "ffn":
        E, F, n = case["n_embd"], case["n_ff"], case["ntok"]
        t, dt = TYPES[case["wtype"]], TYPES[case["dtype"]]
        norm = _normal(_gen(seed, 5), E, mean=1.0, std=0.02)
        x = _rmsnorm(_normal(_gen(seed, 1), n, E).double(), norm, EPS)
        g, u = (_product(t, _blocks(t, E // synth.BLOCK[t][0] * F, _gen(seed, 2 + i)), E, x) for i in (0, 1))
        h = g * torch.sigmoid(g) * u
        return h, _product(dt, _blocks(dt, F // synth.BLOCK[dt][0] * E, _gen(seed, 4)), F, h)
    if kind == "head":
        E, V, t = case["n_embd"], case["n_vocab"], TYPES[case["wtype"]]
        norm = _normal(_gen(seed, 5), E, mean=1.0, std=0.02)
        x = _rmsnorm(_normal(_gen(seed, 1), E).double(), norm, EPS)
        y = _product(t, _blocks(t, E // synth.BLOCK[t][0] * V, _gen(seed, 2)), E, x[None])[0]
        if case["pick"] == "greedy":
            return y, y.argmax().reshape(1).int()
        top = torch.topk(y, 40)
        return y, top.values, top.indices.int()
    q, kv = _attn_inputs(case, seed)
    H, HD, scale = case["n_head"], case["head_dim"], 1.0 / math.sqrt(case["head_dim"])
    q = q.double().reshape(case["batch"], H, HD)
    if kind != "attn":
        k, v = (_cache_values(*seqs[0])[:, :case["keys"]] for seqs in kv)
        return _attention(q, k, v, case["keys"] - case["batch"], scale).reshape(case["batch"], H * HD)
    rows = []
    for b, n in enumerate(_lengths(case)):
        k, v = (_cache_values(*seqs[b])[:, :n] for seqs in kv)
        rows.append(_attention(q[b:b + 1], k, v, n - 1, scale).reshape(1, H * HD))
    return torch.cat(rows)
