"""The measured workloads of the framework: decode attention over the compressed
cache and the encoders that fill it, through the public entry points
(``BitCache`` and ``bitcache_amd.functional``).

A case is a dict of plain values:
  op        what is called (see ``run``)
  batch, heads, kv_heads, dim, seq   the shape; seq is the number of keys per row
  ring      slots per row of a BitCache (>= seq), where the op has one
  residual  the cache holds INT4 residuals (compensated), else sign bits only
  std       standard deviation of the inputs: 1 for keys and queries of unit
            variance per element, 1/sqrt(128) = 0.0884 for rows of unit norm (the
            named benchmark configurations of bitcache_amd/workloads.py)
"""
from __future__ import annotations

import math

import torch

from bitcache_amd import BitCache, default_top_k, functional as BF
from bitcache_amd import layout

UNIT_NORM = 1.0 / math.sqrt(128.0)

# Share of the work of a drawn case: bytes of keys and values it touches at most
# (the largest listed case touches 2.8 GB).
_DRAWN_BYTES = 400e6


def _case(op, batch, heads, kv_heads, dim, seq, ring=0, residual=True, std=1.0):
    return dict(op=op, batch=batch, heads=heads, kv_heads=kv_heads, dim=dim, seq=seq,
                ring=max(ring, seq), residual=residual, std=std)


def listed():
    return [
        # the shortest calls: one sequence at the start of a chat, one token at a
        # time (latency and launches), and one 4K-token sequence
        dict(name="step_short", **_case("step", 1, 32, 8, 128, 301)),
        dict(name="comp_c1", **_case("attention", 1, 32, 32, 128, 4096, std=UNIT_NORM)),
        # the decode loop of a small served batch: append one token, then attend
        dict(name="step_c4", **_case("step", 4, 32, 8, 128, 16384, std=UNIT_NORM)),
        # binary-only attention (the fast, memory-saving mode), 32K tokens
        dict(name="binary_c2", **_case("attention", 8, 32, 32, 128, 32768, residual=False,
                                       std=UNIT_NORM)),
        # the headline: compensated attention at 64K tokens, 2.8 GB of cache
        dict(name="comp_c3", **_case("attention", 8, 32, 32, 128, 65536, std=UNIT_NORM)),
        # the head dims other models have, over partly filled rings of odd lengths
        dict(name="gqa_d64", **_case("attend", 8, 32, 8, 64, 20011, ring=24576)),
        dict(name="mha_d96", **_case("attend", 2, 32, 32, 96, 9973, ring=12000)),
        dict(name="gqa_d256", **_case("attend", 4, 16, 8, 256, 12345, ring=16384)),
        # residuals only on the top 10% of keys, 128K tokens
        dict(name="adaptive_c5", **_case("adaptive", 16, 32, 8, 128, 131072, std=UNIT_NORM)),
        # binary or compensated per head, chosen from the entropy of its scores
        dict(name="modes_16k", **_case("modes", 4, 32, 32, 128, 16384)),
        # the prompt goes into the cache: K and V as projections leave them, [B, S, H, d]
        dict(name="prefill_c4", **_case("prefill", 4, 32, 8, 128, 16384)),
        # one tensor through the two-step encoder (encode, then compute_residual)
        dict(name="encode_c1", **_case("encode", 1, 32, 32, 128, 4095)),
    ]


def draw(rng):
    """One more case of the same ranges: each op, every head dim, head groupings from
    MHA to 16 query heads per KV head, 16 to 131,072 keys."""
    op = rng.choice(["step", "step", "attention", "attention", "attend", "attend", "adaptive",
                     "modes", "prefill", "encode"])
    dim = rng.choice([128, 128, 128, 128, 64, 64, 96, 96, 256, 256, rng.choice([32, 160, 192, 224])])
    group = rng.choice([1, 1, 1, 2, 4, 4, 4, 8, 8, 3, 16])
    kv_heads = rng.choice([1, 2, 4, 8, 8, 8, 16, 32])
    while kv_heads * group > 64:
        kv_heads //= 2
    batch = int(round(2.0 ** rng.uniform(0.0, 4.0)))
    residual = rng.random() < 0.75 or op in ("adaptive", "modes", "encode")
    per = _vec_bytes(dim, residual) * 2 + (4 * dim if op in ("prefill", "encode") else 0)
    most = max(16, int(_DRAWN_BYTES / (per * batch * kv_heads)))
    seq = int(round(2.0 ** rng.uniform(4.0, math.log2(min(131072, most)))))
    ring = int(seq * rng.uniform(1.0, 1.5)) if op == "attend" else seq
    std = rng.choice([1.0, UNIT_NORM, 0.5])
    if op == "modes":
        std = 1.0   # (the heads' entropies are spread by the queries' scale below)
    return _case(op, batch, kv_heads * group, kv_heads, dim, seq, ring, residual, std)


# ---------------------------------------------------------------- sizes
def _vec_bytes(dim, residual):
    """Bytes of one encoded vector: sign bits and scale, INT4 codes and their scale."""
    return dim // 8 + 2 + ((dim // 2 + 2) if residual else 0)


def work(case):
    B, H, Hkv, d, S = (case[k] for k in ("batch", "heads", "kv_heads", "dim", "seq"))
    vecs = B * Hkv * S                      # of K, and of V
    op, res = case["op"], case["residual"]
    binary, full = _vec_bytes(d, False), _vec_bytes(d, True)
    query = B * H * d * 2 * 2               # queries and outputs, fp16
    token = B * Hkv * (d * 2 + _vec_bytes(d, res)) * 2
    if op in ("prefill", "encode"):
        # read fp16, write the encoded vectors; a few operations per element
        n = 2 if op == "prefill" else 1
        return {"bytes": n * vecs * (2 * d + _vec_bytes(d, res)), "flops": n * vecs * d * 8}
    if op == "adaptive":
        # signs and scales of every key and value; residuals where at least one
        # query head of the group selects the key (as if heads chose independently)
        share = 1.0 - 0.9 ** (H // Hkv)
        read = 2 * vecs * (binary + share * (full - binary))
    elif op == "modes":
        # half of the heads are binary; a KV head's residuals are read when any
        # of its query heads is compensated
        share = 1.0 - 0.5 ** (H // Hkv)
        read = 2 * vecs * (binary + share * (full - binary))
    else:
        read = 2 * vecs * (full if res else binary)
    # scores and weighted sum: 2 operations per element each
    return {"bytes": read + query + (token if op == "step" else 0),
            "flops": 4.0 * B * H * S * d}


# ---------------------------------------------------------------- inputs
def _randn(gen, shape, std):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float16)
    return x if std == 1.0 else x.mul_(std)


def _rows(gen, shape, std, outliers):
    """[..., d] fp16 vectors: normal elements, the rows' magnitudes spread log-normally
    (0.25), as keys and values are along a context; `outliers`: four channels per
    head ten times larger, as keys of trained models have them."""
    x = _randn(gen, shape, std)
    x.mul_(torch.exp(0.25 * torch.randn(shape[:-1] + (1,), generator=gen, device="cuda")).half())
    if outliers:
        B, H, _, d = shape
        for h in range(H):
            for c in torch.randperm(d, generator=gen, device="cuda")[:4].tolist():
                x[:, h, :, c].mul_(10.0)
    return x


def _inputs(case, seed):
    """Q [B, H, d] and K, V [B, Hkv, S, d]; the new token of a step."""
    B, H, Hkv, d, S, std = (case[k] for k in ("batch", "heads", "kv_heads", "dim", "seq", "std"))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    x = {"q": _randn(gen, (B, H, d), std)}
    if case["op"] == "modes":
        # half of the heads look at few keys, the others at many
        sharp = torch.rand((B, H, 1), generator=gen, device="cuda") < 0.5
        x["q"] = torch.where(sharp, x["q"], x["q"] * 0.1)
    outliers = case["op"] == "adaptive"
    x["k"] = _rows(gen, (B, Hkv, S, d), std, outliers)
    x["v"] = _rows(gen, (B, Hkv, S, d), std, outliers)
    if case["op"] == "step":
        x["new_k"] = _randn(gen, (B, Hkv, d), std)
        x["new_v"] = _randn(gen, (B, Hkv, d), std)
    return x


def _threshold(case):
    """Entropy from which a head is attended in binary mode: below the uniform log S
    (flat queries lose about 0.3 of it, sharp ones several nats)."""
    return math.log(case["seq"]) - min(1.5, 0.5 * math.log(case["seq"]))


def prepare(case, seed):
    B, H, Hkv, d, S = (case[k] for k in ("batch", "heads", "kv_heads", "dim", "seq"))
    op = case["op"]
    x = _inputs(case, seed)
    if op == "prefill":
        cache = BitCache(B, H, d, case["ring"], compensated=case["residual"], n_kv_heads=Hkv)
        return dict(case=case, cache=cache, k=x["k"].transpose(1, 2).contiguous(),
                    v=x["v"].transpose(1, 2).contiguous())
    if op == "encode":
        return dict(case=case, src=x["k"].reshape(-1, d))
    if op in ("step", "attend"):
        # a ring as a decode loop has it: filled by a prefill; a step's is full,
        # so that every pass attends over the same number of keys
        cache = BitCache(B, H, d, case["ring"], compensated=case["residual"], n_kv_heads=Hkv)
        cache.prefill(x["k"], x["v"])
        return dict(case=case, cache=cache, q=x["q"], k=x.get("new_k"), v=x.get("new_v"))
    state = dict(case=case, q=x["q"])
    for n in ("k", "v"):
        src = x.pop(n).reshape(-1, d)
        if case["residual"]:
            state[n], state[n + "r"] = BF.encode_fused(src)
        else:
            state[n] = BF.encode(src)
    return state


def _written(blob, dim, residual):
    """The bytes of a blob that its vectors take (the rest of the allocation is unused)."""
    n = layout.capacity(blob, residual)
    return blob[:n * ((dim // 2 if residual else dim // 8) + 2)]


def _cache_bytes(cache):
    planes = [(cache._k_bin, False), (cache._v_bin, False)]
    if cache.compensated:
        planes += [(cache._k_res, True), (cache._v_res, True)]
    return [_written(b, cache.head_dim, r) for b, r in planes]


def run(state):
    case = state["case"]
    op, d = case["op"], case["dim"]
    if op == "step":
        out = state["cache"].append_attend(state["k"], state["v"], state["q"])
        return [out] + _cache_bytes(state["cache"])
    if op == "attend":
        return state["cache"].attend(state["q"])
    if op == "prefill":
        state["cache"].prefill(state["k"], state["v"], layout="bshd")
        return _cache_bytes(state["cache"])
    if op == "encode":
        blob = BF.encode(state["src"])
        res = BF.compute_residual(state["src"], blob)
        return [_written(blob, d, False), _written(res, d, True)]
    shape = (case["batch"], case["heads"], case["seq"], d)
    gqa = {} if case["kv_heads"] == case["heads"] else dict(n_kv_heads=case["kv_heads"])
    if op == "adaptive":
        return BF.adaptive_attention(state["q"], state["k"], state["kr"], state["v"], state["vr"],
                                     *shape, **gqa)
    if op == "modes":
        return BF.entropy_dispatch_attention(state["q"], state["k"], state["kr"], state["v"],
                                             state["vr"], *shape, _threshold(case), **gqa)
    if case["residual"]:
        return BF.compensated_attention(state["q"], state["k"], state["kr"], state["v"],
                                        state["vr"], *shape, **gqa)
    return BF.binary_attention(state["q"], state["k"], state["v"], *shape, **gqa)


# ---------------------------------------------------------------- what is right
def tolerance(case):
    if case["op"] in ("prefill", "encode"):
        return "exact"
    # 2.1e-4 to 2.8e-4 against 64 bits, most of it the rounding of the fp16 output
    # (a difference of one step of a value is 2^-10 of it); four times that
    return {"rel": 1e-3, "max": 1e-2}


def _encoded(x, online):
    """(signs +-1, scale, residual codes, residual scale) of fp16 vectors [n, d] as the
    cache holds them, in 64 bits.  The format rounds the scales to fp16 and takes the
    codes from 32-bit products (an element halfway between two codes goes by them)."""
    mean = x.double().abs().mean(-1, keepdim=True).float()
    x = x.float()
    sign = torch.where(x >= 0, 1.0, -1.0)
    scale = mean.half()
    r = x - sign * (mean if online else scale.float())
    top = r.abs().amax(-1, keepdim=True)
    inv = torch.where(top > 0, 7.0 / top.double(), 0.0).float()
    codes = torch.round(r * inv).clamp(-7, 7)
    return sign.double(), scale.double(), codes.double(), top.half().double()


def exact(case, seed):
    op = case["op"]
    if op in ("prefill", "encode"):
        return None     # whole bytes: compared as they are
    B, H, Hkv, d, S = (case[k] for k in ("batch", "heads", "kv_heads", "dim", "seq"))
    G = H // Hkv
    x = _inputs(case, seed)
    if op == "step":    # the ring is full: the token takes the first slot
        x["k"][:, :, 0] = x["new_k"]
        x["v"][:, :, 0] = x["new_v"]
    out = torch.empty((B, H, d), dtype=torch.float64, device="cuda")
    modes = torch.empty((B, H), dtype=torch.uint8, device="cuda")
    online = op in ("step", "attend")
    for b in range(B):
        for h in range(Hkv):
            heads = slice(h * G, (h + 1) * G)
            q = x["q"][b, heads].double()                                   # [G, d]
            ks, kscale, kc, krs = _encoded(x["k"][b, h], online)
            vs, vscale, vc, vrs = _encoded(x["v"][b, h], online)
            match = torch.where(q >= 0, 1.0, -1.0).double() @ ks.T          # 2 popcount - d
            score = q.abs().mean(-1, keepdim=True) * kscale.T * match       # [G, S]
            value, vres = vs * vscale, vc / 7.0 * vrs
            with_res = torch.full((G, S), float(case["residual"]), dtype=torch.float64, device="cuda")
            if op == "adaptive":
                order = torch.sort(kscale.T * match, dim=-1, descending=True, stable=True)[1]
                with_res.zero_().scatter_(1, order[:, :default_top_k(S)], 1.0)
            if op == "modes":
                p = torch.softmax(score, -1)
                entropy = -(p * torch.log(p.clamp_min(1e-300))).sum(-1)
                modes[b, heads] = (entropy < _threshold(case)).to(torch.uint8)
                with_res = with_res * modes[b, heads, None].double()
            if case["residual"]:
                score = score + with_res * (q @ (kc / 7.0 * krs).T)
            p = torch.softmax(score / math.sqrt(d), -1)
            out[b, heads] = p @ value
            if case["residual"]:
                out[b, heads] += (p * with_res) @ vres
    if op == "step":
        return [out] + [None] * (4 if case["residual"] else 2)
    return (out, modes) if op == "modes" else out
