"""Softmax weights far apart in the value phase: one key that takes nearly all
of a head's weight above a long tail, rows of V of very different magnitude,
V scales that are not finite.  Against 64-bit sums over the encoded planes."""
import math

import pytest
import torch

from tests.gpu_util import say

pytestmark = pytest.mark.gpu


def tile_blob(blob, n, row_bytes, rows):
    """A blob of `rows` copies of an n-vector blob, one per kv head (planar
    layout: all rows' sign or code bytes, then all their scales)."""
    per = blob.numel() // n
    out = torch.zeros(rows * n * per, dtype=torch.uint8, device=blob.device)
    main, scales = blob[:n * row_bytes], blob[n * row_bytes:n * (row_bytes + 2)]
    out[:rows * n * row_bytes] = main.repeat(rows)
    out[rows * n * row_bytes:rows * n * (row_bytes + 2)] = scales.repeat(rows)
    return out


def planes64(bin_, res, n, d):
    """(signs +-1, scale, codes / 7, residual scale) of n vectors in 64 bits."""
    from bitcache_amd import layout
    words, scale = layout.binary_planes(bin_, d, n)
    bits = (words.unsqueeze(-1) >> torch.arange(32, device=words.device, dtype=torch.int32)) & 1
    nib, rs = layout.residual_planes(res, d, n)
    c = torch.stack([nib & 15, nib >> 4], -1).reshape(n, d).to(torch.int16)
    c = torch.where(c >= 8, c - 16, c)
    return bits.reshape(n, d).double() * 2 - 1, scale.double()[:, None], c.double() / 7, rs.double()[:, None]


def exact(q, k, v, with_res):
    """[G, d] attention of one kv head in 64 bits; with_res [G, S]: the keys
    whose residuals each head takes."""
    q = q.double()
    ks, kscale, kc, krs = k
    vs, vscale, vc, vrs = v
    w = with_res.double()
    score = q.abs().mean(-1, keepdim=True) * kscale.T * (torch.where(q >= 0, 1.0, -1.0).double() @ ks.T)
    score = score + w * (q @ (kc * krs).T)
    p = torch.softmax(score / math.sqrt(q.shape[-1]), -1)
    return p @ (vs * vscale) + (p * w) @ (vc * vrs)


def make(B, Hq, Hkv, S, d, gap, outliers, seed):
    """Every kv head holds the same S keys and values: key g is the one that
    query head g of a group gives nearly all of its weight, `gap` nats above
    the others; outliers: one row of V in 256 that many times larger."""
    from bitcache_amd import functional as F
    G = Hq // Hkv
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")
    q1 = rnd(G, d)
    k, v = rnd(S, d) * 0.5, rnd(S, d)
    k[:G] = q1 * (gap / (q1 * q1).sum(-1, keepdim=True) * math.sqrt(d))
    if outliers != 1:
        v[5::256] *= outliers
    enc = [F.encode_fused(x.half()) for x in (k, v)]
    q = q1.half().repeat(B * Hkv, 1).view(B, Hq, d).contiguous()
    blobs = []
    for bin_, res in enc:
        blobs += [tile_blob(bin_, S, d // 8, B * Hkv), tile_blob(res, S, d // 2, B * Hkv)]
    return q, blobs, [planes64(*e, S, d) for e in enc]


def attend(mode, q, blobs, B, Hq, Hkv, S, d):
    """(output [B, Hq, d], the keys whose residuals the first group takes [G, S])"""
    from bitcache_amd import functional as F
    kb, kr, vb, vr = blobs
    G, kw = Hq // Hkv, dict(n_kv_heads=Hkv)
    if mode == "binary":
        return F.binary_attention(q, kb, vb, B, Hq, S, d, **kw), torch.zeros((G, S), device="cuda")
    if mode == "compensated":
        return F.compensated_attention(q, kb, kr, vb, vr, B, Hq, S, d, **kw), torch.ones((G, S), device="cuda")
    if mode == "adaptive":
        out, sel = F.adaptive_attention(q, kb, kr, vb, vr, B, Hq, S, d, return_selected=True, **kw)
        return out, sel[0, :G].clone()
    modes = ((torch.arange(Hq, device="cuda") + 1) % 2).to(torch.uint8).repeat(B, 1)
    out = F.head_mode_attention(q, kb, kr, vb, vr, modes, B, Hq, S, d, **kw)
    return out, modes[0, :G, None].expand(G, S)


def rel_error(mode, shape, gap, outliers):
    B, Hq, Hkv, S, d = shape
    if mode == "binary":
        gap *= math.pi / 2   # (its scores are 2 / pi of those with the residual)
    q, blobs, enc = make(B, Hq, Hkv, S, d, gap, outliers, seed=S + d + int(gap))
    out, with_res = attend(mode, q, blobs, B, Hq, Hkv, S, d)
    G = Hq // Hkv
    want = exact(q[0, :G], *enc, with_res)
    got = out[0, :G].double()
    assert torch.isfinite(got).all()
    n = max(G, 2)   # (single heads of mixed calls are of alternating modes)
    assert torch.equal(out.view(-1, n, d), out[0, :n].expand(B * Hq // n, n, d)), "kv heads differ"
    return float(((got - want).norm(dim=-1) / want.norm(dim=-1)).max())


# 2-norm of the error over that of the result, per head: half a step of the
# fp16 output is at most 2^-11 of a value, and the fixed-point scores are within
# 2^-11 nats, which moves a weight by as much
BAR = 2.0 ** -10

# (mode, (B, Hq, Hkv, S, d)): plans of one split of 16K keys per wave
LONG = [("binary", (8, 32, 32, 131072, 64)),
        ("compensated", (32, 32, 8, 65536, 256)),
        ("adaptive", (32, 8, 8, 65536, 160))]


@pytest.mark.parametrize("mode,shape", LONG, ids=lambda x: str(x))
def test_one_key_above_a_long_tail(mode, shape):
    """A tail each of whose weights is near or below the resolution of the
    integer weights: together it is a visible share of the softmax sum."""
    for gap in (12.0, 13.5, 14.5, 15.5):
        err = rel_error(mode, shape, gap, 1)
        say(f"case one key {mode} {shape} gap {gap}: error {err:.2e}")
        assert err <= BAR
    torch.cuda.empty_cache()


@pytest.mark.parametrize("mode", ["binary", "compensated", "adaptive", "mixed"])
@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_value_scale_not_finite(mode, G):
    """A V row whose scale is infinite or NaN (what an infinite element
    encodes to): no sum of the heads that read it is a number, in any mode and
    whatever the row's sign bits; the other kv head's are as without it."""
    from bitcache_amd import functional as F, layout
    B, Hkv, S, d = 1, 2, 500, 128
    Hq = Hkv * G
    q, blobs, _ = make(B, Hq, Hkv, S, d, 1.0, 1, seed=G)
    clean, _ = attend(mode, q, blobs, B, Hq, Hkv, S, d)
    for bad in (math.inf, math.nan):
        for key in (0, 70, 499):
            say(f"case V scale {bad} at key {key}, {mode}, group {G}")
            vb = blobs[2].clone()
            layout.binary_planes(vb, d)[1][key] = bad
            out, _ = attend(mode, q, blobs[:2] + [vb] + blobs[3:], B, Hq, Hkv, S, d)
            assert torch.isnan(out[0, :G]).all()
            assert torch.equal(out[0, G:], clean[0, G:])


@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_residual_scale_not_finite(G):
    """A V residual scale that is infinite or NaN: the compensated heads that
    read it are NaN, a binary head of the same group is as without it."""
    from bitcache_amd import layout
    B, Hkv, S, d = 1, 2, 500, 128
    Hq = Hkv * G
    q, blobs, enc = make(B, Hq, Hkv, S, d, 1.0, 1, seed=G)
    modes = torch.arange(Hq, device="cuda") % 2 == 0   # (attend's: even heads are compensated)
    for bad in (math.inf, math.nan):
        for key in (0, 70, 499):
            say(f"case V residual scale {bad} at key {key}, group {G}")
            vr = blobs[3].clone()
            for kv in range(Hkv):
                layout.residual_planes(vr, d)[1][kv * S + key] = bad
            broken = blobs[:3] + [vr]
            out, with_res = attend("mixed", q, broken, B, Hq, Hkv, S, d)
            assert torch.isnan(out[0, modes]).all()
            want = exact(q[0, :G].repeat(Hkv, 1), *enc, torch.zeros((Hq, S), device="cuda"))
            got = out[0, ~modes].double()
            err = float(((got - want[~modes]).norm(dim=-1) / want[~modes].norm(dim=-1)).max())
            assert err <= BAR, f"binary heads: error {err:.2e}"
            out, _ = attend("compensated", q, broken, B, Hq, Hkv, S, d)
            assert torch.isnan(out).all()


@pytest.mark.parametrize("mode", ["binary", "compensated", "adaptive", "mixed"])
@pytest.mark.parametrize("G", [1, 2, 4, 8])
def test_negative_value_scales(mode, G):
    """V scales of either sign, which no encoder writes and a blob may hold:
    the values are the scales' products with the signs and codes as ever."""
    from bitcache_amd import layout
    B, Hkv, S, d = 1, 2, 3000, 128
    Hq = Hkv * G
    for share in (1, 3):   # every scale negative, every third one
        say(f"case negative V scales {mode} group {G}, one in {share}")
        q, blobs, enc = make(B, Hq, Hkv, S, d, 4.0, 1, seed=G)
        for kv in range(Hkv):
            for planes, blob in ((layout.binary_planes, blobs[2]), (layout.residual_planes, blobs[3])):
                planes(blob, d)[1][kv * S:(kv + 1) * S][::share] *= -1
        flip = torch.ones((S, 1), dtype=torch.float64, device="cuda")
        flip[::share] = -1
        v = (enc[1][0], enc[1][1] * flip, enc[1][2], enc[1][3] * flip)
        out, with_res = attend(mode, q, blobs, B, Hq, Hkv, S, d)
        want = exact(q[0, :G], enc[0], v, with_res)
        got = out[0, :G].double()
        err = float(((got - want).norm(dim=-1) / want.norm(dim=-1)).max())
        assert err <= BAR, f"error {err:.2e}"


@pytest.mark.parametrize("mode", ["binary", "compensated", "adaptive", "mixed"])
@pytest.mark.parametrize("shape", [(1, 8, 8, 16384, 96), (1, 8, 2, 16384, 64), (2, 32, 8, 16384, 128),
                                   (1, 16, 2, 16384, 128), (1, 4, 2, 9000, 256), (8, 32, 32, 65536, 128)],
                         ids=lambda s: str(s))
def test_rows_of_very_different_magnitude(mode, shape):
    """One V row in 256 of 4 to 32 times the others' magnitude, with next to no
    softmax weight: the resolution of the weights is that of the weighted
    values, not of the largest row."""
    for gap, outliers in ((9.0, 8), (9.0, 32), (12.0, 32), (14.0, 4)):
        err = rel_error(mode, shape, gap, outliers)
        say(f"case outlier rows {mode} {shape} gap {gap} x{outliers}: error {err:.2e}")
        assert err <= BAR
    torch.cuda.empty_cache()


@pytest.mark.parametrize("d", [32, 96, 160, 192, 224])
@pytest.mark.parametrize("mode", ["binary", "compensated"])
def test_groups_of_eight_at_every_head_dim(mode, d):
    """Unit-variance heads of 9001 keys: what the kernel's sums add to the
    rounding of the fp16 output is at most a quarter of that rounding (fp32 sums
    of fp16 products with the codes' offset of 8 are past it)."""
    from bitcache_amd import functional as F
    B, Hkv, S, G = 1, 8, 9001, 8
    g = torch.Generator(device="cuda")
    g.manual_seed(d)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").half()
    q, k, v = rnd(B, Hkv * G, d), rnd(Hkv, S, d), rnd(Hkv, S, d)
    kb, kr = F.encode_fused(k.view(-1, d))
    vb, vr = F.encode_fused(v.view(-1, d))
    out, with_res = attend(mode, q, (kb, kr, vb, vr), B, Hkv * G, Hkv, S, d)
    want = torch.cat([exact(q[0, G * h:G * h + G], planes64(*F.encode_fused(k[h]), S, d),
                            planes64(*F.encode_fused(v[h]), S, d), with_res) for h in range(Hkv)])
    err = float((out[0].double() - want).norm() / want.norm())
    rounding = float((want.half().double() - want).norm() / want.norm())
    say(f"case groups of eight {mode} d={d}: error {err:.2e}, of rounding alone {rounding:.2e}")
    assert err <= rounding * math.sqrt(1 + 0.25 ** 2)
