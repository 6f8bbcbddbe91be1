"""Sources and blobs that start at any element or record of a larger
allocation: rows of fp16 at an odd element, binary blobs at a multiple of 36
bytes, residual blobs at a multiple of 130 (2-byte alignment, as stacked
per-layer blobs of an odd number of vectors have it) give the bytes and
outputs of aligned ones, at every head dim."""
import pytest
import torch

from tests.gpu_util import say

pytestmark = pytest.mark.gpu

DIMS = [32, 64, 96, 128, 160, 192, 224, 256]


def at(blob, offset):
    """A copy of a blob `offset` bytes into a larger allocation."""
    big = torch.empty(blob.numel() + offset + 64, dtype=torch.uint8, device=blob.device)
    out = big[offset:offset + blob.numel()]
    out.copy_(blob)
    return out


@pytest.mark.parametrize("d", DIMS)
def test_encode_sources_at_an_odd_element(d):
    from bitcache_amd import functional as F
    n = 1003
    say(f"case source at an odd element d={d}")
    g = torch.Generator(device="cuda")
    g.manual_seed(d)
    big = torch.randn(n * d + 8, generator=g, device="cuda").half()
    src = big[1:1 + n * d].view(n, d)
    own = src.clone()
    bin_, res = F.encode(own), F.compute_residual(own, F.encode(own))
    used = n * (d // 8 + 2), n * (d // 2 + 2)
    assert torch.equal(F.encode(src)[:used[0]], bin_[:used[0]])
    assert torch.equal(F.compute_residual(src, bin_)[:used[1]], res[:used[1]])
    assert torch.equal(F.compute_residual(src, at(bin_, 36 * 5))[:used[1]], res[:used[1]])
    for x, y, m in zip(F.encode_fused(src), F.encode_fused(own), used):
        assert torch.equal(x[:m], y[:m])


@pytest.mark.parametrize("G", [1, 4, 8])
@pytest.mark.parametrize("d", DIMS)
def test_attention_over_blobs_at_a_record_boundary(d, G):
    from bitcache_amd import functional as F
    B, Hkv, S = 1, 3, 333   # 999 vectors
    Hq = Hkv * G
    say(f"case blobs at a record boundary d={d} G={G}")
    g = torch.Generator(device="cuda")
    g.manual_seed(d + G)
    q = torch.randn((B, Hq, d), generator=g, device="cuda").half()
    enc = [F.encode_fused(torch.randn((B * Hkv * S, d), generator=g, device="cuda").half()) for _ in range(2)]
    (kb, kr), (vb, vr) = enc
    shape, kw = (B, Hq, S, d), dict(n_kv_heads=Hkv)
    modes = (torch.arange(Hq, device="cuda") % 2).to(torch.uint8).view(B, Hq)
    calls = {
        "binary": lambda kb, kr, vb, vr: F.binary_attention(q, kb, vb, *shape, **kw),
        "compensated": lambda *b: F.compensated_attention(q, *b, *shape, **kw),
        "adaptive": lambda *b: F.adaptive_attention(q, *b, *shape, **kw),
        "modes": lambda *b: F.head_mode_attention(q, *b, modes, *shape, **kw),
        "entropy": lambda kb, kr, vb, vr: F.compute_head_entropy(q, kb, *shape, **kw),
        "scores": lambda kb, kr, vb, vr: F.binary_scores(q, kb, *shape, **kw)[0],
    }
    for bin_at, res_at in ((36, 130), (36 * 3, 130 * 3), (36 * 4, 130 * 2)):
        moved = [at(kb, bin_at), at(kr, res_at), at(vb, bin_at), at(vr, res_at)]
        for what, call in calls.items():
            assert torch.equal(call(*moved), call(kb, kr, vb, vr)), f"{what}, offsets {bin_at}, {res_at}"
