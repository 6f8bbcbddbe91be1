"""More query heads per kv head than the matrix-core kernel's plan argument
holds (8191 head groups): these calls run on the VALU split kernel, in every
mode, at every head dim and head group, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.gpu_util import bin_from_blob, close, res_from_blob, say, to_np

pytestmark = pytest.mark.gpu

GROUPS = 8193


@pytest.mark.parametrize("G", [1, 2, 4, 8])
@pytest.mark.parametrize("d", [32, 64, 96, 128, 160, 192, 224, 256])
def test_many_head_groups(d, G):
    """One kv head of 200 keys (a ragged last tile) under GROUPS * G query
    heads: a sample of them against the oracle (the bar of the other
    attention tests), binary and compensated heads alternating and in whole
    groups in the per-head modes."""
    from bitcache_amd import functional as F
    B, S, Hq = 1, 200, GROUPS * G
    say(f"case many head groups d={d} G={G}")
    g = torch.Generator(device="cuda")
    g.manual_seed(d + G)
    q = torch.randn((B, Hq, d), generator=g, device="cuda").half()
    k, v = (torch.randn((S, d), generator=g, device="cuda").half() for _ in range(2))
    (kb, kr), (vb, vr) = F.encode_fused(k), F.encode_fused(v)
    Kb, Vb = bin_from_blob(kb, S, d), bin_from_blob(vb, S, d)
    Kr, Vr = res_from_blob(kr, S, d), res_from_blob(vr, S, d)
    pick = np.r_[0:9, Hq // 2:Hq // 2 + 8, Hq - 9:Hq]
    qs = to_np(q)[:, pick]
    n, kw = len(pick), dict(n_kv_heads=1)
    take = lambda t: to_np(t)[:, pick].astype(np.float32)
    _, ref = O.compensated_attention(qs, Kb, Kr, Vb, Vr, B, n, S, n_kv_heads=1, return_f32=True)
    _, refb = O.binary_attention(qs, Kb, Vb, B, n, S, n_kv_heads=1, return_f32=True)
    close(take(F.compensated_attention(q, kb, kr, vb, vr, B, Hq, S, d, **kw)), ref, what="compensated")
    close(take(F.binary_attention(q, kb, vb, B, Hq, S, d, **kw)), refb, what="binary")
    # per-head modes: alternating heads, whole groups of 64 heads, all alike
    h = torch.arange(Hq, device="cuda")
    for what, modes in (("alternating", h % 2), ("runs", (h // 64) % 2), ("binary", h * 0), ("compensated", h * 0 + 1)):
        modes = modes.to(torch.uint8).view(B, Hq)
        out = take(F.head_mode_attention(q, kb, kr, vb, vr, modes, B, Hq, S, d, **kw))
        want = np.where((to_np(modes)[:, pick] != 0)[..., None], ref, refb)
        close(out, want, what=f"per-head modes, {what}")
    top_k = 20
    _, refa, sets = O.adaptive_attention(qs, Kb, Kr, Vb, Vr, B, n, S, top_k, n_kv_heads=1,
                                         return_f32=True, return_sets=True)
    out, sel = F.adaptive_attention(q, kb, kr, vb, vr, B, Hq, S, d, top_k=top_k, return_selected=True, **kw)
    close(take(out), refa, what="adaptive")
    sel = to_np(sel)[:, pick]
    for (b, i), idx in sets.items():
        assert np.array_equal(np.nonzero(sel[b, i])[0], idx), f"selected set of head {pick[i]}"
    torch.cuda.empty_cache()
