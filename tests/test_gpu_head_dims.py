"""The matrix-core attention kernels at every head dim and head group against
the oracle (2e-3 of the largest reference value, cosine >= 0.9999: the bar of
the other attention tests): rows of odd numbers of code pieces and half sign
blocks (d % 64 == 32), one key, ragged tiles, several tiles per wave, a row
stride past the context, inputs whose residual dots take the 16-bit fixed
point (small) and the 24-bit one (unit variance)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.gpu_util import bin_from_blob, close, res_from_blob, say, slice_enc, to_np

pytestmark = pytest.mark.gpu

DIMS = [32, 64, 96, 128, 160, 192, 224, 256]


def rows(e, n_rows, stride, S):
    """The first S of every `stride` vectors of an encoding of n_rows rows."""
    parts = [slice_enc(e, r * stride, r * stride + S) for r in range(n_rows)]
    if isinstance(e, O.BinaryEnc):
        return O.BinaryEnc(*(np.concatenate([getattr(p, f) for p in parts]) for f in ("words", "scale", "mean32")))
    return O.ResidualEnc(codes=np.concatenate([p.codes for p in parts]),
                         scale=np.concatenate([p.scale for p in parts]))


@pytest.mark.parametrize("group", [1, 2, 4, 8])
@pytest.mark.parametrize("d", DIMS)
def test_every_head_dim_and_group(d, group):
    from bitcache_amd import _C, functional as F
    B, Hkv = 1, 2
    Hq = Hkv * group
    for S, scale in ((1, 0.09), (65, 1.0), (700, 0.09), (1100, 1.0)):
        say(f"case d={d} group={group} S={S} scale={scale}")
        stride = S + 3
        rng = np.random.default_rng(d + group + S)
        q = (rng.standard_normal((B, Hq, d)) * scale).astype(np.float16)
        k = (rng.standard_normal((B * Hkv * stride, d)) * scale).astype(np.float16)
        v = (rng.standard_normal((B * Hkv * stride, d)) * scale).astype(np.float16)
        n = B * Hkv * stride
        kb, kr = F.encode_fused(torch.from_numpy(k).cuda())
        vb, vr = F.encode_fused(torch.from_numpy(v).cuda())
        Kb, Vb = (rows(bin_from_blob(x, n, d), B * Hkv, stride, S) for x in (kb, vb))
        Kr, Vr = (rows(res_from_blob(x, n, d), B * Hkv, stride, S) for x in (kr, vr))
        qt = torch.from_numpy(q).cuda()
        kw = dict(n_kv_heads=Hkv, kv_stride=stride)
        what = f"d={d} group={group} S={S}"
        _, ref = O.compensated_attention(q, Kb, Kr, Vb, Vr, B, Hq, S, n_kv_heads=Hkv, return_f32=True)
        out = F.compensated_attention(qt, kb, kr, vb, vr, B, Hq, S, d, **kw)
        close(to_np(out).astype(np.float32), ref, what="compensated " + what)
        _, refb = O.binary_attention(q, Kb, Vb, B, Hq, S, n_kv_heads=Hkv, return_f32=True)
        outb = F.binary_attention(qt, kb, vb, B, Hq, S, d, **kw)
        close(to_np(outb).astype(np.float32), refb, what="binary " + what)
        k_top = (S + 9) // 10
        _, refa, sets = O.adaptive_attention(q, Kb, Kr, Vb, Vr, B, Hq, S, k_top, n_kv_heads=Hkv,
                                             return_f32=True, return_sets=True)
        outa, sel = F.adaptive_attention(qt, kb, kr, vb, vr, B, Hq, S, d, top_k=k_top,
                                         return_selected=True, **kw)
        close(to_np(outa).astype(np.float32), refa, what="adaptive " + what)
        assert int(sel.sum()) == k_top * B * Hq, "selected keys " + what
        # heads of both modes inside every group
        modes = torch.from_numpy((np.arange(Hq) % 2).astype(np.uint8)).cuda().view(B, Hq)
        outm = F.head_mode_attention(qt, kb, kr, vb, vr, modes, B, Hq, S, d, **kw)
        refm = np.where((np.arange(Hq) % 2 == 1)[None, :, None], ref, refb)
        close(to_np(outm).astype(np.float32), refm, what="per-head modes " + what)
