"""Many single heads and pairs over short contexts: calls just inside and just past
the contexts that run on the VALU split kernel, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.gpu_util import bin_from_blob, close, res_from_blob, say, to_np

pytestmark = pytest.mark.gpu

# (mode, d, group, kv heads of one sequence, contexts around the line on 256 CUs)
CASES = [("adaptive", 192, 1, 512, (1, 17, 288, 289)), ("adaptive", 224, 1, 1024, (63, 400, 401)),
         ("adaptive", 160, 1, 2048, (17, 64, 65)), ("adaptive", 96, 1, 2048, (64, 65)),
         ("adaptive", 192, 2, 512, (64, 65)),
         ("compensated", 160, 1, 2048, (17, 40, 41)), ("compensated", 192, 1, 2048, (40, 41)),
         ("compensated", 224, 1, 2048, (1, 40, 41))]


@pytest.mark.parametrize("mode,d,G,Hkv,contexts", CASES, ids=lambda x: str(x))
def test_around_the_line(mode, d, G, Hkv, contexts):
    """Every kv head holds one of four key sets, so that a few heads checked
    against the oracle stand for all (equal heads give equal outputs)."""
    from bitcache_amd import functional as F
    B, Hq, n = 1, Hkv * G, 4
    for S in contexts:
        say(f"case {mode} d={d} group={G} kv heads={Hkv} S={S}")
        g = torch.Generator(device="cuda")
        g.manual_seed(d + S)
        rnd = lambda *s: torch.randn(s, generator=g, device="cuda").half()
        q = rnd(1, n * G, d).repeat(1, Hkv // n, 1)
        k, v = rnd(n * S, d), rnd(n * S, d)
        (kb, kr), (vb, vr) = F.encode_fused(k.repeat(Hkv // n, 1)), F.encode_fused(v.repeat(Hkv // n, 1))
        enc = [f(b, n * S, d) for f, b in ((bin_from_blob, F.encode(k)), (res_from_blob, F.encode_fused(k)[1]),
                                           (bin_from_blob, F.encode(v)), (res_from_blob, F.encode_fused(v)[1]))]
        qs, kw = to_np(q)[:, :n * G], dict(n_kv_heads=Hkv)
        if mode == "adaptive":
            top_k = max(1, S // 10)
            _, ref, sets = O.adaptive_attention(qs, *enc, B, n * G, S, top_k, n_kv_heads=n,
                                                return_f32=True, return_sets=True)
            out, sel = F.adaptive_attention(q, kb, kr, vb, vr, B, Hq, S, d, top_k=top_k, return_selected=True, **kw)
            for (b, i), idx in sets.items():
                assert np.array_equal(np.nonzero(to_np(sel)[b, i])[0], idx), f"selected set of head {i}"
            assert torch.equal(sel, sel[:, :n * G].repeat(1, Hkv // n, 1))
        else:
            _, ref = O.compensated_attention(qs, *enc, B, n * G, S, n_kv_heads=n, return_f32=True)
            out = F.compensated_attention(q, kb, kr, vb, vr, B, Hq, S, d, **kw)
        close(to_np(out)[:, :n * G].astype(np.float32), ref, what=f"{mode} S={S}")
        assert torch.equal(out, out[:, :n * G].repeat(1, Hkv // n, 1))
