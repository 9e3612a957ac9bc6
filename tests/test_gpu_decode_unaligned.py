"""The LDS-streamed decode on tiers whose meta rows and weight rows start off 16 bytes: token
counts of every residue, one and two meta groups per token (block-affine V and the legacy
layout), several (batch, kv-head)s, both tier orders, with weights and importance."""
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


def _reference(q, k, v):
    g = q.shape[1] // k.shape[1]
    k, v = (x.double().repeat_interleave(g, dim=1) for x in (k, v))
    p = torch.softmax((q.double() @ k.transpose(2, 3).contiguous()) * q.shape[-1] ** -0.5, dim=-1)
    return p @ v, p


@pytest.mark.parametrize("G,M,hot_first", [(64, 1, False), (64, 3, True), (128, 1, True), (32, 2, False)])
@pytest.mark.parametrize("Nw", [31, 32, 33, 97, 354, 703])
@pytest.mark.parametrize("Nh", [5, 18])
def test_unaligned_rows(G, M, hot_first, Nw, Nh):
    import akv
    announce(f"decode unaligned G{G} M{M} hot_first={hot_first} Nw={Nw} Nh={Nh}")
    g = torch.Generator(device="cuda").manual_seed(Nw * 100 + Nh + G)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    B, Hkv, Hq = 2, 3, 6
    kw, vw, kh, vh, q = r(B, Hkv, Nw, 128), r(B, Hkv, Nw, 128), r(B, Hkv, Nh, 128), r(B, Hkv, Nh, 128), r(B, Hq, M, 128)
    warm = akv.quantize_kv(kw, vw, 3, 4, 32, G)
    kd, vd = akv.dequantize(warm)
    order = (lambda w, h: torch.cat([h, w], dim=2)) if hot_first else (lambda w, h: torch.cat([w, h], dim=2))
    exp, p = _reference(q, order(kd, kh), order(vd, vh))
    s0 = torch.rand(Nw + Nh, generator=g, device="cuda")
    for _ in range(2):
        s = s0.clone()
        out, w = akv.decode_attention(q, kh, vh, warm, hot_first=hot_first, scores=s, decay=0.9, return_weights=True)
        # 16-bit probabilities and output: a few 2^-11 of the values averaged
        assert float((out.double() - exp).abs().max()) <= 2e-3
        # fp32 logits of |s| < 32 and exp2: 32 * 2^-23 relative, a few times over
        torch.testing.assert_close(w.double(), p, rtol=2e-5, atol=1e-9)
        torch.testing.assert_close(s.double(), s0.double() * 0.9 + p.sum((0, 1, 2)) / (B * Hq), rtol=2e-5, atol=1e-8)
        s = s0.clone()  # the stash instead of returned weights
        out2 = akv.decode_attention(q, kh, vh, warm, hot_first=hot_first, scores=s, decay=0.9)
        assert float((out2.double() - exp).abs().max()) <= 2e-3
        torch.testing.assert_close(s.double(), s0.double() * 0.9 + p.sum((0, 1, 2)) / (B * Hq), rtol=2e-5, atol=1e-8)
