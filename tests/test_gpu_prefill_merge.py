"""The two split merges of the prefill (up to 8 splits, and more than a wave's batch of them)
on chunks with rows to spare, against float64 attention over the dequantized cache."""
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,Hq,Hkv,bk,bv", [(17, 4, 2, 3, 3), (5, 2, 2, 2, 4), (40, 8, 1, 4, 3)])
@pytest.mark.parametrize("splits,causal", [(2, False), (7, True), (8, False), (9, True), (63, False), (80, True)])
def test_split_merges(dt, M, Hq, Hkv, bk, bv, splits, causal):
    import akv
    announce(f"prefill merge {dt} M{M} Hq{Hq} Hkv{Hkv} bits {bk}/{bv} splits {splits} causal {causal}")
    g = torch.Generator(device="cuda").manual_seed(M * 100 + splits)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    B, Nw, Nh = 2, 2590, 45
    warm = akv.quantize_kv(r(B, Hkv, Nw, 128), r(B, Hkv, Nw, 128), bk, bv, 32, 64)
    kh, vh, q = r(B, Hkv, Nh, 128), r(B, Hkv, Nh, 128), r(B, Hq, M, 128).to(dt)
    kc, vc = (r(B, Hkv, M, 128).to(dt), r(B, Hkv, M, 128).to(dt)) if causal else (None, None)
    got = akv.prefill_attention(q, kh, vh, warm, num_splits=splits, k_chunk=kc, v_chunk=vc)
    kd, vd = akv.dequantize(warm)
    k, v = (torch.cat([a, b] + ([c.half()] if causal else []), dim=2).double().repeat_interleave(Hq // Hkv, dim=1)
            for a, b, c in ((kh, kd, kc), (vh, vd, vc)))
    s = (q.half().double() @ k.transpose(2, 3).contiguous()) * 128 ** -0.5
    if causal:
        j = torch.arange(k.shape[2], device="cuda") - (Nh + Nw)
        s.masked_fill_(j[None, :] > torch.arange(M, device="cuda")[:, None], float("-inf"))
    exp = torch.softmax(s, -1) @ v
    # 16-bit probabilities average out; the output's own rounding: 2^-9 (bf16) or 2^-11 of values below 0.5
    assert float((got.double() - exp).abs().max()) <= (3e-3 if dt == torch.bfloat16 else 1e-3)


@pytest.mark.parametrize("M,Hq,Hkv", [(1, 2, 2), (3, 2, 2), (5, 6, 2), (2, 8, 1)])
@pytest.mark.parametrize("splits", [3, 8, 40])
def test_few_rows_keep_to_their_workspace(M, Hq, Hkv, splits, monkeypatch):
    """1, 3, 15 and 16 rows per kv head: partials of that many rows, and nothing past the bytes asked for."""
    import akv
    from akv import _native as nat
    announce(f"prefill few rows M{M} Hq{Hq} Hkv{Hkv} splits {splits}")
    g = torch.Generator(device="cuda").manual_seed(M * 10 + splits)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    B, Nw, Nh = 2, 1300, 45
    asked = []

    def workspace(nbytes, device, zero_prefix=0):
        asked.append((nbytes, torch.full((nbytes + 4096,), 0x5A, dtype=torch.uint8, device=device)))
        return asked[-1][1][:nbytes]

    warm = akv.quantize_kv(r(B, Hkv, Nw, 128), r(B, Hkv, Nw, 128), 3, 4, 32, 32)
    kh, vh, q = r(B, Hkv, Nh, 128), r(B, Hkv, Nh, 128), r(B, Hq, M, 128)
    monkeypatch.setattr(nat, "workspace", workspace)
    got = akv.prefill_attention(q, kh, vh, warm, num_splits=splits)
    assert len(asked) == 1 and bool((asked[0][1][asked[0][0]:] == 0x5A).all())
    kd, vd = akv.dequantize(warm)
    k, v = (torch.cat(x, dim=2).double().repeat_interleave(Hq // Hkv, dim=1) for x in ((kh, kd), (vh, vd)))
    exp = torch.softmax((q.double() @ k.transpose(2, 3).contiguous()) * 128 ** -0.5, -1) @ v
    assert float((got.double() - exp).abs().max()) <= 1e-3
