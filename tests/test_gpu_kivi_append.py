"""The one-pass KIVI overflow: tier and views equal to quantize_rows /
dequantize_rows on the same tokens, over dtypes, layouts, widths, group sizes past head_dim
and chunk lengths around the workgroup's tokens: bit-exact."""
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,D,kb,vb,gs,res", [(1, 2, 128, 2, 2, 128, 32), (2, 3, 64, 4, 8, 128, 5), (1, 1, 64, 2, 4, 32, 0),
                                                (2, 2, 128, 8, 8, 64, 7)])
def test_overflow_in_one_pass(dt, B, H, D, kb, vb, gs, res):
    from akv.baselines import KIVIFusedCache, KIVIFusedConfig, dequantize_rows, quantize_rows
    announce(f"KIVI append {dt} B{B} H{H} D{D} bits {kb}/{vb} gs{gs} res{res}")
    cache = KIVIFusedCache(KIVIFusedConfig(key_bits=kb, value_bits=vb, group_size=gs, residual_length=res))
    g = torch.Generator(device="cuda").manual_seed(D + gs + res)
    seen = [None, None]
    for n in (res + 1, 1, 63, 64, 65, 1, 1, 200, 3):
        kv = [(torch.randn(B, n, H, D, generator=g, device="cuda") * 2).to(dt).transpose(1, 2) for _ in range(2)]
        kv[0][:, :, 0] = 0.5  # a constant token: the scale's floor
        kv[1][0, 0, n // 2, 3] = float("nan")
        kv[1][0, -1, n - 1, 5] = float("inf")
        got = cache.update(kv[0], kv[1], 0)
        seen = [x if s is None else torch.cat([s, x], dim=2) for s, x in zip(seen, kv)]
        n_q = seen[0].shape[2] - res
        for x, view, bits, tier in zip(seen, got, (kb, vb), (cache._quant_keys[0], cache._quant_values[0])):
            codes, sc, ze = quantize_rows(x[:, :, :n_q], bits, gs)
            deq = dequantize_rows(codes, sc, ze, bits, gs, D).view(B, H, n_q, D)
            exp = torch.cat([deq, x[:, :, n_q:]], dim=2)
            assert view.dtype == exp.dtype and view.is_contiguous()
            assert torch.equal(view.view(torch.uint8), exp.view(torch.uint8))  # NaN patterns too
            assert tier.n == n_q and torch.equal(tier.codes[:, :n_q], codes)
            for a, e in ((tier.sc, sc), (tier.ze, ze), (tier.sc16, sc.half()), (tier.ze16, ze.half())):
                assert torch.equal(torch.nan_to_num(a[:, :n_q], nan=7.0), torch.nan_to_num(e, nan=7.0))
            assert not tier.codes[:, n_q:].any() and not tier.sc16[:, n_q:].any() and not tier.ze[:, n_q:].any()


def test_residual_autograd_and_refusal():
    from akv.baselines import KIVIFusedCache, KIVIFusedConfig
    announce("KIVI autograd / refusal")
    cache = KIVIFusedCache(KIVIFusedConfig(residual_length=4))
    k = torch.randn(1, 2, 10, 128, device="cuda", dtype=torch.float16, requires_grad=True)
    fk, _ = cache.update(k, k.detach(), 0)
    fk[:, :, -4:].float().sum().backward()
    assert torch.equal(k.grad[:, :, -4:], torch.ones_like(k.grad[:, :, -4:])) and not k.grad[:, :, :-4].any()
    bad = KIVIFusedCache(KIVIFusedConfig(key_bits=4, value_bits=3, residual_length=4))
    with pytest.raises(NotImplementedError):
        bad.update(k.detach(), k.detach(), 0)


def test_the_keys_say_how_many_tokens_leave():
    """A value more than keys stays in the values' residual window; fewer values than the overflow
    needs, other heads and another head_dim are refused, before anything changes."""
    from akv.baselines import KIVIFusedCache, KIVIFusedConfig, dequantize_rows, quantize_rows
    announce("KIVI overflow of unequal keys and values")
    g = torch.Generator(device="cuda").manual_seed(2)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    cfg = dict(key_bits=2, value_bits=4, group_size=64, residual_length=16)
    c = KIVIFusedCache(KIVIFusedConfig(**cfg))
    k, v = r(1, 2, 30, 64), r(1, 2, 31, 64)
    for step, (n, nk, nv) in enumerate(((14, 30, 31), (15, 31, 32))):
        kv = (k, v) if step == 0 else (r(1, 2, 1, 64), r(1, 2, 1, 64))
        got = c.update(*kv, 0)
        k, v = (k, v) if step == 0 else (torch.cat([k, kv[0]], dim=2), torch.cat([v, kv[1]], dim=2))
        for x, view, bits, m in ((k, got[0], 2, nk), (v, got[1], 4, nv)):
            deq = dequantize_rows(*quantize_rows(x[:, :, :n], bits, 64), bits, 64, 64).view(1, 2, n, 64)
            assert view.shape[2] == m and torch.equal(view, torch.cat([deq, x[:, :, n:]], dim=2))
    for k, v, err in ((r(1, 2, 30, 64), r(1, 2, 30, 128), ValueError), (r(1, 2, 30, 64), r(1, 3, 30, 64), RuntimeError),
                      (r(1, 2, 30, 64), r(1, 2, 13, 64), RuntimeError)):
        c = KIVIFusedCache(KIVIFusedConfig(**cfg))
        with pytest.raises(err):
            c.update(k, v, 0)
        assert not c._quant_keys and c._residual_keys[0] is k and c._residual_values[0] is v
