"""Decode over tiers whose meta rows, outlier values and weight rows start off 16 bytes: token
counts of every residue, one, two and four meta groups per token (block-affine V and the legacy
layout), one and three protected channels, several (batch, kv-head)s, both tier orders, with
weights and importance."""
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


def _legacy_tier(B, H, n, bits, G, g):
    """A legacy tier of one (scale, zero) per token and group, its descriptor and its dense values."""
    from akv import _native as nat
    per = 8 // bits
    q = torch.randint(0, 1 << bits, (B, H, n, 128), generator=g, device="cuda", dtype=torch.uint8)
    sh = torch.tensor([8 - bits * (i + 1) for i in range(per)], device="cuda")
    packed = (q.view(B, H, n, 128 // per, per).int() << sh).sum(-1).to(torch.uint8).contiguous()
    s, z = (0.1 * torch.randn(B, H, n, 128 // G, generator=g, device="cuda").half() for _ in range(2))
    s = s.abs() + 0.01
    dense = (q.view(B, H, n, 128 // G, G).float() * s.unsqueeze(-1).float() + z.unsqueeze(-1).float()).half()
    return packed, s, z, dense.view(B, H, n, 128), nat


@pytest.mark.parametrize("bits,G", [(4, 64), (2, 64), (2, 128)])
@pytest.mark.parametrize("Nw", [33, 777])
def test_unaligned_legacy_rows(bits, G, Nw):
    """Legacy tiers, one per (batch, kv head), of odd length with one and two groups."""
    import ctypes

    announce(f"decode unaligned legacy bits{bits} G{G} Nw={Nw}")
    g = torch.Generator(device="cuda").manual_seed(Nw + G + bits)
    B, Hkv, Hq, M, Nh = 2, 3, 6, 2, 21
    kc, ks, kz, kd, nat = _legacy_tier(B, Hkv, Nw, bits, G, g)
    vc, vs, vz, vd, _ = _legacy_tier(B, Hkv, Nw, bits, G, g)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    kh, vh, q = r(B, Hkv, Nh, 128), r(B, Hkv, Nh, 128), r(B, Hq, M, 128)
    out = torch.empty_like(q)
    a = nat.DecodeArgs()
    a.abi_version = nat.ABI_VERSION
    a.q_dtype = nat.DT_F16
    a.B, a.Hq, a.Hkv, a.M, a.D = B, Hq, Hkv, M, 128
    a.q, a.out, a.k_hot, a.v_hot, a.n_hot = q.data_ptr(), out.data_ptr(), kh.data_ptr(), vh.data_ptr(), Nh
    a.sm_scale = 128 ** -0.5
    w = a.warm
    w.kind, w.bits_k, w.bits_v, w.n_warm, w.group_size = nat.WARM_LEGACY, bits, bits, Nw, G
    w.meta_dtype, w.legacy_sym, w.warm_heads = nat.DT_F16, 0, B * Hkv
    w.k_codes, w.k_scale, w.k_zero = kc.data_ptr(), ks.data_ptr(), kz.data_ptr()
    w.v_codes, w.v_scale, w.v_zero = vc.data_ptr(), vs.data_ptr(), vz.data_ptr()
    lib = nat.load()
    ws = torch.zeros(lib.akv_decode_workspace_bytes(ctypes.byref(a)), dtype=torch.uint8, device="cuda")
    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    nat.check(lib.akv_decode_attn(ctypes.byref(a), nat.stream_of(q)), "decode")
    exp, _ = _reference(q, torch.cat([kd, kh], dim=2), torch.cat([vd, vh], dim=2))
    # 16-bit probabilities, values and output: a few 2^-11 of the values averaged
    assert float((out.double() - exp).abs().max()) <= 2e-3


@pytest.mark.parametrize("B,Hkv,Hq,M,bits,Nw,Nh", [(3, 4, 28, 3, 2, 9001, 333), (1, 4, 28, 3, 2, 20001, 333),
                                                   (3, 4, 28, 1, 3, 4001, 17)])
def test_odd_two_group_tiers_repeat(B, Hkv, Hq, M, bits, Nw, Nh):
    """Affine tiers of odd length with V groups of 64: decode_split_kernel, bit for bit the same each call."""
    import akv
    announce(f"decode repeat B{B} Hkv{Hkv} Hq{Hq} M{M} bits{bits} Nw={Nw}")
    g = torch.Generator(device="cuda").manual_seed(Nw)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    kw, vw, kh, vh = r(B, Hkv, Nw, 128), r(B, Hkv, Nw, 128), r(B, Hkv, Nh, 128), r(B, Hkv, Nh, 128)
    q = r(B, Hq, M, 128)
    warm = akv.quantize_kv(kw, vw, bits, bits, 32, 64)
    s0 = torch.rand(Nw + Nh, generator=g, device="cuda")
    runs = []
    for _ in range(6):
        s = s0.clone()
        runs.append((*akv.decode_attention(q, kh, vh, warm, scores=s, decay=0.9, return_weights=True), s))
    for run in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(run, runs[0]))


@pytest.mark.parametrize("B,Hkv,Hq,M,frac", [(1, 1, 4, 1, 0.01), (2, 3, 6, 2, 0.01), (2, 2, 2, 1, 0.024)])
@pytest.mark.parametrize("Nw", [31, 777, 4001])
@pytest.mark.parametrize("weights", [False, True])
def test_odd_outlier_counts(B, Hkv, Hq, M, frac, Nw, weights):
    """One and three protected channels over tiers of odd length: a head's outlier values are an odd
    number of 16-bit values, so every second head's start at half a dword."""
    import akv
    announce(f"decode odd outliers B{B} Hkv{Hkv} M{M} frac{frac} Nw={Nw} weights={weights}")
    g = torch.Generator(device="cuda").manual_seed(Nw + B)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    Nh = 37
    kw, vw, kh, vh, q = r(B, Hkv, Nw, 128), r(B, Hkv, Nw, 128), r(B, Hkv, Nh, 128), r(B, Hkv, Nh, 128), r(B, Hq, M, 128)
    kw[..., 5] *= 8  # the channel that is protected carries most of a logit
    vw[..., 77] *= 8
    warm = akv.quantize_kv(kw, vw, 4, 2, 32, 32, outlier_fraction=frac)
    assert warm.n_out % 2 == 1
    kd, vd = akv.dequantize(warm)
    exp, p = _reference(q, torch.cat([kd, kh], dim=2), torch.cat([vd, vh], dim=2))
    s0 = torch.rand(Nw + Nh, generator=g, device="cuda")
    s = s0.clone()
    out = akv.decode_attention(q, kh, vh, warm, scores=s, decay=0.9, return_weights=weights)
    if weights:
        out, w = out
        # fp32 logits of |s| < 128 and exp2: 128 * 2^-23 relative, a few times over
        torch.testing.assert_close(w.double(), p, rtol=1e-4, atol=1e-9)
    # 16-bit probabilities and output: 2^-11 of values up to 40 in the protected channel, averaged
    assert float((out.double() - exp).norm() / exp.norm()) <= 1e-3
    torch.testing.assert_close(s.double(), s0.double() * 0.9 + p.sum((0, 1, 2)) / (B * Hq), rtol=1e-4, atol=1e-8)
