"""Protected channels that share one 8-channel chunk: every one of them is replaced by its stored
value, however many a lane's chunk holds (decode_split_kernel takes the counts above 4, head_dim 64
and V groups other than 32)."""
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,bk,bv,G,n_out,first", [(128, 4, 2, 32, 3, 40), (128, 3, 3, 64, 3, 40), (128, 4, 2, 32, 8, 40),
                                                   (128, 2, 4, 128, 16, 64), (64, 3, 2, 32, 6, 25), (64, 4, 4, 64, 8, 56)])
@pytest.mark.parametrize("Nw", [64, 333])
def test_channels_of_one_chunk(D, bk, bv, G, n_out, first, Nw):
    import akv
    announce(f"decode outliers of one chunk D{D} bits{bk}/{bv} G{G} n_out={n_out} Nw={Nw}")
    g = torch.Generator(device="cuda").manual_seed(Nw + n_out)
    r = lambda *s: torch.randn(s, generator=g, device="cuda").half()  # noqa: E731
    B, Hkv, Hq, Nh = 2, 2, 4, 19
    kw, vw, kh, vh, q = r(B, Hkv, Nw, D), r(B, Hkv, Nw, D), r(B, Hkv, Nh, D), r(B, Hkv, Nh, D), r(B, Hq, 1, D)
    kw[..., first:first + n_out] *= 4  # adjacent channels are the largest, so they are protected together
    vw[..., first:first + n_out] *= 4
    warm = akv.quantize_kv(kw, vw, bk, bv, 32, G, outlier_fraction=(n_out + 0.5) / D)
    want = torch.arange(first, first + n_out, device="cuda")
    assert warm.n_out == n_out and bool((warm.v_oidx.sort(-1).values == want).all())
    kd, vd = akv.dequantize(warm)
    k, v = (torch.cat(x, dim=2).double().repeat_interleave(Hq // Hkv, dim=1) for x in ((kd, kh), (vd, vh)))
    p = torch.softmax((q.double() @ k.transpose(2, 3).contiguous()) * D ** -0.5, dim=-1)
    out = akv.decode_attention(q, kh, vh, warm)
    # 16-bit probabilities, values and output: two or three roundings of 2^-11
    exp = p @ v
    assert float((out.double() - exp).norm() / exp.norm()) <= 1e-3
