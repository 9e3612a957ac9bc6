"""Batches and block counts past what the tile kernels' grids hold quantize as smaller ones do."""
import ctypes

import pytest
import torch

from gpu_util import announce


def _args(B, n, T, n_out=1, D=64):
    from akv import _native as nat
    a = nat.QuantArgs()
    a.abi_version, a.B, a.H, a.D, a.n_src, a.n_sel = nat.ABI_VERSION, B, 1, D, n, n
    a.in_dtype, a.layout = nat.DT_F16, nat.QUANT_AFFINE
    a.bits_k, a.bits_v, a.block_t, a.group_v, a.n_out = 3, 3, T, 32, n_out
    a.k = a.v = a.k_codes = a.v_codes = a.k_scale = a.k_zero = a.v_scale = a.v_zero = 0x10000  # planning only
    a.k_oidx = a.v_oidx = a.k_odata = a.v_odata = 0x20000
    return nat.load().akv_quant_workspace_bytes(ctypes.byref(a))


def test_the_plan_knows_the_grid():
    """Scratch is planned for the tile kernels alone: none where they do not take the call."""
    assert _args(32767, 1024, 1024) > 0
    assert _args(32768, 1024, 1024) == 0  # keys and values: 65,536 tensors
    assert _args(1, 1024 * 65535, 1024) > 0
    assert _args(1, 1024 * 65536, 1024) == 0


@pytest.mark.parametrize("n,T,scratch", [(512, 512, False), (513, 512, False), (512, 4096, False), (513, 513, True),
                                         (4000, 4096, True), (4000, 32, False)])
def test_short_blocks_need_no_scratch(n, T, scratch):
    """The binding asks for scratch past 512 tokens of a block and of the selection only."""
    assert (_args(2, n, T) > 0) == scratch


@pytest.mark.gpu
@pytest.mark.parametrize("n_out", [0, 1])
def test_many_sequences(n_out):
    import akv
    announce(f"quantize 33,000 sequences, n_out={n_out}")
    B, n, D = 33000, 5, 64
    g = torch.Generator(device="cuda").manual_seed(3)
    k, v = (torch.randn(B, 1, n, D, generator=g, device="cuda").half() for _ in range(2))
    f = n_out / D if n_out else 0.0
    whole = akv.quantize_kv(k, v, 3, 4, 32, 32, outlier_fraction=f)
    for a in (0, 1234, B - 8):
        part = akv.quantize_kv(k[a:a + 8].contiguous(), v[a:a + 8].contiguous(), 3, 4, 32, 32, outlier_fraction=f)
        for name in ("k_codes", "k_scale", "k_zero", "v_codes", "v_scale", "v_zero") + (
                ("k_oidx", "k_odata", "v_oidx", "v_odata") if n_out else ()):
            assert torch.equal(getattr(whole, name)[a:a + 8], getattr(part, name)), (a, name)
