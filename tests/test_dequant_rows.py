"""Output rows of the dequantizer: ``out_tokens`` belongs to output slots and says nothing without
them, whatever a caller left there; outputs of more rows than tokens have an entry point."""
import ctypes

import pytest
import torch

from gpu_util import announce


def _legacy(n, cap, B=1, H=3, D=64):
    from akv import _native as nat
    a = nat.DequantArgs()
    a.abi_version, a.B, a.Hkv, a.D, a.out_dtype = nat.ABI_VERSION, B, H, D, nat.DT_F16
    w = a.warm
    w.kind, w.bits_k, w.bits_v, w.n_warm, w.token_stride = nat.WARM_LEGACY, 4, 4, n, cap
    w.group_size, w.meta_dtype, w.warm_heads, w.legacy_sym = 32, nat.DT_F16, H, 0
    w.k_codes = w.v_codes = w.k_scale = w.k_zero = w.v_scale = w.v_zero = 0x10000  # no output: never read
    return a, nat


@pytest.mark.parametrize("left", [0, 7, 16, 999])
def test_out_tokens_without_slots(left):
    a, nat = _legacy(16, 16)
    a.out_tokens = left
    assert nat.load().akv_dequant_unpack(ctypes.byref(a), None) == nat.AKV_OK, nat.load().akv_last_error()


def test_rows_are_checked():
    a, nat = _legacy(16, 16)
    lib = nat.load()
    assert lib.akv_dequant_unpack_rows(ctypes.byref(a), 16, None) == nat.AKV_OK
    assert lib.akv_dequant_unpack_rows(ctypes.byref(a), 15, None) == nat.AKV_E_SHAPE
    assert lib.akv_dequant_unpack_rows(ctypes.byref(a), 0, None) == nat.AKV_E_SHAPE
    assert lib.akv_dequant_unpack_rows(None, 16, None) == nat.AKV_E_INVALID
    a.out_slot = 0x20000
    assert lib.akv_dequant_unpack_rows(ctypes.byref(a), 16, None) == nat.AKV_E_INVALID


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [33, 40])
@pytest.mark.parametrize("shift", [0, 1])  # whole chunks / element by element
def test_dense_and_strided_outputs(rows, shift):
    announce(f"dequant rows {rows} shift {shift}")
    n, H, D = 33, 3, 64
    a, nat = _legacy(n, n, H=H, D=D)
    g = torch.Generator(device="cuda").manual_seed(rows)
    codes = [torch.randint(0, 256, (H, n, D // 2), generator=g, device="cuda", dtype=torch.uint8) for _ in range(2)]
    meta = [torch.randn(H, n, D // 32, generator=g, device="cuda").half() for _ in range(4)]
    w = a.warm
    w.k_codes, w.v_codes = (x.data_ptr() for x in codes)
    w.k_scale, w.k_zero, w.v_scale, w.v_zero = (x.data_ptr() for x in meta)
    want = []
    for c, s, z in ((codes[0], meta[0], meta[1]), (codes[1], meta[2], meta[3])):
        u = torch.stack([c >> 4, c & 15], dim=-1).view(H, n, D // 32, 32).float()
        want.append((u * s.float().unsqueeze(-1) + z.float().unsqueeze(-1)).half().view(H, n, D))
    lib = nat.load()
    for r in (n, rows):
        outs = [torch.full((H * r * D + 8,), 9.0, dtype=torch.float16, device="cuda") for _ in range(2)]
        a.k_out, a.v_out = (o.data_ptr() + 2 * shift for o in outs)
        a.out_tokens = 35  # left over from another call
        rc = (lib.akv_dequant_unpack(ctypes.byref(a), nat.stream_of(codes[0])) if r == n else
              lib.akv_dequant_unpack_rows(ctypes.byref(a), r, nat.stream_of(codes[0])))
        nat.check(rc, "dequant")
        for o, e in zip(outs, want):
            o = o[shift:shift + H * r * D].view(H, r, D)
            assert torch.equal(o[:, :n], e) and bool((o[:, n:] == 9.0).all())
