"""The whole-chunk dequant kernel against the element-by-element one (which takes outputs off
a 16-byte boundary): odd lengths around a workgroup's tokens, strides, event blocks, output
slots, outlier channels, every width and output dtype; values include infinities and NaN."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu
DT = {"fp16": (torch.float16, 0), "bf16": (torch.bfloat16, 1), "fp32": (torch.float32, 2)}


def _u8(shape, g):
    return torch.randint(0, 256, shape, generator=g, dtype=torch.uint8).cuda()


def _meta(shape, g, dt):
    x = torch.randn(shape, generator=g)
    x.view(-1)[::97] = float("inf")
    x.view(-1)[5::211] = float("nan")
    x.view(-1)[3::89] *= 1e-7
    return x.to(dt).cuda()


def _run(d, B, H, D, out_dt, rows, shift, extra):
    from akv import _native as nat
    dt, code = DT[out_dt]
    outs = [torch.zeros(rows * D + 16, dtype=dt, device="cuda") for _ in range(2)]
    ws = torch.zeros(256, dtype=torch.uint8, device="cuda")
    a = nat.DequantArgs()
    a.abi_version, a.B, a.Hkv, a.D, a.out_dtype, a.warm = nat.ABI_VERSION, B, H, D, code, d
    a.k_out, a.v_out = (o.data_ptr() + shift * o.element_size() for o in outs)
    a.workspace = ws.data_ptr()
    for k, v in extra.items():
        setattr(a, k, v)
    nat.check(nat.load().akv_dequant_unpack(ctypes.byref(a), nat.stream_of(ws)), "dequant")
    torch.cuda.synchronize()
    return [o[shift:shift + rows * D].clone() for o in outs]


def _same(got, ref):
    for a, b in zip(got, ref):
        nan = torch.isnan(a)
        assert torch.equal(nan, torch.isnan(b))
        iv = torch.int32 if a.element_size() == 4 else torch.int16
        a, b = a.masked_fill(nan, 0).view(iv), b.masked_fill(nan, 0).view(iv)
        assert torch.equal(a, b), f"{int((a != b).sum())} of {a.numel()} differ"


@pytest.mark.parametrize("D,bk,bv,T,Gv,n_out,n,cap,events,out_dt", [
    (128, 3, 2, 32, 32, 0, 64, 64, False, "fp16"), (128, 4, 3, 48, 128, 2, 65, 65, False, "fp32"),
    (64, 2, 3, 1, 64, 1, 129, 200, True, "fp16"), (96, 8, 4, 16, 8, 0, 63, 63, False, "fp32"),
    (96, 3, 3, 16, 32, 0, 63, 63, False, "fp16"), (128, 3, 3, 7, 128, 3, 1, 5, True, "fp32")])
def test_affine_chunks(D, bk, bv, T, Gv, n_out, n, cap, events, out_dt):
    from akv import _native as nat
    announce(f"dequant chunks D={D} bits={bk}/{bv} T={T} Gv={Gv} n_out={n_out} n={n}/{cap} events={events}")
    g = torch.Generator().manual_seed(D + n)
    B, H, nblk = 2, 3, 9 if events else -(-n // T)
    row = (lambda b: D * b // 8)
    t = dict(k_codes=_u8((B, H, cap, row(bk)), g), v_codes=_u8((B, H, cap, row(bv)), g),
             k_scale=_meta((B, H, nblk, D), g, torch.float16), k_zero=_meta((B, H, nblk, D), g, torch.float16),
             v_scale=_meta((B, H, cap, D // Gv), g, torch.float16), v_zero=_meta((B, H, cap, D // Gv), g, torch.float16))
    if n_out:
        pick = torch.stack([torch.randperm(D, generator=g)[:n_out] for _ in range(2 * B * nblk)]).cuda()
        t.update(k_oidx=pick[: B * nblk].contiguous(), v_oidx=pick[B * nblk:].contiguous(),
                 k_odata=_meta((B, H, cap, n_out), g, torch.float16), v_odata=_meta((B, H, cap, n_out), g, torch.float16))
    d = nat.WarmDesc()
    d.kind, d.bits_k, d.bits_v, d.n_warm, d.token_stride = nat.WARM_AFFINE, bk, bv, n, cap
    d.block_t, d.group_v, d.n_out = T, Gv, n_out
    for k, x in t.items():
        setattr(d, k, x.data_ptr())
    extra, rows = {}, n
    if events:
        rows = 2 * n + 3
        blk = torch.randint(0, nblk, (n,), generator=g, dtype=torch.int32).cuda()
        slot = torch.randperm(rows, generator=g)[:n].cuda()
        extra = dict(block_of_token=blk.data_ptr(), n_blocks=nblk, out_slot=slot.data_ptr(), out_tokens=rows)
    ref = _run(d, B, H, D, out_dt, B * H * rows, 1, extra)
    _same(_run(d, B, H, D, out_dt, B * H * rows, 0, extra), ref)


@pytest.mark.parametrize("D,bits,gs,meta,sym,n,cap,out_dt", [
    (128, 4, 64, "fp16", 0, 65, 80, "fp16"), (64, 2, 128, "fp32", 1, 33, 33, "bf16"),
    (128, 8, 32, "bf16", -1, 64, 64, "fp32"), (64, 4, 32, "fp32", -1, 127, 127, "fp16")])
def test_legacy_chunks(D, bits, gs, meta, sym, n, cap, out_dt):
    from akv import _native as nat
    announce(f"dequant legacy chunks D={D} bits={bits} gs={gs} meta={meta} sym={sym} n={n}/{cap}")
    g = torch.Generator().manual_seed(D + n)
    H, pD = 5, -(-D // gs) * gs
    dt, code = DT[meta]
    kc, vc = _u8((H, cap, pD * bits // 8), g), _u8((H, cap, pD * bits // 8), g)
    m = [_meta((H, cap, pD // gs), g, dt) for _ in range(4)]
    if sym == -1:
        m[1].zero_()  # the keys' branch is detected as symmetric, the values' is not
    d = nat.WarmDesc()
    d.kind, d.bits_k, d.bits_v, d.n_warm, d.token_stride = nat.WARM_LEGACY, bits, bits, n, cap
    d.k_codes, d.v_codes = kc.data_ptr(), vc.data_ptr()
    d.k_scale, d.k_zero, d.v_scale, d.v_zero = (x.data_ptr() for x in m)
    d.group_size, d.meta_dtype, d.warm_heads, d.legacy_sym = gs, code, H, sym
    ref = _run(d, 1, H, D, out_dt, H * n, 1, {})
    _same(_run(d, 1, H, D, out_dt, H * n, 0, {}), ref)
