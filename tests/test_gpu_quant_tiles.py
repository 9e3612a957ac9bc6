"""The whole-tile quantize kernels: block lengths on each side of their statistics rules (32,
128, 512 tokens; chunked partials with a workspace), remainders, dtypes, outlier channels.
Bit-exact with the oracle, and with the element-by-element kernel (which takes inputs off a
16-byte boundary) on infinities, NaN and signed zeros."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import announce, bits_equal, to_dev
from oracle import affine as oaff

pytestmark = pytest.mark.gpu
DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
KEYS = ("k_codes", "k_scale", "k_zero", "v_codes", "v_scale", "v_zero")
OUT_KEYS = ("k_oidx", "k_odata", "v_oidx", "v_odata")


def _inputs(B, H, N, D, dtype, seed, heavy):
    rng = np.random.default_rng(seed)
    k = rng.standard_normal((B, H, N, D)).astype(np.float32)
    v = rng.standard_normal((B, H, N, D)).astype(np.float32)
    if heavy:  # well-separated channel norms: the choice does not hang on the order of a sum
        ch = rng.permutation(D)[:4]
        k[..., ch] *= np.array([16, 12, 9, 6], np.float32)
        v[..., ch] *= np.array([9, 16, 6, 12], np.float32)
    t = [to_dev(x).to(DT[dtype]) for x in (k, v)]
    return t, [x.float().cpu().numpy() for x in t]


@pytest.mark.parametrize("dtype,D,T,G,bk,bv,frac,N", [
    ("fp16", 128, 33, 32, 3, 4, 0.0, 100),       # two tiles a block, one token in the second
    ("fp16", 128, 128, 64, 2, 3, 0.0, 321),      # a block's tiles held in registers
    ("fp16", 64, 129, 64, 3, 3, 0.0, 300),       # one tile more; 24-byte rows off 16-byte boundaries
    ("fp16", 128, 512, 128, 4, 2, 0.0, 700),     # the longest block of one workgroup
    ("fp16", 128, 513, 128, 3, 3, 0.0, 513),     # the shortest with chunked statistics
    ("fp16", 128, 3000, 128, 3, 3, 0.02, 2999),  # chunks, outlier norms in the workspace
    ("fp16", 64, 40000, 64, 4, 4, 0.0, 33333),   # more than 64 chunks' worth of tokens
    ("bf16", 128, 1500, 128, 4, 2, 0.02, 1500),
    ("bf16", 64, 1, 64, 4, 2, 0.02, 5),          # one-token blocks
    ("bf16", 128, 32, 32, 2, 4, 0.01, 77),
    ("fp32", 128, 700, 128, 4, 3, 0.0, 1401),
    ("fp32", 64, 32, 32, 3, 2, 0.04, 65),
    ("fp16", 128, 600, 128, 8, 8, 0.0, 601),     # raw codes
])
def test_tiles_match_oracle(dtype, D, T, G, bk, bv, frac, N):
    import akv
    from oracle.fp import round_bf16
    announce(f"tiles {dtype} D={D} T={T} G={G} bits={bk}/{bv} f={frac} N={N}")
    (k, v), (kn, vn) = _inputs(2, 3, N, D, dtype, T + N, frac > 0)
    if dtype == "fp16":
        kn, vn = kn.astype(np.float16), vn.astype(np.float16)
    ref = oaff.quantize_kv_blocked(kn, vn, bk, bv, T=T, G=G, outlier_fraction=frac,
                                   dt="bfloat16" if dtype == "bf16" else None)
    wt = akv.quantize_kv(k, v, bk, bv, block_t=T, group_v=G, outlier_fraction=frac)
    for name in KEYS + (OUT_KEYS if frac else ()):
        bits_equal(getattr(wt, name), ref[name])


def _raw(k, v, bk, bv, T, G, n_out, sel, layout, ws, shift):
    """akv_quant_pack(_ws) on inputs `shift` elements past a 16-byte boundary."""
    from akv import _native as nat
    from akv.warm_tier import packed_row_bytes
    lib = nat.load()
    B, H, N, D = k.shape
    ins = []
    for x in (k, v):
        buf = torch.empty(x.numel() + 16, dtype=x.dtype, device="cuda")
        buf[shift:shift + x.numel()] = x.reshape(-1)
        ins.append(buf)
    n = N if sel is None else sel.shape[1]
    affine = layout == nat.QUANT_AFFINE
    pD = -(-D // G) * G
    nblk = -(-n // T)
    row = (lambda b: packed_row_bytes(D, b)) if affine else (lambda b: pD if b in (3, 8) else pD * b // 8)
    mdt = torch.float16 if affine else k.dtype
    mk = (lambda *s, dt: torch.zeros(*s, dtype=dt, device="cuda"))
    out = {"k_codes": mk(B, H, n, row(bk), dt=torch.uint8), "v_codes": mk(B, H, n, row(bv), dt=torch.uint8)}
    kshape = (B, H, nblk, D) if affine else (B, H, n, pD // G)
    for name, s in (("k_scale", kshape), ("k_zero", kshape), ("v_scale", (B, H, n, pD // G)),
                    ("v_zero", (B, H, n, pD // G))):
        out[name] = mk(*s, dt=mdt)
    if n_out:
        out.update(k_oidx=mk(B, nblk, n_out, dt=torch.int64), v_oidx=mk(B, nblk, n_out, dt=torch.int64),
                   k_odata=mk(B, H, n, n_out, dt=torch.float16), v_odata=mk(B, H, n, n_out, dt=torch.float16))
    a = nat.QuantArgs()
    a.abi_version, a.B, a.H, a.D = nat.ABI_VERSION, B, H, D
    a.in_dtype, a.layout = nat.dtype_code(k.dtype), layout
    a.k, a.v = (x.data_ptr() + shift * x.element_size() for x in ins)
    a.n_src, a.n_sel = N, n
    a.sel = sel.data_ptr() if sel is not None else None
    a.bits_k, a.bits_v, a.block_t, a.group_v, a.n_out = bk, bv, T, G, n_out
    for name, t in out.items():
        setattr(a, name, t.data_ptr())
    need = lib.akv_quant_workspace_bytes(ctypes.byref(a))
    assert need >= 0
    w = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
    args = (ctypes.byref(a), w.data_ptr(), need) if ws and need else (ctypes.byref(a), None, 0)
    nat.check(lib.akv_quant_pack_ws(*args, nat.stream_of(k)), "quant")
    torch.cuda.synchronize()
    return out, need


@pytest.mark.parametrize("dtype", ["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("D,T,G,bk,bv,n_out,layout,picked", [
    (128, 1200, 128, 3, 4, 2, "AFFINE", True), (64, 700, 32, 4, 2, 0, "AFFINE", False),
    (128, 64, 64, 2, 3, 1, "AFFINE", True), (128, 32, 64, 4, 2, 0, "ARENA", False),
    (64, 32, 128, 2, 8, 0, "ARENA", True), (128, 32, 32, 3, 8, 0, "TOKEN_GROUPS", False)])
def test_tiles_match_the_element_kernel(dtype, D, T, G, bk, bv, n_out, layout, picked):
    """Values no oracle case holds: whole channels and tokens of NaN, infinities of both signs,
    zeros of both signs, subnormals; with and without the workspace."""
    from akv import _native as nat
    announce(f"element kernel {dtype} {layout} D={D} T={T} G={G} bits={bk}/{bv} n_out={n_out}")
    (k, v), _ = _inputs(1, 3, 1501, D, dtype, D + T, n_out > 0)
    inf = float("inf")
    for x in (k, v):
        x[0, 0, 7, :] = float("nan")
        x[0, 0, :, 5] = float("nan")
        x[0, 0, 40, 9], x[0, 1, 41, 9], x[0, 1, 42, 10] = inf, -inf, float("nan")
        x[0, 1, :, 11], x[0, 1, 100:200, 12] = 0.0, -0.0
        x[0, 2, ::2, 13], x[0, 2, 1::2, 13] = 0.0, -0.0
        x[0, 2, :, 14] = x[0, 2, :, 14] * 1e-7
        x[0, 2, 50, :] = -0.0
    if n_out:  # the choice must not meet NaN norms in every head
        k[0, 0, :, 5] = v[0, 0, :, 5] = 1.0
    sel = None
    if picked:
        g = torch.Generator().manual_seed(3)
        sel = torch.sort(torch.randperm(1501, generator=g)[:1333]).values.view(1, -1).cuda()
    lay = getattr(nat, "QUANT_" + layout)
    ref, none = _raw(k, v, bk, bv, T, G, n_out, sel, lay, False, 1)
    assert none == 0  # off the boundary: the element kernel, which takes no workspace
    for ws in (False, True):
        got, need = _raw(k, v, bk, bv, T, G, n_out, sel, lay, ws, 0)
        assert (need > 0) == (T > 512)
        for name in ref:
            a, b = got[name].contiguous(), ref[name].contiguous()
            if a.is_floating_point() and name != "k_odata" and name != "v_odata":
                nan = torch.isnan(a) & torch.isnan(b)  # NaN payloads aside
                a, b = a.masked_fill(nan, 0), b.masked_fill(nan, 0)
            iv = {1: torch.uint8, 2: torch.int16, 4: torch.int32, 8: torch.int64}[a.element_size()]
            a, b = a.view(iv), b.view(iv)
            assert torch.equal(a, b), f"{name}: {int((a != b).sum())} of {a.numel()} differ (ws={ws})"
