"""The KIVI baselines of akv/baselines.py on the device.

``KIVICache`` (akv/baselines.py:249-403) quantizes the tokens that overflow a
full-precision residual window; ``KIVIFusedCache`` (:426-510) is its fused-kernel
cost profile: each overflow chunk is quantized once, appended, and dequantized once
into a float16 working copy.  The quantizer (``_quantize_tensor``, :345-370) is fp32
min / max per (row, group) of the last axis, scale clamped at 1e-10, codes
rounded half-to-even; for KIVICache it is one ``akv_quant_pack`` launch (layout
``AKV_QUANT_ARENA`` on fp32 input, which is that arithmetic) and the dequant
(``_dequantize_tensor``, :372-380: fp32 ``codes * s + z`` cast to fp16) one
``akv_dequant_unpack`` launch -- both bit-exact with the reference -- and for
KIVIFusedCache one ``akv_kivi_append`` launch does both for an overflow's keys and values.

Storage: per layer and for K and V, the codes bit-packed (2 / 4 / 8 bits; 4-bit
high nibble first, 2-bit MSB first) in ``[B * H][capacity][pD * bits / 8]`` and the
fp32 scales / zeros in ``[B * H][capacity][G]``, tokens in order, the capacity
doubling as the cache grows.  The reference keeps unpacked uint8 codes and
concatenates chunk after chunk along its flattened row axis
(``_concat_quant_chunks``, :513-535); the ``_quant_keys`` / ``_quant_values``
tiers here (indexable like those dicts: 'data', 'scales', 'zeros', 'shape', ...)
hold the packed codes in (batch, head, token) order instead.
``memory_bytes`` counts what the dicts and the residual hold, as the reference does.

``KIVIFusedCache.fused_attention`` (not in the reference: the throughput leg that
compares the baseline on the same kernels) is one ``akv_decode_attn`` launch over
the packed tier, read in place (legacy layout, one tier per (batch, head), fp16
copies of the scales / zeros kept beside the fp32 ones) and the residual window.

Head_dim 64 or 128, group sizes 32 / 64 / 128 and 2 / 4 / 8 bits are supported, as
for every quantizer of this build; other shapes raise ``NotImplementedError``.
"""
from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Optional

import torch

from . import _native as nat
from ._legacy import legacy_desc, padded_dim
from .row_moves import RowMoves, row_moves


@dataclass
class KIVIConfig:
    """akv/baselines.py:236-246."""
    key_bits: int = 2
    value_bits: int = 2
    group_size: int = 128
    residual_length: int = 128


@dataclass
class KIVIFusedConfig(KIVIConfig):
    """akv/baselines.py:406-423."""


def _check_shape(D: int, bits: int, gs: int):
    if bits not in (2, 4, 8):
        raise NotImplementedError(f"the MI355X KIVI tier packs 2, 4 or 8 bits, got {bits}")
    if D not in (64, 128) or gs not in (32, 64, 128):
        raise NotImplementedError("the MI355X KIVI tier takes head_dim 64 or 128 and group_size 32, 64 or 128")


def quantize_rows(x: torch.Tensor, bits: int, group_size: int):
    """KIVICache._quantize_tensor (akv/baselines.py:345-370) for x (B, H, n, D):
    packed codes (B * H, n, pD * bits / 8) uint8 and fp32 scales / zeros
    (B * H, n, G), one launch."""
    nat.require_device(x)
    B, H, n, D = x.shape
    _check_shape(D, bits, group_size)
    xf = nat.dev_contig(x.float())
    pD = padded_dim(D, group_size)
    G = pD // group_size
    codes = torch.empty(1, B * H, n, pD * bits // 8, dtype=torch.uint8, device=x.device)
    sc = torch.empty(1, B * H, n, G, dtype=torch.float32, device=x.device)
    ze = torch.empty_like(sc)
    if n:
        a = nat.QuantArgs()
        a.abi_version = nat.ABI_VERSION
        a.B, a.H, a.D = 1, B * H, D
        a.in_dtype = nat.DT_F32
        a.layout = nat.QUANT_ARENA
        a.k = xf.data_ptr()
        a.n_src = a.n_sel = n
        a.bits_k = a.bits_v = bits
        a.block_t = 32
        a.group_v = group_size
        a.k_codes, a.k_scale, a.k_zero = codes.data_ptr(), sc.data_ptr(), ze.data_ptr()
        nat.check(nat.load().akv_quant_pack(ctypes.byref(a), nat.stream_of(xf)), "KIVI quantize")
    return codes[0], sc[0], ze[0]


def dequantize_rows(codes: torch.Tensor, sc: torch.Tensor, ze: torch.Tensor, bits: int, group_size: int,
                    D: int, n: Optional[int] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """KIVICache._dequantize_tensor (akv/baselines.py:372-380): (R, n, D) float16 of
    fp32 codes * s + z, for contiguous codes (R, S, pD * bits / 8) and fp32 meta
    (R, S, G) of which the first n <= S tokens of each row are read (n = S unless
    given), in one launch; into the first n of the rows of ``out`` (R, >= n, D) if given."""
    R, S = codes.shape[0], codes.shape[1]
    n = S if n is None else n
    if out is None:
        out = torch.empty(R, n, D, dtype=torch.float16, device=codes.device)
    if R * n == 0:
        return out
    keep = []
    desc = legacy_desc(codes, sc, ze, codes, sc, ze, bits, group_size, S, D, warm_heads=R, sym=0, keep=keep)
    desc.n_warm = n
    desc.token_stride = S
    a = nat.DequantArgs()
    a.abi_version = nat.ABI_VERSION
    a.B, a.Hkv, a.D = 1, R, D
    a.out_dtype = nat.DT_F16
    a.warm = desc
    a.k_out = out.data_ptr()
    nat.check(nat.load().akv_dequant_unpack_rows(ctypes.byref(a), out.shape[1], nat.stream_of(out)), "KIVI dequantize")
    return out


class _Tier:
    """One layer's quantized K or V: packed codes and fp32 (and, for KIVIFusedCache's
    attention, fp16) scales / zeros per (batch * head, token), tokens in order."""

    def __init__(self, B: int, H: int, D: int, bits: int, gs: int, device):
        self.B, self.H, self.rows, self.D, self.bits, self.gs = B, H, B * H, D, bits, gs
        pD = padded_dim(D, gs)
        self.row_bytes, self.G = pD * bits // 8, pD // gs
        self.n, self.cap, self.dirty = 0, 0, 0
        self.device = device
        self.codes = self.sc = self.ze = self.sc16 = self.ze16 = None

    def reserve(self, n: int):
        """Room for n more rows.  Rows past the tier read as zeros: those of a grown tier, up to row
        ``dirty``, have to be cleared by the launch that appends."""
        if self.n + n <= self.cap:
            return
        cap = max(64, self.cap)
        while cap < self.n + n:
            cap *= 2
        mv, grown = row_moves(), {}
        for name, width, dtype in (("codes", self.row_bytes, torch.uint8), ("sc", self.G, torch.float32),
                                   ("ze", self.G, torch.float32), ("sc16", self.G, torch.float16),
                                   ("ze16", self.G, torch.float16)):
            old, new = getattr(self, name), torch.empty(self.rows, cap, width, dtype=dtype, device=self.device)
            if old is not None:
                mv.copy(new.unsqueeze(0), old.unsqueeze(0), self.n)
            grown[name] = new
        mv.run()
        self.__dict__.update(grown, cap=cap, dirty=cap)

    def fill(self, codes, sc, ze):
        """A tier that holds these tokens and no float16 meta (KIVICache makes one per overflow)."""
        self.codes, self.sc, self.ze = codes, sc, ze
        self.n = self.cap = codes.shape[1]
        return self

    def __getitem__(self, key: str):
        """The reference's quant dict entries over the tier ('data', 'scales', 'zeros':
        rows in (batch, head, token) order; 'shape', 'bits', 'group_size')."""
        n = self.n
        if key == "data":
            return self.codes[:, :n].reshape(self.rows * n, self.row_bytes)
        if key in ("scales", "zeros"):
            return (self.sc if key == "scales" else self.ze)[:, :n].reshape(self.rows * n, self.G)
        return {"shape": (self.B, self.H, n, self.D), "bits": self.bits, "group_size": self.gs}[key]

    def dequantize(self) -> torch.Tensor:
        """(B, H, n, D) float16, one launch over the tier in place."""
        return dequantize_rows(self.codes, self.sc, self.ze, self.bits, self.gs, self.D,
                               n=self.n).view(self.B, self.H, self.n, self.D)

    def nbytes(self) -> int:
        n = self.n
        return self.rows * n * (self.row_bytes + 2 * 4 * self.G)


class KIVICache:
    """akv/baselines.py:249-403: every overflow re-quantizes the merged history and
    every update dequantizes the whole quantized tier."""

    def __init__(self, config: Optional[KIVIConfig] = None):
        self.config = config or KIVIConfig()
        self._quant_keys: dict = {}      # layer -> _Tier
        self._quant_values: dict = {}
        self._residual_keys: dict = {}
        self._residual_values: dict = {}
        self._seq_lens: dict = {}

    def update(self, key_states: torch.Tensor, value_states: torch.Tensor, layer_idx: int,
               attention_weights: Optional[torch.Tensor] = None):
        """akv/baselines.py:268-289: (B, H, N, D) in, the layer's full K / V out."""
        cfg = self.config
        nat.require_device(key_states, value_states)
        if layer_idx not in self._residual_keys:
            rk, rv = key_states, value_states
            self._seq_lens[layer_idx] = key_states.shape[2]
        else:
            rk = torch.cat([self._residual_keys[layer_idx], key_states], dim=2)
            rv = torch.cat([self._residual_values[layer_idx], value_states], dim=2)
            self._seq_lens[layer_idx] += key_states.shape[2]
        self._residual_keys[layer_idx], self._residual_values[layer_idx] = rk, rv
        views = self._quantize_overflow(layer_idx) if rk.shape[2] > cfg.residual_length else None
        return self._get_full_kv(layer_idx) if views is None else views

    def _new_tier(self, x: torch.Tensor, bits: int) -> "_Tier":
        B, H, _, D = x.shape
        return _Tier(B, H, D, bits, self.config.group_size, x.device)

    def _quantize_overflow(self, layer_idx: int):
        """akv/baselines.py:291-322: quantize the overflow; merge by dequantizing the
        old tier, concatenating and quantizing the whole again."""
        cfg = self.config
        res_k, res_v = self._residual_keys[layer_idx], self._residual_values[layer_idx]
        n_q = res_k.shape[2] - cfg.residual_length
        tk, tv = res_k[:, :, :n_q], res_v[:, :, :n_q]
        if layer_idx in self._quant_keys:
            tk = torch.cat([self._quant_keys[layer_idx].dequantize(), tk], dim=2)
            tv = torch.cat([self._quant_values[layer_idx].dequantize(), tv], dim=2)
        kt = self._new_tier(tk, cfg.key_bits).fill(*quantize_rows(tk, cfg.key_bits, cfg.group_size))
        vt = self._new_tier(tv, cfg.value_bits).fill(*quantize_rows(tv, cfg.value_bits, cfg.group_size))
        self._quant_keys[layer_idx], self._quant_values[layer_idx] = kt, vt
        self._residual_keys[layer_idx] = res_k[:, :, n_q:].contiguous()
        self._residual_values[layer_idx] = res_v[:, :, n_q:].contiguous()

    def _get_full_kv(self, layer_idx: int):
        """akv/baselines.py:324-343."""
        rk, rv = self._residual_keys[layer_idx], self._residual_values[layer_idx]
        if layer_idx in self._quant_keys:
            return (torch.cat([self._quant_keys[layer_idx].dequantize(), rk], dim=2),
                    torch.cat([self._quant_values[layer_idx].dequantize(), rv], dim=2))
        return rk, rv

    def get_seq_length(self, layer_idx: int = 0) -> int:
        return self._seq_lens.get(layer_idx, 0)

    def reset(self):
        self._quant_keys.clear()
        self._quant_values.clear()
        self._residual_keys.clear()
        self._residual_values.clear()
        self._seq_lens.clear()

    def memory_bytes(self) -> int:
        """akv/baselines.py:392-403: quantized tiers (codes as stored here, packed) plus
        the residual windows."""
        total = sum(t.nbytes() for t in self._quant_keys.values()) + sum(t.nbytes() for t in self._quant_values.values())
        total += sum(k.nbytes for k in self._residual_keys.values()) + sum(v.nbytes for v in self._residual_values.values())
        return int(total)

    def __len__(self):
        return self.get_seq_length()


class KIVIFusedCache(KIVICache):
    """akv/baselines.py:426-510: incremental quantization of each overflow chunk.  The
    reference keeps a float16 working copy extended by that chunk's dequant; the same values
    come from the packed tier here, dequantized straight into each returned view."""

    def __init__(self, config: Optional[KIVIFusedConfig] = None):
        super().__init__(config or KIVIFusedConfig())
        self._dequant_keys_cache: dict = {}    # layer -> the tier its dequantized rows come from
        self._dequant_values_cache: dict = {}
        self._ws: dict = {}  # per-device decode workspace of fused_attention

    def _quantize_overflow(self, layer_idx: int):
        """akv/baselines.py:455-496; returns the layer's full K / V.  One launch quantizes,
        appends and dequantizes the overflow of both tensors and writes its rows of the view, one
        cuts the residuals and completes the view.  Everything is allocated before the first
        launch, and tiers and residuals change after the last: a call that fails before leaves
        the tokens in the residual window."""
        cfg = self.config
        res = (self._residual_keys[layer_idx], self._residual_values[layer_idx])
        for bits, r in ((cfg.key_bits, res[0]), (cfg.value_bits, res[1])):
            _check_shape(r.shape[3], bits, cfg.group_size)
        n = res[0].shape[2] - cfg.residual_length  # the keys say how many tokens of both leave
        if res[0].shape[3] != res[1].shape[3]:
            raise ValueError("KIVIFusedCache takes keys and values of one head_dim")
        if res[0].shape[:2] != res[1].shape[:2] or res[1].shape[2] < n:
            raise RuntimeError("keys and values of different heads, or fewer values than the overflow's keys")
        sides, args, mv = [], [], row_moves()
        for bits, tiers, r in ((cfg.key_bits, self._quant_keys, res[0]), (cfg.value_bits, self._quant_values, res[1])):
            B, H, _, D = r.shape
            x, left = r[:, :, :n], r[:, :, n:]
            tier = tiers[layer_idx] if layer_idx in tiers else self._new_tier(x, bits)
            tier.reserve(n)
            if x.dtype not in (torch.float16, torch.bfloat16, torch.float32):
                x = x.float()
            e = x.element_size()
            if x.stride(3) != 1 or x.data_ptr() % 16 or any(st * e % 16 for st in x.stride()[:3]):
                x = nat.dev_contig(x)
            dt = torch.promote_types(torch.float16, left.dtype)
            view = old = None
            if mv.takes(dt, left) and dt in (torch.float16, torch.float32):
                view, old = self._new_view(tier, tier.n, n, left, dt, mv)
            if mv.takes(left.dtype, left) and left.stride(3) == 1:
                kept = torch.empty(left.shape, dtype=left.dtype, device=left.device)
                mv.copy(kept, left, left.shape[2])
            else:
                kept = left.contiguous()
            sides.append((tier, view, old, kept))
            args.append((x, B, H, D, n, dt, nat.KiviSide(
                x.data_ptr(), x.stride(0) * e, x.stride(1) * e, x.stride(2) * e, tier.codes.data_ptr(),
                tier.sc.data_ptr(), tier.ze.data_ptr(), tier.sc16.data_ptr(), tier.ze16.data_ptr(),
                None if view is None else view.data_ptr(), tier.cap, tier.n, tier.dirty,
                0 if view is None else view.shape[2], bits, 0)))
        groups = [args] if args[0][1:6] == args[1][1:6] and args[0][0].dtype == args[1][0].dtype else [args[:1], args[1:]]
        for g in groups:
            x, B, H, D, n, dt, _ = g[0]
            arr = (nat.KiviSide * len(g))(*(s[6] for s in g))
            nat.check(nat.load().akv_kivi_append(
                arr, len(g), B, H, D, n, nat.dtype_code(x.dtype), cfg.group_size,
                nat.DT_F16 if dt == torch.float16 else nat.DT_F32, nat.stream_of(x)), "KIVI append")
        for tier, view, old, _ in sides:
            if view is not None:
                self._fill_view(tier, view, old, tier.n)
        mv.run()
        (kt, _, _, rk), (vt, _, _, rv) = sides
        kt.n, vt.n, kt.dirty, vt.dirty = kt.n + n, vt.n + n, 0, 0
        self._quant_keys[layer_idx], self._quant_values[layer_idx] = kt, vt
        self._dequant_keys_cache[layer_idx], self._dequant_values_cache[layer_idx] = kt, vt
        self._residual_keys[layer_idx], self._residual_values[layer_idx] = rk, rv
        return tuple(torch.cat([tier.dequantize(), kept], dim=2) if view is None else view
                     for tier, view, _, kept in sides)

    @staticmethod
    def _new_view(tier: _Tier, had: int, n: int, left: torch.Tensor, dt: torch.dtype, mv: RowMoves):
        """The view over ``had`` rows of the tier, n more that the caller writes and the residual
        ``left``, whose move is queued: (view, and for a float32 view the float16 buffer of those
        ``had`` rows, whose move is queued too)."""
        view = torch.empty(tier.B, tier.H, had + n + left.shape[2], tier.D, dtype=dt, device=left.device)
        old = None
        if had and dt != torch.float16:
            old = torch.empty(tier.rows, had, tier.D, dtype=torch.float16, device=left.device)
            mv.copy(view, old.view(tier.B, tier.H, had, tier.D), had)
        mv.copy(view, left if left.stride(3) == 1 else left.contiguous(), left.shape[2], at=had + n)
        return view, old

    @staticmethod
    def _fill_view(tier: _Tier, view: torch.Tensor, old: Optional[torch.Tensor], had: int):
        """Dequantize the first ``had`` rows of the tier into ``view`` (float32: into ``old``)."""
        if had:
            dequantize_rows(tier.codes, tier.sc, tier.ze, tier.bits, tier.gs, tier.D, n=had,
                            out=view.view(tier.rows, view.shape[2], tier.D) if old is None else old)

    def _get_full_kv(self, layer_idx: int):
        """akv/baselines.py:498-510."""
        rs = (self._residual_keys[layer_idx], self._residual_values[layer_idx])
        if layer_idx not in self._dequant_keys_cache:
            return rs
        mv, out = row_moves(), []
        for tier, r in zip((self._dequant_keys_cache[layer_idx], self._dequant_values_cache[layer_idx]), rs):
            dt = torch.promote_types(torch.float16, r.dtype)
            if not mv.takes(dt, r) or r.shape[:2] != (tier.B, tier.H) or r.shape[3] != tier.D:
                out.append(torch.cat([tier.dequantize(), r], dim=2))
                continue
            view, old = self._new_view(tier, tier.n, 0, r, dt, mv)
            self._fill_view(tier, view, old, tier.n)
            out.append(view)
        mv.run()
        return out[0], out[1]

    def fused_attention(self, query: torch.Tensor, layer_idx: int, sm_scale: Optional[float] = None) -> torch.Tensor:
        """softmax(q K^T * sm_scale) V over the layer's quantized tier (in place) and its
        residual window, query (B, Hq, M, D) with Hq a multiple of the cache's heads;
        float16 out.  One decode launch."""
        cfg = self.config
        if cfg.key_bits != cfg.value_bits:
            raise NotImplementedError("fused_attention reads one code width for K and V")
        nat.require_device(query)
        rk, rv = self._residual_keys[layer_idx], self._residual_values[layer_idx]
        if rk.dtype != torch.float16:
            raise TypeError("fused_attention takes a float16 cache")
        B, H, n_res, D = rk.shape
        q = nat.dev_contig(query.to(torch.float16))
        _, Hq, M, _ = q.shape
        rk, rv = nat.dev_contig(rk), nat.dev_contig(rv)
        kt, vt = self._quant_keys.get(layer_idx), self._quant_values.get(layer_idx)
        out = torch.empty_like(q)
        a = nat.DecodeArgs()
        a.abi_version = nat.ABI_VERSION
        a.B, a.Hq, a.Hkv, a.M, a.D = B, Hq, H, M, D
        a.q_dtype = nat.DT_F16
        a.q = q.data_ptr()
        if n_res:
            a.k_hot, a.v_hot = rk.data_ptr(), rv.data_ptr()
        a.n_hot = n_res
        a.hot_first = 0
        a.sm_scale = D ** -0.5 if sm_scale is None else float(sm_scale)
        if kt is not None and kt.n:
            w = a.warm
            w.kind = nat.WARM_LEGACY
            w.bits_k = w.bits_v = cfg.key_bits
            w.n_warm = kt.n
            w.token_stride = kt.cap
            w.k_codes, w.v_codes = kt.codes.data_ptr(), vt.codes.data_ptr()
            w.k_scale, w.k_zero = kt.sc16.data_ptr(), kt.ze16.data_ptr()
            w.v_scale, w.v_zero = vt.sc16.data_ptr(), vt.ze16.data_ptr()
            w.group_size = cfg.group_size
            w.meta_dtype = nat.DT_F16
            w.warm_heads = B * H
            w.legacy_sym = 0
        else:
            a.warm.kind = nat.WARM_NONE
        a.out = out.data_ptr()
        lib = nat.load()
        nbytes = lib.akv_decode_workspace_bytes(ctypes.byref(a))
        if nbytes < 0:
            nat.check(lib.akv_decode_attn(ctypes.byref(a), None), "KIVIFusedCache.fused_attention")
        # one workspace per device, shared by every layer, batch size and query length
        ws = self._ws.setdefault(q.device, nat.DecodeWorkspace()).get(
            nbytes, lib.akv_decode_counter_bytes(ctypes.byref(a)), q.device)
        a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
        nat.check(lib.akv_decode_attn(ctypes.byref(a), nat.stream_of(q)), "KIVIFusedCache.fused_attention")
        return out

    def reset(self):
        super().reset()
        self._dequant_keys_cache.clear()
        self._dequant_values_cache.clear()


def create_baseline(name: str, **kwargs):
    """akv/baselines.py:1023-1054 for the KIVI baselines ('kivi', 'kivi_fused' and its
    synonyms); the other baselines of the reference are not part of this build."""
    key = name.lower().replace("-", "").replace("_", "")
    if key == "kivi":
        return KIVICache(KIVIConfig(**kwargs))
    if key in ("kivifused", "fusedkivi", "kiviincremental"):
        return KIVIFusedCache(KIVIFusedConfig(**kwargs))
    if key in ("full", "h2o", "snapkv", "scissorhands", "scissors", "streamingllm", "streaming", "pyramidkv",
               "pyramid"):
        raise NotImplementedError(f"baseline {name!r} is not part of the MI355X build (KIVI baselines only)")
    raise ValueError(f"Unknown baseline: {key}. Choose from: full, h2o, kivi, kivi_fused, snapkv, "
                     f"scissorhands, streamingllm, pyramidkv")
