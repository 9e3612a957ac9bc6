"""The drop-in cache: AKVCache (presets, protected layers, per-layer update)
and AKVLayer (hot fp16 tier + packed warm tier, akv/drop_in.py:169-1200).

``_PRESETS`` and the preset resolution of ``AKVCache.__init__`` follow
akv/drop_in.py:89-124 and :910-964.  ``select_demote_indices`` is
akv/drop_in.py:392-413 (first 4 and last min(16, hot_budget // 4) hot tokens
protected, lowest scores first, indices returned in ascending order).
``AKVLayer.update`` keeps each demotion event packed (codes + scale / zero) and
serves the chronological view from one dequant launch; the reference keeps a
float16 working copy of the same values (_quantize_per_head at
akv/drop_in.py:315-374 quantizes and immediately dequantizes).
``AKVCache.demote`` quantizes a chosen token set into a warm tier of 32-token
K blocks, for callers that drive the tiers themselves.
"""
from __future__ import annotations

import ctypes
from typing import Optional

import torch

from . import _native as nat
from .row_moves import GATHER, KEEP, SCATTER, RowMoves, row_moves
from .warm_tier import WarmTier, packed_row_bytes, quantize_kv

# Protected layers join keys and values of fewer bytes with torch.cat, whose host time is the shorter (1,000 tokens of
# 8 heads x 128: 12.3 us a token against 23.2 as row moves); past them the launch counts (16,000: 49.6 against 22.9).
_CAT_BYTES = 16 << 20
_PRESETS = {
    "quality": {
        "warm_bits": 4,
        "hot_budget": 256,
        "description": "Near-lossless 4-bit. +1-2% PPL.",
    },
    "balanced": {
        "warm_bits": 3,
        "hot_budget": 128,
        "description": "Block-affine 3-bit. +3.3% PPL, 5x compression.",
    },
    "compact": {
        "warm_bits": 2,
        "hot_budget": 64,
        "description": "Block-affine 2-bit. +11% PPL, 8x compression.",
    },
    "k4v2": {
        "warm_bits": 4,
        "warm_key_bits": 4,
        "warm_value_bits": 2,
        "hot_budget": 128,
        "description": "Asymmetric K4/V2. Keys preserved, values aggressively compressed.",
    },
    "k4v3": {
        "warm_bits": 4,
        "warm_key_bits": 4,
        "warm_value_bits": 3,
        "hot_budget": 128,
        "description": "Asymmetric K4/V3. Near-quality keys with balanced value compression.",
    },
}


def select_demote_indices(importance: Optional[torch.Tensor], n_demote: int, hot_len: int,
                          hot_budget: int, device=None) -> torch.Tensor:
    """akv/drop_in.py:392-413 on the device (importance (hot_len,) or (B, hot_len)).

    With no scores, or scores of another length, the reference falls back to FIFO
    (``arange(n_demote)``, akv/drop_in.py:401-403); that index lands on ``device``
    (else on the scores' device), where the gather that consumes it runs."""
    if importance is None or importance.shape[-1] != hot_len:
        dev = device if device is not None else (importance.device if importance is not None else None)
        if dev is None:
            raise ValueError("select_demote_indices: no scores and no device for the FIFO fallback")
        return torch.arange(n_demote, device=dev)
    nat.require_device(importance)
    if not 0 <= n_demote <= hot_len:
        raise ValueError(f"n_demote {n_demote} outside [0, {hot_len}]")
    protect_initial = 4
    protect_recent = min(16, hot_budget // 4)
    scores = nat.dev_contig(importance, torch.float32)
    rows = scores.numel() // hot_len if hot_len else 0
    idx = torch.empty(importance.shape[:-1] + (n_demote,), dtype=torch.int64, device=importance.device)
    lib = nat.load()
    nat.check(lib.akv_select_demote(scores.data_ptr(), rows, hot_len, n_demote, protect_initial, protect_recent,
                                    idx.data_ptr(), nat.stream_of(scores)), "select_demote_indices")
    return idx


def quantize_per_head(k: torch.Tensor, v: torch.Tensor, key_bits: int = 3, value_bits: int = 3,
                      per_head_bits: Optional[list] = None, group_size: int = 64,
                      outlier_fraction: float = 0.0) -> tuple[torch.Tensor, torch.Tensor, int]:
    """AKVLayer._quantize_per_head (akv/drop_in.py:315-374) on the device.

    k, v (B, H, n, D): one AffineQuantizer call per batch element over the n tokens
    (K per channel, V per token, outliers shared by the heads) -- or, when
    ``per_head_bits`` names a width for each head, one call per (batch element, head)
    with a quantizer of that width for K and V (the reference's pool keyed by bits;
    a head-count mismatch falls back to the global widths).  Returns the dequantized
    K, V (fp16, bit-exact with the reference) and the measured packed bytes of the
    event (packed_layout.measure_packed_bytes).  The reference squeezes a batch of
    one; here each batch element is its own call."""
    from .affine_quantizer import AffineQuantConfig, AffineQuantizer
    from .packed_layout import measure_packed_bytes
    nat.require_device(k, v)
    B, H, n, D = k.shape
    out_k = torch.empty(B, H, n, D, dtype=torch.float16, device=k.device)
    out_v = torch.empty_like(out_k)
    packed = 0
    if not per_head_bits or len(per_head_bits) != H:
        qz = AffineQuantizer(AffineQuantConfig(key_bits=key_bits, value_bits=value_bits, group_size=group_size,
                                               outlier_fraction=outlier_fraction))
        for b in range(B):
            qk, qv = qz.quantize_keys(k[b]), qz.quantize_values(v[b])
            packed += measure_packed_bytes(qk, key_bits) + measure_packed_bytes(qv, value_bits)
            out_k[b] = qz.dequantize_keys(qk)
            out_v[b] = qz.dequantize_values(qv)
        return out_k, out_v, packed
    pool = {}
    for bits in set(per_head_bits):
        pool[bits] = AffineQuantizer(AffineQuantConfig(key_bits=bits, value_bits=bits, group_size=group_size,
                                                       outlier_fraction=outlier_fraction))
    for b in range(B):
        for h, bits in enumerate(per_head_bits):
            qz = pool[bits]
            qk, qv = qz.quantize_keys(k[b, h:h + 1]), qz.quantize_values(v[b, h:h + 1])
            packed += measure_packed_bytes(qk, bits) + measure_packed_bytes(qv, bits)
            out_k[b, h] = qz.dequantize_keys(qk)[0]
            out_v[b, h] = qz.dequantize_values(qv)[0]
    return out_k, out_v, packed


class _EventTier:
    """The packed warm tier of one AKVLayer: demotion events appended in order.

    Per (batch, head) the codes, V scale / zero and outlier values of every warm
    token (``cap`` token rows), and per event the K scale / zero rows (``ecap``)
    and per batch element its outlier channels; ``blk`` maps each warm token to
    its event and ``pos`` to its chronological position.  Capacities double as
    tokens arrive."""

    def __init__(self, B, H, D, bits_k, bits_v, n_out, dev, rows: int = 0):
        """``rows``: the first event's tokens, for which the first capacity makes room."""
        self.B, self.H, self.D, self.bits_k, self.bits_v, self.n_out = B, H, D, bits_k, bits_v, n_out
        self.dev = dev
        self.n = 0
        self.n_events = 0
        self.cap, self.ecap = 256 if rows <= 256 else 2 * rows, 16
        self.t = self._alloc(self.cap, self.ecap)

    def _alloc(self, cap, ecap):
        B, H, D, n_out, dev = self.B, self.H, self.D, self.n_out, self.dev
        f16, u8 = torch.float16, torch.uint8
        t = {
            "kc": torch.empty(B, H, cap, packed_row_bytes(D, self.bits_k), dtype=u8, device=dev),
            "vc": torch.empty(B, H, cap, packed_row_bytes(D, self.bits_v), dtype=u8, device=dev),
            "vs": torch.empty(B, H, cap, 1, dtype=f16, device=dev),
            "vz": torch.empty(B, H, cap, 1, dtype=f16, device=dev),
            "ks": torch.empty(B, H, ecap, D, dtype=f16, device=dev),
            "kz": torch.empty(B, H, ecap, D, dtype=f16, device=dev),
            "blk": torch.empty(cap, dtype=torch.int32, device=dev),
            "pos": torch.empty(cap, dtype=torch.int64, device=dev),
        }
        if n_out:
            t["kod"] = torch.empty(B, H, cap, n_out, dtype=f16, device=dev)
            t["vod"] = torch.empty(B, H, cap, n_out, dtype=f16, device=dev)
            t["koi"] = torch.empty(B, ecap, n_out, dtype=torch.int64, device=dev)
            t["voi"] = torch.empty(B, ecap, n_out, dtype=torch.int64, device=dev)
        return t

    _TOKEN_AXIS = {"kc": 2, "vc": 2, "vs": 2, "vz": 2, "kod": 2, "vod": 2, "blk": 0, "pos": 0}

    @staticmethod
    def _rows4(name, x):
        """A tier tensor as (B, H, rows, C): the outlier indices have no head axis."""
        return x.unsqueeze(1) if name in ("koi", "voi") else x

    def _grow(self, cap, ecap):
        t = self._alloc(cap, ecap)
        mv = row_moves()
        for name, old in self.t.items():
            mv.copy(self._rows4(name, t[name]), self._rows4(name, old),
                    self.n if name in self._TOKEN_AXIS else self.n_events)
        mv.run()
        self.t, self.cap, self.ecap = t, cap, ecap

    def append(self, w: WarmTier, positions: torch.Tensor, mv: RowMoves):
        """One demotion event: ``w`` holds its n tokens as a single K block; their positions
        are those of ``positions`` at the list ``mv`` is run with.  Returns what takes the event
        into the tier, to be called once ``mv`` has run."""
        n = w.n_warm
        if self.n + n > self.cap or self.n_events + 1 > self.ecap:
            self._grow(max(self.cap, 2 * (self.n + n)), max(self.ecap, 2 * (self.n_events + 1)))
        t, a, e = self.t, self.n, self.n_events
        for name, x in (("kc", w.k_codes), ("vc", w.v_codes), ("vs", w.v_scale), ("vz", w.v_zero)):
            mv.copy(t[name], x, n, at=a)
        mv.copy(t["ks"], w.k_scale, 1, at=e)
        mv.copy(t["kz"], w.k_zero, 1, at=e)
        if self.n_out:
            mv.copy(t["kod"], w.k_odata, n, at=a)
            mv.copy(t["vod"], w.v_odata, n, at=a)
            mv.copy(t["koi"].unsqueeze(1), w.k_oidx.unsqueeze(1), 1, at=e)
            mv.copy(t["voi"].unsqueeze(1), w.v_oidx.unsqueeze(1), 1, at=e)
        mv.count(t["blk"], n, e, 0, at=a)
        mv.copy(t["pos"], positions, n, GATHER, at=a)

        def commit():
            self.n, self.n_events = a + n, e + 1
        return commit

    def positions(self) -> torch.Tensor:
        return self.t["pos"][: self.n]

    def resident_bytes(self) -> int:
        """Bytes of the used extents (codes, meta, outliers, event map, positions)."""
        total = 0
        for name, x in self.t.items():
            if name in self._TOKEN_AXIS:
                total += x.narrow(self._TOKEN_AXIS[name], 0, self.n).nbytes
            else:
                total += x.narrow(2 if name in ("ks", "kz") else 1, 0, self.n_events).nbytes
        return total

    def dequantize_into(self, out_k: torch.Tensor, out_v: Optional[torch.Tensor], slots: bool = True):
        """Dequantize every warm token into out_k / out_v (B, H, rows, D): at its
        chronological position when ``slots``, else at its warm-tier index (keys only
        when ``out_v`` is None)."""
        if self.n == 0:
            return
        t = self.t
        d = nat.WarmDesc()
        d.kind = nat.WARM_AFFINE
        d.bits_k, d.bits_v = self.bits_k, self.bits_v
        d.n_warm = self.n
        d.token_stride = self.cap
        d.block_t = 1
        d.group_v = self.D
        d.n_out = self.n_out
        d.k_codes, d.v_codes = t["kc"].data_ptr(), t["vc"].data_ptr()
        d.k_scale, d.k_zero = t["ks"].data_ptr(), t["kz"].data_ptr()
        d.v_scale, d.v_zero = t["vs"].data_ptr(), t["vz"].data_ptr()
        if self.n_out:
            d.k_oidx, d.v_oidx = t["koi"].data_ptr(), t["voi"].data_ptr()
            d.k_odata, d.v_odata = t["kod"].data_ptr(), t["vod"].data_ptr()
        a = nat.DequantArgs()
        a.abi_version = nat.ABI_VERSION
        a.B, a.Hkv, a.D = self.B, self.H, self.D
        a.out_dtype = nat.dtype_code(out_k.dtype)
        a.warm = d
        a.k_out = out_k.data_ptr()
        a.v_out = out_v.data_ptr() if out_v is not None else None
        a.block_of_token = t["blk"].data_ptr()
        a.n_blocks = self.ecap
        if slots:
            a.out_slot = t["pos"].data_ptr()
        a.out_tokens = out_k.shape[2]
        nat.check(nat.load().akv_dequant_unpack(ctypes.byref(a), nat.stream_of(out_k)), "AKVLayer warm view")

    def pull(self, idx: torch.Tensor, vector: Optional[torch.Tensor] = None):
        """The float16 K, V (B, H, n, D) of the warm tokens of the ascending list ``idx``, then
        ``vector`` without them and what takes them out of the tier, as ``remove`` gives both."""
        n = idx.numel()
        sub = _EventTier.__new__(_EventTier)
        sub.__dict__.update({k: v for k, v in self.__dict__.items() if k != "t"})
        sub.t = {}
        mv = row_moves()
        for name, x in self.t.items():
            if name in self._TOKEN_AXIS:
                shape = list(x.shape)
                shape[self._TOKEN_AXIS[name]] = n
                sub.t[name] = torch.empty(shape, dtype=x.dtype, device=x.device)
                mv.copy(sub.t[name], x, n, GATHER)
            else:
                sub.t[name] = x
        k = torch.empty(self.B, self.H, n, self.D, dtype=torch.float16, device=self.dev)
        v = torch.empty_like(k)
        kept, commit = self.remove(idx, n, vector, mv)
        sub.n, sub.cap = n, n
        sub.dequantize_into(k, v, slots=False)
        return k, v, kept, commit

    def remove(self, idx: torch.Tensor, n: int, vector: Optional[torch.Tensor] = None,
               mv: Optional[RowMoves] = None):
        """The tier without the ``n`` warm tokens of the ascending list ``idx`` (their events' K
        meta rows stay): ``vector`` (one float32 per warm token) without theirs, and what takes
        them out of the tier.  The kept rows go to fresh tensors: rows shift by up to n, so a
        move in place would race.  ``mv``: jobs on the same list that go with the launch."""
        kept = self.n - n
        mv = mv or row_moves()
        fresh = {name: torch.empty_like(self.t[name]) for name in self._TOKEN_AXIS if name in self.t}
        for name, x in fresh.items():
            mv.copy(x, self.t[name], kept, KEEP)
        out = None
        if vector is not None:
            out = torch.empty(kept, dtype=vector.dtype, device=vector.device)
            mv.copy(out, vector, kept, KEEP)
        mv.run(idx, n)

        def commit():
            self.t.update(fresh)
            self.n = kept
        return out, commit

    def index_batch(self, beam_idx: torch.Tensor):
        for name in list(self.t):
            if name not in ("blk", "pos"):
                self.t[name] = self.t[name].index_select(0, beam_idx.to(self.dev))
        self.B = self.t["kc"].shape[0]


class _HeadBitsTier:
    """The packed warm tier when each head has its own code width (a calibration's
    ``per_head_bits``, akv/drop_in.py:315-374): one ``_EventTier`` per width over that
    width's heads, each (batch element, head) its own row -- the reference quantizes
    every head with its own AffineQuantizer of that width (the pool keyed by bits), so
    keys are per channel over the event's tokens of that head and the outlier channels
    are chosen per head.  Same interface as ``_EventTier``."""

    def __init__(self, B, H, D, per_head_bits, dev):
        self.B, self.H, self.D, self.dev = B, H, D, dev
        self.n = 0
        self.groups = []  # [bits, head indices on the device, _EventTier or None]
        for bits in sorted(set(per_head_bits)):
            heads = [h for h, b in enumerate(per_head_bits) if b == bits]
            self.groups.append([bits, torch.tensor(heads, dtype=torch.long, device=dev), None])

    def demote(self, hk, hv, idx, outlier_fraction, positions):
        """Quantize hot tokens ``idx`` (at ``positions[idx]``) of every head with its width as one event; returns
        the measured packed bytes (codes + scale + zero of K and V, per head) and what takes the event
        into the tier."""
        B, _, _, D = hk.shape
        n = idx.numel()
        packed, staged = 0, []
        for bits, heads, tier in self.groups:
            hs = heads.numel()
            k = hk.index_select(1, heads).index_select(2, idx).reshape(B * hs, 1, n, D)
            v = hv.index_select(1, heads).index_select(2, idx).reshape(B * hs, 1, n, D)
            w = quantize_kv(k, v, bits, bits, block_t=max(n, 1), group_v=D, outlier_fraction=outlier_fraction)
            if tier is None:
                tier = _EventTier(B * hs, 1, D, bits, bits, w.n_out, self.dev, n)
            mv = row_moves()
            staged.append((tier, tier.append(w, positions, mv)))
            mv.run(idx, n)
            packed += (w.k_codes.nbytes + w.k_scale.nbytes + w.k_zero.nbytes
                       + w.v_codes.nbytes + w.v_scale.nbytes + w.v_zero.nbytes)

        def commit():
            for g, (tier, take) in zip(self.groups, staged):
                g[2] = tier
                take()
            self.n += n
        return packed, commit

    def resident_bytes(self) -> int:
        return sum(g[2].resident_bytes() for g in self.groups if g[2] is not None)

    def dequantize_into(self, out_k: torch.Tensor, out_v: Optional[torch.Tensor], slots: bool = True):
        rows = out_k.shape[2]
        for bits, heads, tier in self.groups:
            hs = heads.numel()
            tk = torch.empty(self.B * hs, 1, rows, self.D, dtype=out_k.dtype, device=out_k.device)
            tv = torch.empty_like(tk) if out_v is not None else None
            tier.dequantize_into(tk, tv, slots)
            out_k.index_copy_(1, heads, tk.view(self.B, hs, rows, self.D))
            if out_v is not None:
                out_v.index_copy_(1, heads, tv.view(self.B, hs, rows, self.D))

    def _taken(self, n: int, commits: list):
        def commit():
            for take in commits:
                take()
            self.n -= n
        return commit

    def pull(self, idx: torch.Tensor, vector: Optional[torch.Tensor] = None):
        n = idx.numel()
        k = torch.empty(self.B, self.H, n, self.D, dtype=torch.float16, device=self.dev)
        v = torch.empty_like(k)
        kept, commits = None, []
        for i, (bits, heads, tier) in enumerate(self.groups):
            tk, tv, out, commit = tier.pull(idx, vector if i == 0 else None)
            kept = out if i == 0 else kept
            commits.append(commit)
            k.index_copy_(1, heads, tk.view(self.B, heads.numel(), n, self.D))
            v.index_copy_(1, heads, tv.view(self.B, heads.numel(), n, self.D))
        return k, v, kept, self._taken(n, commits)

    def remove(self, idx: torch.Tensor, n: int, vector: Optional[torch.Tensor] = None):
        out, commits = None, []
        for i, g in enumerate(self.groups):
            kept, commit = g[2].remove(idx, n, vector if i == 0 else None)
            out = kept if i == 0 else out
            commits.append(commit)
        return out, self._taken(n, commits)

    def positions(self) -> torch.Tensor:
        return self.groups[0][2].positions()

    def index_batch(self, beam_idx: torch.Tensor):
        beam_idx = beam_idx.to(self.dev)
        for g in self.groups:
            hs = g[1].numel()
            rows = (beam_idx.unsqueeze(1) * hs + torch.arange(hs, device=self.dev)).flatten()
            g[2].index_batch(rows)
        self.B = beam_idx.numel()


class AKVLayer:
    """One layer of the drop-in cache (akv/drop_in.py:169-873) with the warm tier
    kept packed on the device.

    ``update`` follows akv/drop_in.py:591-787: new tokens join the hot tier with
    their positions; the importance vector decays by 0.3 and appends ones
    (:375-389); past the (adaptive) budget the lowest-importance unprotected
    tokens are chosen on the device (``select_demote_indices``), gathered and
    quantized as one demotion event (one ``akv_quant_pack`` launch: keys per
    channel over the event's tokens, values per token over all channels,
    outliers per event and batch element, the reference's AffineQuantizer), and
    the event's codes and scale / zero rows are appended to the packed tier --
    no float16 working copy is kept.  The returned view is chronological: one
    ``akv_dequant_unpack`` launch writes every warm token at its position and the
    hot tokens are scattered in beside it (float16, or float32 when the hot
    tokens are float32 / bfloat16, as the reference's torch.cat promotes).  The
    measured packed bytes count codes + scale + zero per event
    (packed_layout.measure_packed_bytes).

    Promotion (:415-589): with the proxy on, the EMA of |cos| between the mean
    new key and each warm token's key (dequantized, averaged over batch and
    heads) is kept per warm token; warm tokens above ``promotion_threshold`` --
    by the attention weights' warm columns when ``cache_kwargs`` carries them,
    else by the proxy -- return to the front of the hot tier with their float16
    values and importance 2.0, at most max(1, hot_budget // 8) per step, and
    leave the packed tier.

    Each batch element is its own quantizer call over (H, n, D) -- the
    reference's call on ``k.squeeze(0)`` at batch 1.  With ``per_head_bits`` naming
    a width for every head (a calibration's), each (batch element, head) is its own
    call at its width (``_HeadBitsTier``); of another head count, the global widths
    apply, as in the reference."""

    def __init__(self, warm_bits: int = 3, hot_budget: int = 128, group_size: int = 64, protect: bool = False,
                 enable_promotion: bool = True, promotion_threshold: float = 0.05,
                 per_head_bits: Optional[list] = None,
                 enable_promotion_proxy: bool = True, proxy_decay: float = 0.7, adaptive_hot_frac: float = 0.0,
                 warm_key_bits: Optional[int] = None, warm_value_bits: Optional[int] = None,
                 outlier_fraction: float = 0.0):
        self.warm_bits = warm_bits
        self.hot_budget = hot_budget
        self.group_size = group_size
        self.protect = protect
        self.enable_promotion = enable_promotion
        self.promotion_threshold = promotion_threshold
        self.enable_promotion_proxy = enable_promotion_proxy
        self.proxy_decay = proxy_decay
        self.adaptive_hot_frac = adaptive_hot_frac
        self.warm_key_bits = warm_key_bits or warm_bits
        self.warm_value_bits = warm_value_bits or warm_bits
        self.outlier_fraction = outlier_fraction
        self.per_head_bits = list(per_head_bits) if per_head_bits is not None else None
        self._hot_keys: Optional[torch.Tensor] = None
        self._hot_values: Optional[torch.Tensor] = None
        self._positions: Optional[torch.Tensor] = None       # see _hot_positions
        self._warm: Optional[_EventTier] = None
        self._warm_len = 0
        self._total_len = 0
        self._warm_bytes_packed = 0
        self._importance: Optional[torch.Tensor] = None      # (N_hot,) float32, device
        self._proxy_score: Optional[torch.Tensor] = None     # (N_warm,) float32, device
        self._decay = 0.3
        self._step = 0
        self.keys = self.values = None

    def get_seq_length(self) -> int:
        return self._total_len

    @property
    def _hot_positions(self) -> Optional[torch.Tensor]:
        """(N_hot,) int64, device: the hot tokens' positions.  While every token is hot and in order
        (before the first demotion or crop, always in protected layers) none are kept."""
        if self._positions is None and self._hot_keys is not None:
            return torch.arange(self._hot_keys.shape[2], device=self._hot_keys.device)
        return self._positions

    @_hot_positions.setter
    def _hot_positions(self, positions: Optional[torch.Tensor]):
        self._positions = positions

    def __setstate__(self, state: dict):
        """Layers saved while the positions were an attribute load too."""
        self.__dict__.update(state)
        if "_hot_positions" in state:
            self._positions = self.__dict__.pop("_hot_positions")

    @property
    def _warm_positions(self) -> Optional[torch.Tensor]:
        """(N_warm,) int64, device: the warm tokens' positions in demotion order."""
        return None if self._warm is None else self._warm.positions()

    @staticmethod
    def _join(mv: RowMoves, parts: list) -> torch.Tensor:
        """torch.cat(parts, dim=2) as jobs of ``mv`` (one part: itself), torch's own where the
        parts do not fit each other or row moves do not do them."""
        if len(parts) == 1:
            return parts[0]
        first, dt = parts[0], parts[0].dtype
        for x in parts[1:]:
            dt = torch.promote_types(dt, x.dtype)
        if not mv.takes(dt, *parts) or any(x.dim() != 4 or x.device != first.device or x.shape[:2] != first.shape[:2]
                                          or x.shape[3] != first.shape[3] for x in parts):
            return torch.cat(parts, dim=2)
        out = torch.empty(first.shape[0], first.shape[1], sum(x.shape[2] for x in parts), first.shape[3], dtype=dt,
                          device=first.device)
        at = 0
        for x in parts:
            n = x.shape[2]
            mv.copy(out, x if x.stride(3) == 1 or x.shape[3] <= 1 else x.contiguous(), n, at=at)
            at += n
        return out

    def _append_hot(self, k, v, promoted=None):
        """The hot tier with the promoted tokens in front and the new ones (k, v) behind, their
        positions, and the importance: 2 for the promoted, decayed for the old, 1 for the new
        (akv/drop_in.py:375-389, :433-484); one launch.  ``promoted``: (K, V, the warm tier's
        positions, their indices among them, what takes them out of the warm tier).  The tiers
        change after the launch: a call that fails before leaves them as they were."""
        dev = k.device
        old = 0 if self._hot_keys is None else self._hot_keys.shape[2]
        new = k.shape[2]
        front = 0 if promoted is None else promoted[0].shape[2]
        in_order = self._positions is None and front == 0 and old == self._total_len
        mv, imp = row_moves(), None
        if self._hot_keys is None and front == 0:
            keys, values = k, v
            imp = None if self.protect else torch.ones(new, dtype=torch.float32, device=dev)
        elif self.protect and in_order and self._hot_keys.nbytes + self._hot_values.nbytes < _CAT_BYTES:
            keys = torch.cat([self._hot_keys, k], dim=2)
            values = torch.cat([self._hot_values, v], dim=2)
        else:
            parts_k = ([] if promoted is None else [promoted[0]]) + ([] if self._hot_keys is None else [self._hot_keys]) + [k]
            parts_v = ([] if promoted is None else [promoted[1]]) + ([] if self._hot_keys is None else [self._hot_values]) + [v]
            keys, values = self._join(mv, parts_k), self._join(mv, parts_v)
            if not self.protect:
                imp = torch.empty(front + old + new, dtype=torch.float32, device=dev)
                mv.fill(imp, front, 2.0)
                if self._importance is not None and self._importance.shape[0] == old:
                    mv.copy(imp, self._importance, old, at=front, value=self._decay)
                else:
                    mv.fill(imp, old, 1.0, at=front)
                mv.fill(imp, new, 1.0, at=front + old)
        pos = None
        if not in_order:
            pos = torch.empty(front + old + new, dtype=torch.int64, device=dev)
            if front:
                mv.copy(pos, promoted[2], front, GATHER)
            if old:
                mv.copy(pos, self._hot_positions.to(dev), old, at=front)
            mv.count(pos, new, self._total_len, at=front + old)
        mv.run(None if promoted is None else promoted[3], front)
        if promoted is not None:
            promoted[4]()
        self._hot_keys, self._hot_values, self._positions, self._importance = keys, values, pos, imp
        self._total_len += new

    def _proxy_similarity(self, key_states: torch.Tensor) -> Optional[torch.Tensor]:
        """akv/drop_in.py:486-525 over the packed tier: the cosine of every warm token's key
        with the mean new key; only the keys are dequantized (one launch, warm-tier order, no
        copy of the packed arrays), to float32."""
        if self._warm is None or self._warm.n == 0:
            self._proxy_score = None
            return None
        probe = key_states.detach().float().mean(dim=(0, 1, 2))
        probe = probe / (probe.norm() + 1e-6)
        w = self._warm
        wk = torch.empty(w.B, w.H, w.n, w.D, dtype=torch.float32, device=w.dev)
        w.dequantize_into(wk, None, slots=False)
        wk_flat = wk.mean(dim=(0, 1))
        wk_norm = wk_flat / (wk_flat.norm(dim=-1, keepdim=True) + 1e-6)
        return wk_norm @ probe

    def _choose(self, scores: torch.Tensor, proxy: bool) -> torch.Tensor:
        """The promotion choice of ``akv_promote_select``: (1 + cap,) int64, how many, then the
        warm indices.  ``proxy``: ``scores`` are similarities that first go into the running
        proxy scores (their EMA where the tokens are the same)."""
        n = scores.shape[0]
        cap = min(n, max(1, self.hot_budget // 8))
        scores = nat.dev_contig(scores, torch.float32)
        out = torch.empty(1 + cap, dtype=torch.int64, device=scores.device)
        prev = new = None
        if proxy:
            if self._proxy_score is not None and self._proxy_score.shape[0] == n:
                prev = nat.dev_contig(self._proxy_score)
            new = torch.empty(n, dtype=torch.float32, device=scores.device)
        d = self.proxy_decay
        nat.check(nat.load().akv_promote_select(scores.data_ptr(), nat.ptr(prev), nat.ptr(new), n, d, 1 - d,
                                                self.promotion_threshold, cap, out.data_ptr(), nat.stream_of(scores)),
                  "promotion choice")
        if proxy:
            self._proxy_score = new
        return out

    def _take_promoted(self, chosen: torch.Tensor, use_proxy: bool):
        """akv/drop_in.py:433-484 / :543-589: what ``_append_hot`` puts in front of the hot tier, or
        None; its last entry takes the chosen warm tokens out of the packed tier.  The count is
        the one value an update waits for: the shapes that follow depend on it."""
        n = int(chosen[0])
        if n == 0:
            return None
        idx = chosen[1:1 + n]
        warm_len = self._warm.n
        positions = self._warm.positions()
        pk, pv, kept, take = self._warm.pull(idx, self._proxy_score if use_proxy else None)

        def commit():
            take()
            if use_proxy:
                self._proxy_score = kept
            self._warm_bytes_packed = int(self._warm_bytes_packed * (max(0, warm_len - n) / warm_len))
            self._warm_len -= n
        return pk, pv, positions, idx, commit

    def _demote(self, n_demote: int, hot_len: int):
        """The tiers change once everything is allocated and launched: a call that fails before
        leaves the tokens in the hot tier, over its budget until the next one."""
        hk, hv = self._hot_keys, self._hot_values
        dev = hk.device
        B, H, _, D = hk.shape
        idx = select_demote_indices(self._importance, n_demote, hot_len, self.hot_budget, device=dev)
        mv = row_moves()  # the event's rows into the packed tier, the kept ones of the hot tier
        warm, positions = self._warm, self._hot_positions
        if self.per_head_bits and len(self.per_head_bits) == H:
            if warm is None:
                warm = _HeadBitsTier(B, H, D, self.per_head_bits, dev)
            packed, take = warm.demote(hk, hv, idx, self.outlier_fraction, positions)
        else:
            w = quantize_kv(hk, hv, self.warm_key_bits, self.warm_value_bits, block_t=max(n_demote, 1), group_v=D,
                            outlier_fraction=self.outlier_fraction, sel=idx.unsqueeze(0).expand(B, n_demote))
            if warm is None:
                warm = _EventTier(B, H, D, self.warm_key_bits, self.warm_value_bits, w.n_out, dev, n_demote)
            take = warm.append(w, positions, mv)
            # measure_packed_bytes per batch element: packed codes + fp16 scale and zero, K and V
            packed = (w.k_codes.nbytes + w.k_scale.nbytes + w.k_zero.nbytes
                      + w.v_codes.nbytes + w.v_scale.nbytes + w.v_zero.nbytes)
        proxy = self._proxy_score
        if proxy is not None:  # new warm tokens start with no evidence
            old = proxy.shape[0]
            proxy = torch.empty(old + n_demote, dtype=torch.float32, device=dev)
            mv.copy(proxy, self._proxy_score, old)
            mv.fill(proxy, n_demote, 0.0, at=old)
        kept = hot_len - n_demote
        pos = torch.empty(kept, dtype=torch.int64, device=dev)
        imp = torch.empty(kept, dtype=torch.float32, device=dev)
        mv.copy(pos, positions, kept, KEEP)
        mv.copy(imp, self._importance, kept, KEEP)
        if mv.takes(hk.dtype, hk) and mv.takes(hv.dtype, hv):
            tiers = []
            for x in (hk, hv):
                x = x if x.stride(3) == 1 or D <= 1 else x.contiguous()
                tiers.append(torch.empty(B, H, kept, D, dtype=x.dtype, device=dev))
                mv.copy(tiers[-1], x, kept, KEEP)
        else:
            keep = torch.ones(hot_len, dtype=torch.bool, device=dev)
            keep[idx] = False
            tiers = [hk[:, :, keep], hv[:, :, keep]]
        mv.run(idx, n_demote)
        take()
        self._warm, self._proxy_score = warm, proxy
        self._warm_len += n_demote
        self._warm_bytes_packed += packed
        self._hot_keys, self._hot_values = tiers
        self._positions, self._importance = pos, imp

    def update(self, key_states: torch.Tensor, value_states: torch.Tensor,
               cache_kwargs: Optional[dict] = None) -> tuple[torch.Tensor, torch.Tensor]:
        """Append new KV, demote past the budget, return the chronological view."""
        nat.require_device(key_states, value_states)
        B, H, N, D = key_states.shape
        if self.protect:
            self._append_hot(key_states, value_states)
            self.keys, self.values = self._hot_keys, self._hot_values
            return self._hot_keys, self._hot_values
        for hot, x in ((self._hot_keys, key_states), (self._hot_values, value_states)):
            if hot is not None and (x.shape[:2] != hot.shape[:2] or x.shape[3] != hot.shape[3]):
                torch.cat([hot, x], dim=2)  # raises, before any tier changes
        self._step += 1
        chosen, use_proxy = None, False
        if self.enable_promotion_proxy:
            sim = self._proxy_similarity(key_states)
            if sim is not None:
                chosen, use_proxy = self._choose(sim, proxy=True), True
        if not self.enable_promotion:
            chosen = None
        elif cache_kwargs and "attention_weights" in cache_kwargs:
            chosen, use_proxy = None, False
            aw = cache_kwargs["attention_weights"]
            hot_len = N + (0 if self._hot_keys is None else self._hot_keys.shape[2])
            if self._warm is not None and self._warm.n and aw.dim() == 4 and aw.shape[-1] >= self._warm.n + hot_len:
                chosen = self._choose(aw[:, :, :, : self._warm.n].float().mean(dim=(0, 1, 2)), proxy=False)
        self._append_hot(key_states, value_states,
                         None if chosen is None else self._take_promoted(chosen, use_proxy))
        hot_len = self._hot_keys.shape[2]
        budget = self.hot_budget
        if self.adaptive_hot_frac > 0.0:
            budget = max(self.hot_budget, int(self.adaptive_hot_frac * self._total_len))
        if hot_len > budget:
            self._demote(hot_len - budget, hot_len)
        if self._warm is None:
            self.keys, self.values = self._hot_keys, self._hot_values
            return self._hot_keys, self._hot_values
        hk, hv = self._hot_keys, self._hot_values
        out_dt = torch.float16 if hk.dtype == torch.float16 else torch.float32
        fk = torch.empty(B, H, self._total_len, D, dtype=out_dt, device=hk.device)
        fv = torch.empty_like(fk)
        self._warm.dequantize_into(fk, fv)
        hp = self._hot_positions
        mv = row_moves()
        if mv.takes(out_dt, hk, hv):
            mv.copy(fk, hk, hk.shape[2], SCATTER)
            mv.copy(fv, hv, hv.shape[2], SCATTER)
            mv.run(hp, hp.shape[0])
        else:
            fk.index_copy_(2, hp, hk.to(out_dt))
            fv.index_copy_(2, hp, hv.to(out_dt))
        self.keys, self.values = fk, fv
        return fk, fv

    def crop(self, max_length: int):
        """Keep positions 0 .. max_length-1 (the cache's ``crop``): hot tokens at or past
        it leave the hot tier with their importance, warm ones leave the packed tier with
        their proxy scores, and the length becomes max_length."""
        if self._total_len <= max_length:
            return
        take = hot = None
        if self._warm is not None and self._warm.n:
            warm_len = self._warm.n
            drop = (self._warm.positions() >= max_length).nonzero().flatten()
            n_drop = drop.numel()
            if n_drop:
                proxy = self._proxy_score
                fits = proxy is not None and proxy.shape[0] == warm_len
                kept, take = self._warm.remove(drop, n_drop, proxy if fits else None)
        if self._hot_keys is not None:
            positions = self._hot_positions
            keep = positions < max_length
            if not bool(keep.all()):
                imp = self._importance
                if imp is not None and imp.shape[0] == keep.shape[0]:
                    imp = imp[keep]
                hot = self._hot_keys[:, :, keep], self._hot_values[:, :, keep], positions[keep], imp
        if take is not None:
            take()
            if fits:
                self._proxy_score = kept
            self._warm_bytes_packed = int(self._warm_bytes_packed * ((warm_len - n_drop) / warm_len))
            self._warm_len -= n_drop
        if hot is not None:
            self._hot_keys, self._hot_values, self._positions, self._importance = hot
        self._total_len = max_length

    def warm_view(self) -> tuple[Optional[torch.Tensor], Optional[torch.Tensor]]:
        """The dequantized warm tier in demotion order (the reference's working copy)."""
        if self._warm is None:
            return None, None
        w = self._warm
        k = torch.empty(w.B, w.H, w.n, w.D, dtype=torch.float16, device=w.dev)
        v = torch.empty_like(k)
        w.dequantize_into(k, v, slots=False)
        return k, v

    def memory_usage_bytes(self) -> dict:
        """akv/drop_in.py:789-873; ``warm_bytes_live`` is what the packed tier holds
        resident (codes, meta, outlier values, event and position maps)."""
        H, D = 1, 128
        hot_bytes = 0
        if self._hot_keys is not None:
            hot_bytes = self._hot_keys.nbytes + self._hot_values.nbytes
            H, D = self._hot_keys.shape[1], self._hot_keys.shape[3]
        warm_live = self._warm.resident_bytes() if self._warm is not None else 0
        packed = int(self._warm_bytes_packed)
        formula = 0
        if self._warm_len > 0:
            groups = (D + self.group_size - 1) // self.group_size
            formula = self._warm_len * ((H * D * self.warm_bits + 7) // 8 + groups * H * 4) * 2
        total = hot_bytes + packed
        fp16_equiv = self._total_len * H * D * 2 * 2
        return {"hot_bytes": hot_bytes, "warm_bytes": packed, "warm_bytes_live": warm_live,
                "warm_bytes_packed": packed, "warm_bytes_formula": formula, "total_bytes": total,
                "fp16_equivalent_bytes": fp16_equiv, "savings_ratio": fp16_equiv / max(total, 1)}


class AKVCache:
    """The drop-in cache (akv/drop_in.py:885-1200): preset resolution, protected
    layers, lazily created ``AKVLayer``s driven by ``update`` (the method an HF
    model calls per layer), and ``demote`` (the warm-tier hot path with 32-token
    K blocks, for callers that manage the tiers themselves), with the reference's other
    cache methods (length queries, iteration, the legacy tuple form, crop, the beam
    helpers, reset, for_model, from_calibration).  Subclassing HF's ``DynamicCache`` is
    not part of this build."""

    def __init__(self, preset: Optional[str] = None, warm_bits: Optional[int] = None,
                 warm_key_bits: Optional[int] = None, warm_value_bits: Optional[int] = None,
                 hot_budget: Optional[int] = None, group_size: int = 64, outlier_fraction: float = 0.0,
                 protect_first: int = 0, protect_last: int = 0, protect_layers: Optional[list] = None,
                 num_hidden_layers: Optional[int] = None, enable_promotion: bool = True,
                 promotion_threshold: float = 0.05, enable_promotion_proxy: bool = True,
                 proxy_decay: float = 0.7, adaptive_hot_frac: float = 0.0,
                 block_t: int = 32, group_v: int = 32):
        if preset is not None:
            if preset not in _PRESETS:
                raise ValueError(f"Unknown preset {preset!r}. Choose from: {sorted(_PRESETS.keys())}")
            if warm_bits is not None or hot_budget is not None:
                raise ValueError(
                    "preset= is mutually exclusive with warm_bits/hot_budget. "
                    "Pick a preset OR pass explicit params.")
            p = _PRESETS[preset]
            self.warm_bits = p["warm_bits"]
            self.hot_budget = p["hot_budget"]
        else:
            self.warm_bits = warm_bits or 3
            self.hot_budget = hot_budget or 128
        if preset and "warm_key_bits" in _PRESETS.get(preset, {}):
            self.warm_key_bits = _PRESETS[preset]["warm_key_bits"]
            self.warm_value_bits = _PRESETS[preset]["warm_value_bits"]
        else:
            self.warm_key_bits = warm_key_bits or self.warm_bits
            self.warm_value_bits = warm_value_bits or self.warm_bits
        self.preset = preset
        self.group_size = group_size
        self.outlier_fraction = outlier_fraction
        self.num_hidden_layers = num_hidden_layers
        self.enable_promotion = enable_promotion
        self.promotion_threshold = promotion_threshold
        self.enable_promotion_proxy = enable_promotion_proxy
        self.proxy_decay = proxy_decay
        self.adaptive_hot_frac = adaptive_hot_frac
        self._protect_first = protect_first
        self._protect_last = protect_last
        self._protect_explicit = list(protect_layers) if protect_layers else []
        self.block_t = block_t
        self.group_v = group_v
        # protected layers (akv/drop_in.py:971-998)
        if protect_last > 0 and num_hidden_layers is None:
            raise ValueError("protect_last requires num_hidden_layers. "
                             "Use AKVCache.for_model(model, ...) or pass num_hidden_layers=.")
        self._protected_set: set = set(range(protect_first))
        if num_hidden_layers is not None:
            for i in range(protect_last):
                self._protected_set.add(num_hidden_layers - 1 - i)
            for p in self._protect_explicit:
                self._protected_set.add(p if p >= 0 else num_hidden_layers + p)
        else:
            for p in self._protect_explicit:
                if p < 0:
                    raise ValueError("Negative protect_layers indices require num_hidden_layers. "
                                     "Use AKVCache.for_model(model, ...).")
                self._protected_set.add(p)
        self.layers: list = []
        self._seen_tokens = 0
        self._calibration_per_head_bits: dict = {}

    def _is_protected(self, layer_idx: int) -> bool:
        return layer_idx in self._protected_set

    def update(self, key_states: torch.Tensor, value_states: torch.Tensor, layer_idx: int,
               cache_kwargs: Optional[dict] = None) -> tuple[torch.Tensor, torch.Tensor]:
        """akv/drop_in.py:1066-1096: create layers lazily, count tokens on layer 0, delegate."""
        while len(self.layers) <= layer_idx:
            idx = len(self.layers)
            self.layers.append(AKVLayer(
                warm_bits=self.warm_bits, hot_budget=self.hot_budget, group_size=self.group_size,
                protect=self._is_protected(idx), enable_promotion=self.enable_promotion,
                promotion_threshold=self.promotion_threshold, enable_promotion_proxy=self.enable_promotion_proxy,
                proxy_decay=self.proxy_decay, adaptive_hot_frac=self.adaptive_hot_frac,
                warm_key_bits=self.warm_key_bits, warm_value_bits=self.warm_value_bits,
                outlier_fraction=self.outlier_fraction,
                per_head_bits=self._calibration_per_head_bits.get(idx) if self._calibration_per_head_bits else None))
        if layer_idx == 0:
            self._seen_tokens += key_states.shape[2]
        return self.layers[layer_idx].update(key_states, value_states, cache_kwargs)

    def get_seq_length(self, layer_idx: int = 0) -> int:
        return self.layers[layer_idx].get_seq_length() if layer_idx < len(self.layers) else 0

    def get_usable_length(self, max_length: int, layer_idx: int = 0) -> int:
        return self.get_seq_length(layer_idx)

    def get_max_length(self) -> Optional[int]:
        return None

    @property
    def seen_tokens(self) -> int:
        return self._seen_tokens

    @seen_tokens.setter
    def seen_tokens(self, value: int):
        self._seen_tokens = value

    def reorder_cache(self, beam_idx: torch.Tensor):
        """akv/drop_in.py:1119-1128: reorder the batch axis of both tiers."""
        for layer in self.layers:
            if layer._hot_keys is not None:
                layer._hot_keys = layer._hot_keys.index_select(0, beam_idx)
                layer._hot_values = layer._hot_values.index_select(0, beam_idx)
            if layer._warm is not None:
                layer._warm.index_batch(beam_idx)

    def memory_usage(self) -> dict:
        """akv/drop_in.py:1130-1160."""
        keys = ("hot_bytes", "warm_bytes", "warm_bytes_live", "warm_bytes_packed", "warm_bytes_formula",
                "total_bytes", "fp16_equivalent_bytes")
        totals = {k: 0 for k in keys}
        for layer in self.layers:
            stats = layer.memory_usage_bytes()
            for k in keys:
                totals[k] += stats.get(k, 0)
        totals["savings_ratio"] = totals["fp16_equivalent_bytes"] / max(totals["total_bytes"], 1)
        totals["num_layers"] = len(self.layers)
        return totals

    def memory_report(self) -> dict:
        """akv/drop_in.py:1162-1184."""
        stats = self.memory_usage()
        return {"compressed_bytes": stats["total_bytes"], "fp16_equiv_bytes": stats["fp16_equivalent_bytes"],
                "savings_ratio": round(stats["savings_ratio"], 2), "key_bits": self.warm_key_bits,
                "value_bits": self.warm_value_bits, "num_layers": stats["num_layers"],
                "seq_length": self.get_seq_length(0)}

    def __len__(self) -> int:
        return len(self.layers)

    def __getitem__(self, layer_idx: int):
        """akv/drop_in.py:1188-1198: (warm working copy in demotion order, then hot)."""
        if layer_idx < len(self.layers):
            layer = self.layers[layer_idx]
            if layer._hot_keys is not None:
                wk, wv = layer.warm_view()
                if wk is None:
                    return layer._hot_keys, layer._hot_values
                return (torch.cat([wk, layer._hot_keys], dim=2), torch.cat([wv, layer._hot_values], dim=2))
        return torch.tensor([]), torch.tensor([])

    def __iter__(self):
        for i in range(len(self.layers)):
            yield self[i]

    def to_legacy_cache(self):
        """akv/drop_in.py:1203-1205: ((keys, values) per layer) as ``__getitem__`` gives them."""
        return tuple(self[i] for i in range(len(self.layers)))

    @classmethod
    def from_legacy_cache(cls, past_key_values=None) -> "AKVCache":
        """akv/drop_in.py:1273-1280: a default cache fed layer by layer through ``update``."""
        cache = cls()
        if past_key_values is not None:
            for layer_idx, (k, v) in enumerate(past_key_values):
                cache.update(k, v, layer_idx)
        return cache

    @property
    def key_cache(self) -> list:
        """akv/drop_in.py:1214-1221: each layer's keys as ``__getitem__`` gives them."""
        return [self[i][0] for i in range(len(self.layers))]

    @property
    def value_cache(self) -> list:
        """akv/drop_in.py:1223-1229."""
        return [self[i][1] for i in range(len(self.layers))]

    def crop(self, max_length: int):
        """akv/drop_in.py:1231-1243 (speculative-decoding rewind): every layer keeps the
        positions before ``max_length`` (a negative value counts back from the current
        length, as transformers' caches take it).  The reference trims the hot tier from
        its end, where the newest tokens are; a token past max_length that was already
        demoted leaves the packed tier too here, so every layer's view stays whole."""
        for layer in self.layers:
            n = max_length if max_length >= 0 else max(0, layer.get_seq_length() + max_length)
            layer.crop(n)

    def batch_select_indices(self, indices: torch.Tensor) -> "AKVCache":
        """akv/drop_in.py:1256-1265 (beam search): keep / reorder batch elements."""
        self.reorder_cache(indices)
        return self

    def batch_repeat_interleave(self, repeats: int) -> "AKVCache":
        """akv/drop_in.py:1245-1254 (beam expansion): each batch element ``repeats`` times
        in a row, in both tiers."""
        for layer in self.layers:
            if layer._hot_keys is None:
                continue
            idx = torch.arange(layer._hot_keys.shape[0], device=layer._hot_keys.device).repeat_interleave(repeats)
            layer._hot_keys = layer._hot_keys.index_select(0, idx)
            layer._hot_values = layer._hot_values.index_select(0, idx)
            if layer._warm is not None:
                layer._warm.index_batch(idx)
        return self

    def reset(self):
        """akv/drop_in.py:1267-1270: empty (every layer dropped, no tokens seen)."""
        self.layers.clear()
        self._seen_tokens = 0

    @classmethod
    def for_model(cls, model, **kwargs) -> "AKVCache":
        """akv/drop_in.py:1012-1053: a cache sized from ``model.config``
        (num_hidden_layers, or n_layer), the other arguments as given.  The reference
        also applies per-family defaults from its model-adapter registry (preset and
        protected layers) when the caller leaves them out; that registry is not part of
        this build, so pass them explicitly."""
        config = getattr(model, "config", None)
        if config is None:
            raise ValueError("model has no .config attribute")
        n_layers = getattr(config, "num_hidden_layers", None) or getattr(config, "n_layer", None)
        if n_layers is None:
            raise ValueError("Could not find num_hidden_layers in model.config. Pass num_hidden_layers= explicitly.")
        return cls(num_hidden_layers=n_layers, **kwargs)

    @classmethod
    def from_calibration(cls, calibration_path, **overrides) -> "AKVCache":
        """akv/drop_in.py:1282-1315: a cache from a calibration report (JSON, the
        reference's CalibrationReport fields): its protected layers and layer count, its
        average width when within [2, 4] bits (else its preset), and its per-(layer, head)
        widths; ``overrides`` win."""
        import json
        with open(calibration_path) as f:
            rep = json.load(f)
        kwargs = dict(protect_first=rep["recommended_protect_first"], protect_last=rep["recommended_protect_last"],
                      num_hidden_layers=rep["num_layers"])
        avg = float(rep["recommended_average_bits"])
        if 2.0 <= avg <= 4.0:
            kwargs["warm_bits"] = int(round(avg))
        else:
            kwargs["preset"] = rep["recommended_preset"]
        kwargs.update(overrides)
        cache = cls(**kwargs)
        cache._calibration_per_head_bits = {int(k): list(v) for k, v in rep.get("per_head_bits", {}).items()}
        return cache

    def demote(self, keys: torch.Tensor, values: torch.Tensor, importance: Optional[torch.Tensor],
               n_demote: int) -> tuple[WarmTier, torch.Tensor]:
        """Pick ``n_demote`` hot tokens per sequence (lowest importance, protected
        ends kept) and quantize them into a packed warm tier.

        keys / values: (B, H, hot_len, D) on the device; importance: (B, hot_len)
        or (hot_len,).  Returns (warm tier, selected indices (B, n_demote))."""
        B, H, hot_len, D = keys.shape
        idx = select_demote_indices(importance, n_demote, hot_len, self.hot_budget, device=keys.device)
        if idx.dim() == 1:
            idx = idx.unsqueeze(0).expand(B, -1)
        warm = quantize_kv(keys, values, self.warm_key_bits, self.warm_value_bits, self.block_t,
                           self.group_v, self.outlier_fraction, sel=idx)
        return warm, idx


def recommend_preset(model, tokenizer=None, sample_text: Optional[str] = None) -> dict:
    """akv/drop_in.py:1321-1366: a preset suggestion from ``model.config`` by a rough
    size estimate, layers x kv-heads x head_dim^2 x 4 (the reference's heuristic and
    its thresholds: above 5e9 balanced 3-bit, above 1e9 quality 4-bit with a 256-token
    hot window, else quality 4-bit with 512 and two protected layers at each end)."""
    config = getattr(model, "config", None)
    if config is None:
        return {"preset": "balanced", "reason": "No config found, using default"}
    n_layers = getattr(config, "num_hidden_layers", 32)
    n_heads = getattr(config, "num_key_value_heads", getattr(config, "num_attention_heads", 32))
    head_dim = getattr(config, "head_dim", getattr(config, "hidden_size", 4096) // getattr(config, "num_attention_heads", 32))
    est = n_layers * n_heads * head_dim * head_dim * 4
    if est > 5e9:
        return {"preset": "balanced", "warm_bits": 3, "hot_budget": 128, "protect_first": 2, "protect_last": 2,
                "reason": f"Large model ({est / 1e9:.0f}B est.) \u2014 robust to 3-bit"}
    if est > 1e9:
        return {"preset": "quality", "warm_bits": 4, "hot_budget": 256, "protect_first": 1, "protect_last": 1,
                "reason": f"Medium model ({est / 1e9:.1f}B est.) \u2014 use 4-bit for safety"}
    return {"preset": "quality", "warm_bits": 4, "hot_budget": 512, "protect_first": 2, "protect_last": 2,
            "reason": f"Small model ({est / 1e9:.1f}B est.) \u2014 protect more layers"}
