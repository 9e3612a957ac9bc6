"""An update that runs out of memory leaves the caches whole: every allocation of it is made to fail
in turn, and the updates that follow give what an undisturbed cache gives."""
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


class _Failing:
    """``torch.empty`` and ``torch.empty_like`` raising at the k-th call."""

    def __init__(self, monkeypatch, k):
        self.left, self.hit = k, False
        for name in ("empty", "empty_like"):
            monkeypatch.setattr(torch, name, self._wrap(getattr(torch, name)))

    def _wrap(self, f):
        def call(*a, **kw):
            self.left -= 1
            if self.left == 0:
                self.hit = True
                raise torch.OutOfMemoryError("planted")
            return f(*a, **kw)
        return call


def _sweep(make, update, chunks, at, same):
    """``chunks[at]`` fails at every allocation in turn; the views of the later chunks (the failed
    one's tokens among them, if the cache took them) equal those of a cache that never failed."""
    want = []
    ref = make()
    for c in chunks:
        want.append([t.clone() for t in update(ref, c)])
    k = 0
    while True:
        k += 1
        cache = make()
        for c in chunks[:at]:
            update(cache, c)
        taken = cache_len(cache)
        with pytest.MonkeyPatch.context() as mp:
            fail = _Failing(mp, k)
            try:
                update(cache, chunks[at])
            except torch.OutOfMemoryError:
                pass
        if not fail.hit:
            return k - 1
        if cache_len(cache) == taken:  # refused whole: the caller tries again
            update(cache, chunks[at])
        got = [update(cache, c) for c in chunks[at + 1:]]
        for g, w in zip(got, want[at + 1:]):
            same(g, w, k)


def cache_len(cache):
    return cache.get_seq_length() if hasattr(cache, "get_seq_length") else cache._total_len


def _chunks(lens, B, H, D, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [tuple(torch.randn(B, H, n, D, generator=g, device="cuda").to(dtype) for _ in range(2)) for n in lens]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("lens,at", [((40, 50, 1, 2), 1), ((90, 1, 70, 1, 1), 2), ((20, 30, 1), 1)])
def test_kivi_update(dtype, lens, at):
    import akv
    announce(f"failed KIVI update {dtype} {lens} at {at}")

    def same(g, w, k):
        assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(g, w)), k

    n = _sweep(lambda: akv.create_baseline("kivi_fused", key_bits=2, value_bits=4, group_size=64, residual_length=32),
               lambda c, kv: c.update(*kv, 0), _chunks(lens, 2, 3, 128, dtype, 5), at, same)
    assert n >= 4  # the views, the residuals and, where the tier grows, its tensors


def test_kivi_refused_launch(monkeypatch):
    """A refused append leaves tier and residual as they were; the tokens go in with the next one."""
    import akv
    from akv import _native as nat
    announce("refused KIVI append")
    chunks = _chunks((90, 5, 1), 1, 2, 64, torch.float16, 6)
    caches = [akv.create_baseline("kivi_fused", key_bits=4, value_bits=4, group_size=32, residual_length=16)
              for _ in range(2)]
    for c in caches:
        c.update(*chunks[0], 0)
    caches[0].update(*chunks[1], 0)
    with pytest.MonkeyPatch.context() as mp:
        lib = nat.load()
        mp.setattr(nat, "load", lambda: type("L", (), {
            "__getattr__": lambda self, name: (lambda *a: nat.AKV_E_SHAPE) if name == "akv_kivi_append" else getattr(lib, name)})())
        with pytest.raises(Exception):
            caches[1].update(*chunks[1], 0)
    assert caches[1]._quant_keys[0].n == 74 and caches[1]._residual_keys[0].shape[2] == 21
    for a, b in zip(caches[0].update(*chunks[2], 0), caches[1].update(*chunks[2], 0)):
        assert torch.equal(a, b)


def _whole(layer, seen, k):
    """Every token is in one tier once, at its position, and the views hold the tokens."""
    total = layer.get_seq_length()
    pos = [layer._hot_positions] + ([layer._warm_positions] if layer._warm is not None else [])
    pos = torch.cat(pos).sort().values
    assert torch.equal(pos, torch.arange(total, device="cuda")), k
    n_warm = total - layer._hot_keys.shape[2]
    assert layer._warm_len == n_warm and layer._importance.shape[0] == layer._hot_keys.shape[2], k
    assert bool(torch.isfinite(layer._importance).all()), k
    if layer._proxy_score is not None:
        assert layer._proxy_score.shape[0] <= n_warm and bool(torch.isfinite(layer._proxy_score).all()), k
    for view, x in zip((layer.keys, layer.values), seen):
        # 4 bits over a range of ~9, twice where a token was promoted and demoted again
        assert float((view - x).abs().max()) < 1.0, k


@pytest.mark.parametrize("kw", [dict(), dict(outlier_fraction=0.03), dict(per_head_bits=[4, 3, 4])])
@pytest.mark.parametrize("lens,at", [((70, 9), 0), ((40, 50, 1), 1), ((120, 30, 1, 1), 2), ((90, 200, 1), 1)])
def test_layer_update(kw, lens, at):
    from akv.drop_in import AKVLayer
    announce(f"failed layer update {kw} {lens} at {at}")
    chunks = _chunks(lens, 2, 3, 64, torch.float16, 8)
    k = 0
    while True:
        k += 1
        layer = AKVLayer(warm_bits=4, hot_budget=64, promotion_threshold=0.02, **kw)
        for c in chunks[:at]:
            layer.update(*c)
        taken = layer.get_seq_length()
        with pytest.MonkeyPatch.context() as mp:
            fail = _Failing(mp, k)
            try:
                layer.update(*chunks[at])
            except torch.OutOfMemoryError:
                pass
        if not fail.hit:
            break
        if layer.get_seq_length() == taken:
            layer.update(*chunks[at])
        seen = [torch.cat([c[i] for c in chunks[:at + 1]], dim=2) for i in range(2)]
        for c in chunks[at + 1:]:
            seen = [torch.cat([s, x], dim=2) for s, x in zip(seen, c)]
            layer.update(*c)
        if len(chunks) > at + 1 or layer.keys.shape[2] == seen[0].shape[2]:
            _whole(layer, seen, k)
    assert k > 8


@pytest.mark.parametrize("kw", [dict(), dict(per_head_bits=[4, 3, 4])])
def test_layer_crop(kw):
    from akv.drop_in import AKVLayer
    announce(f"failed crop {kw}")
    chunks = _chunks((150, 1, 3), 1, 3, 64, torch.float16, 9)
    k = 0
    while True:
        k += 1
        layer = AKVLayer(warm_bits=4, hot_budget=64, **kw)
        for c in chunks[:2]:
            layer.update(*c)
        with pytest.MonkeyPatch.context() as mp:
            fail = _Failing(mp, k)
            try:
                layer.crop(60)
            except torch.OutOfMemoryError:
                assert layer.get_seq_length() == 151
                assert layer._hot_keys.shape[2] + layer._warm_len == 151
        layer.crop(60)
        layer.update(*chunks[2])
        _whole(layer, [torch.cat([chunks[0][i][:, :, :60], chunks[2][i]], dim=2) for i in range(2)], k)
        if not fail.hit:
            break
    assert k > 4  # the packed tier loses tokens too


def test_a_layer_saved_with_its_positions_goes_on():
    """Copies of a layer, in the present form and with the positions as a host attribute, go on as it does."""
    import copy

    from akv.drop_in import AKVLayer
    announce("copied layers")
    chunks = _chunks((90, 1, 5), 1, 2, 64, torch.float16, 12)
    for protect in (False, True):
        layer = AKVLayer(warm_bits=4, hot_budget=64, protect=protect)
        layer.update(*chunks[0])
        a, b = copy.deepcopy(layer), AKVLayer.__new__(AKVLayer)
        state = copy.deepcopy(layer.__dict__)
        state.pop("_positions")
        state["_hot_positions"] = layer._hot_positions.cpu()
        b.__setstate__(state)
        for c in chunks[1:]:
            want = layer.update(*c)
            for x in (a, b):
                assert all(torch.equal(p, q) for p, q in zip(x.update(*c), want))
                assert torch.equal(x._hot_positions, layer._hot_positions)
