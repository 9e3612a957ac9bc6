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
