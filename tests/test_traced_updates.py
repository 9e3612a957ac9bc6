"""What a program sees of a cache layer's update when something looks at its operations: fake
tensors, a dispatch mode, a trace.  Before a demotion, and always in protected layers, the update is
joins and fills that such a program has to find."""
import pytest
import torch

from gpu_util import announce


def _kv(n, seed, H=2, D=64, dtype=torch.float16):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return tuple(torch.randn(1, H, n, D, generator=g, device="cuda").to(dtype) for _ in range(2))


@pytest.mark.parametrize("protect", [False, True])
def test_fake_tensors(protect):
    from torch._subclasses.fake_tensor import FakeTensorMode

    from akv.drop_in import AKVLayer
    with FakeTensorMode():
        layer = AKVLayer(hot_budget=64, protect=protect)
        for n in (5, 1, 2):
            k, v = layer.update(*(torch.empty(1, 2, n, 64, dtype=torch.float16, device="cuda") for _ in range(2)))
        assert k.shape == v.shape == (1, 2, 8, 64) and k.device.type == "cuda"
        assert layer._hot_positions.shape == (8,) and layer._total_len == 8


def test_default_device_context_is_no_observer():
    from akv.row_moves import observed
    with torch.device("cpu"):
        assert not observed()
    assert not observed()


@pytest.mark.gpu
@pytest.mark.parametrize("protect", [False, True])
def test_a_trace_holds_the_joins(protect):
    """make_fx over two updates: the graph, run on other tokens, joins those."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from akv.drop_in import AKVLayer
    announce(f"traced layer updates, protect={protect}")

    def step(k0, v0, k1, v1):
        layer = AKVLayer(hot_budget=64, protect=protect)
        layer.update(k0, v0)
        k, v = layer.update(k1, v1)
        return k, v, layer._hot_positions

    graph = make_fx(step)(*_kv(5, 1), *_kv(2, 2))
    a, b = _kv(5, 3), _kv(2, 4)
    k, v, pos = graph(*a, *b)
    assert torch.equal(k, torch.cat([a[0], b[0]], dim=2)) and torch.equal(v, torch.cat([a[1], b[1]], dim=2))
    assert torch.equal(pos, torch.arange(7, device="cuda"))


@pytest.mark.gpu
def test_a_dispatch_mode_changes_nothing():
    """Prompt, demotion, promotions and crop under a mode that looks on: the same tiers and views."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from akv.drop_in import AKVLayer

    class Look(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    announce("layer updates under a dispatch mode")
    layers = [AKVLayer(hot_budget=64, outlier_fraction=0.02, promotion_threshold=0.02) for _ in range(2)]
    for i, n in enumerate((150, 1, 1, 90, 1)):
        kv = _kv(n, 10 + i, H=3)
        got = layers[0].update(*kv)
        with Look():
            seen = layers[1].update(*kv)
        assert all(torch.equal(a, b) for a, b in zip(got, seen)), i
    layers[0].crop(120)
    with Look():
        layers[1].crop(120)
    a, b = layers
    assert torch.equal(a._warm_positions, b._warm_positions) and torch.equal(a._hot_positions, b._hot_positions)
    assert torch.equal(a._importance, b._importance) and torch.equal(a._hot_keys, b._hot_keys)
    assert (a._proxy_score is None) == (b._proxy_score is None)
    assert all(torch.equal(x, y) for x, y in zip(a.warm_view(), b.warm_view()))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_kivi_views_under_a_dispatch_mode(dtype):
    from torch.utils._python_dispatch import TorchDispatchMode

    import akv

    class Look(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    announce(f"KIVI updates under a dispatch mode {dtype}")
    caches = [akv.create_baseline("kivi_fused", key_bits=2, value_bits=2, group_size=64, residual_length=16)
              for _ in range(2)]
    for i, n in enumerate((40, 1, 80, 3)):
        kv = _kv(n, 20 + i, dtype=dtype)
        got = caches[0].update(*kv, 0)
        with Look():
            seen = caches[1].update(*kv, 0)
        assert all(torch.equal(a, b) for a, b in zip(got, seen)), i
