"""akv_rows_move against torch indexing (every map, unit width, dtype pair and stride) and
akv_promote_select against the mask / topk rule it stands for: exact."""
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


def _x(shape, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    if dt in (torch.uint8, torch.int32, torch.int64):
        return torch.randint(0, 200, shape, generator=g, device="cuda").to(dt)
    return torch.randn(shape, generator=g, device="cuda").to(dt)


@pytest.mark.parametrize("B,H,T,C", [(1, 1, 1, 1), (2, 3, 63, 48), (1, 2, 64, 7), (2, 1, 65, 128), (3, 2, 200, 5), (1, 4, 1000, 16)])
def test_row_moves_match_indexing(B, H, T, C):
    from akv.row_moves import GATHER, KEEP, SCATTER, RowMoves
    announce(f"row moves {B}x{H}x{T}x{C}")
    perm = torch.randperm(T, device="cuda")
    drop = perm[: T // 3].sort().values
    left = torch.ones(T, dtype=torch.bool, device="cuda")
    left[drop] = False
    nk = T - drop.numel()
    for s, (a, b) in enumerate([(torch.uint8, torch.uint8), (torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                (torch.float16, torch.float32), (torch.float32, torch.float32), (torch.int64, torch.int64)]):
        x = _x((B, H, T, C), a, s)
        wide = _x((B, H, T, C + 3), a, s + 50)[..., 1:C + 1]      # rows off every boundary
        turned = _x((B, T, H, C), a, s + 90).transpose(1, 2)      # the (B, N, H, D) layout of a model
        for src in (x, wide, turned):
            e = lambda n: torch.full((B, H, n, C), 9, dtype=b, device="cuda")  # noqa: E731
            same, keep, gath, scat = e(T + 2), e(nk), e(T), e(T + 5)
            mv = RowMoves()
            mv.copy(same, src, T, at=1)
            mv.copy(keep, src, nk, KEEP)
            mv.run(drop, drop.numel())
            mv.copy(gath, src, T, GATHER)
            mv.copy(scat, src, T, SCATTER)
            mv.run(perm, T)
            y = src.to(b)
            assert torch.equal(same[:, :, 1:T + 1], y) and bool((same[:, :, [0, T + 1]] == 9).all())
            assert torch.equal(keep, y[:, :, left]) and torch.equal(gath, y[:, :, perm])
            assert torch.equal(scat[:, :, perm], y) and bool((scat[:, :, T:] == 9).all())
    v, f, c, d = _x((T,), torch.float32, 7), *(torch.zeros(T + 1, dtype=dt, device="cuda") for dt in
                                                (torch.float32, torch.int64, torch.int32))
    mv = RowMoves()
    mv.copy(f, v, T, at=1, value=0.3)
    mv.fill(f, 1, 2.0)
    mv.count(c, T, 5, at=1)
    mv.count(d, T, 3, 0)
    mv.run()
    assert torch.equal(f, torch.cat([torch.full((1,), 2.0, device="cuda"), v * 0.3]))
    assert c.tolist() == [0] + list(range(5, 5 + T)) and d.tolist() == [3] * T + [0]


@pytest.mark.parametrize("n", [1, 64, 2048, 2049, 8193, 40000, 70001])
@pytest.mark.parametrize("kind", ["few", "many", "none", "nan", "ties"])
def test_promote_select(n, kind):
    import ctypes
    from akv import _native as nat
    announce(f"promote {n} {kind}")
    g = torch.Generator(device="cuda").manual_seed(n)
    sim, prev = (torch.rand(n, generator=g, device="cuda") - 0.5 for _ in range(2))
    prev = prev.abs()
    thr, cap = {"few": 0.99, "none": 2.0}.get(kind, 0.05), 16
    if kind == "nan":
        sim[:: max(1, n // 5)] = float("nan")
    if kind == "ties":
        sim, prev = (sim * 4).round() / 4, torch.zeros_like(prev)
    if kind == "few":
        sim[torch.randperm(n, generator=g, device="cuda")[:7]] = 20.0
    for p in (prev, None):
        new = torch.empty(n, device="cuda")
        out = torch.full((1 + cap,), -1, dtype=torch.int64, device="cuda")
        f = ctypes.c_float
        nat.check(nat.load().akv_promote_select(sim.data_ptr(), nat.ptr(p), new.data_ptr(), n, f(0.7), f(1 - 0.7), f(thr),
                                                cap, out.data_ptr(), nat.stream_of(sim)))
        s = sim.abs() if p is None else 0.7 * p + (1 - 0.7) * sim.abs()
        assert torch.equal(new.view(torch.int32), s.view(torch.int32))
        mask = s > thr
        if int(mask.sum()) > cap:  # NaN first, then the largest, equal ones lowest index first
            order = torch.sort(torch.nan_to_num(s, nan=float("inf")), descending=True, stable=True).indices[:cap]
            mask = torch.zeros_like(mask)
            mask[order] = True
        exp = mask.nonzero().flatten().tolist()
        assert out[0].item() == len(exp) and out[1:1 + len(exp)].tolist() == exp


def test_update_keeps_autograd_and_refuses_other_shapes():
    """Hot tokens that require grad reach the returned view with their graph; tokens of another
    head count are refused before a tier changes."""
    from akv.drop_in import AKVLayer
    announce("layer update autograd / refusal")
    layer = AKVLayer(hot_budget=32)
    layer.update(*(_x((1, 2, 50, 64), torch.float16, i) for i in range(2)))
    k = _x((1, 2, 1, 64), torch.float16, 5).requires_grad_()
    fk, fv = layer.update(k, _x((1, 2, 1, 64), torch.float16, 6))
    fk[:, :, -1].float().sum().backward()
    assert torch.equal(k.grad, torch.ones_like(k))
    n = layer._warm.n, layer._hot_keys.shape[2], layer.get_seq_length()
    with pytest.raises(RuntimeError):
        layer.update(*(_x((1, 3, 1, 64), torch.float16, i) for i in range(2)))
    assert n == (layer._warm.n, layer._hot_keys.shape[2], layer.get_seq_length())


@pytest.mark.parametrize("T,n", [(3100, 1025), (3100, 2047), (3100, 2049), (20011, 1024), (20011, 4097), (20011, 15000), (20011, 20010)])
@pytest.mark.parametrize("kind", ["random", "run", "ends", "every"])
def test_keep_against_long_lists(T, n, kind):
    """Lists past the 1024 samples of the kernel's first search: the second search sees 2 to 20
    entries between two samples, in lists without any structure and with all of it."""
    from akv.row_moves import KEEP, RowMoves
    announce(f"row moves KEEP T={T} n={n} {kind}")
    g = torch.Generator(device="cuda").manual_seed(T + n)
    if kind == "random":
        drop = torch.randperm(T, generator=g, device="cuda")[:n]
    elif kind == "run":  # a prompt's oldest tokens
        drop = torch.arange(n, device="cuda") + min(4, T - n)
    elif kind == "ends":  # rows 0 and T - 1 among them
        drop = torch.cat([torch.arange(n // 2, device="cuda"), torch.arange(T - (n - n // 2), T, device="cuda")])
    else:
        drop = torch.linspace(0, T - 1, n, device="cuda", dtype=torch.float64).round().long().unique()
    drop = drop.sort().values
    left = torch.ones(T, dtype=torch.bool, device="cuda")
    left[drop] = False
    nk = T - drop.numel()
    x, pos = _x((2, 3, T, 24), torch.float16, n), torch.arange(T, device="cuda") * 7
    a, b = torch.zeros(2, 3, nk + 1, 24, dtype=torch.float16, device="cuda"), torch.zeros(nk + 1, dtype=torch.int64, device="cuda")
    mv = RowMoves()
    mv.copy(a, x, nk, KEEP)
    mv.copy(b, pos, nk, KEEP)
    mv.run(drop, drop.numel())
    assert torch.equal(a[:, :, :nk], x[:, :, left]) and not bool(a[:, :, nk].any())
    assert torch.equal(b[:nk], pos[left]) and int(b[nk]) == 0
