"""The importance update with its query sum split over workgroups (20 query rows and more, or
40 (batch, head, query) rows with pooling):
every dtype, row lengths at and around the 16-byte chunk and the 64-lane tile, partial query
blocks, head counts off 8, pooling and windows, scores shorter and longer than the rows."""
import numpy as np
import pytest
import torch

from gpu_util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,M,N,W,ks,ns", [
    (1, 1, 20, 8, 0, 1, 8), (1, 3, 21, 9, 0, 1, 9), (2, 4, 24, 255, 0, 1, 255), (1, 8, 29, 511, 0, 1, 511),
    (1, 8, 5, 300, 0, 7, 300), (2, 12, 2, 700, 0, 7, 700),
    (1, 9, 33, 513, 0, 1, 600), (2, 6, 40, 1000, 32, 7, 1000), (1, 16, 64, 1025, 9, 64, 1025), (1, 2, 300, 77, 0, 5, 40),
    (2, 1, 257, 2047, 0, 1, 2047),
])
def test_split_query_sum(dt, B, H, M, N, W, ks, ns):
    from akv import _native as nat
    from akv.importance import accumulate
    announce(f"importance split {dt} B{B} H{H} M{M} N{N} W{W} ks{ks} ns{ns}")
    g = torch.Generator(device="cuda").manual_seed(M * N + H)
    attn = torch.softmax(3 * torch.randn(B, H, M, N, generator=g, device="cuda"), -1).to(dt)
    s0 = torch.rand(ns, generator=g, device="cuda")
    a = nat.ImportanceArgs()
    a.abi_version, a.attn_dtype, a.attn = nat.ABI_VERSION, nat.dtype_code(dt), attn.data_ptr()
    a.B, a.H, a.M, a.N, a.n_scores, a.scores = B, H, M, N, ns, s0.data_ptr()
    a.q_window, a.pool_kernel = W, ks
    assert nat.load().akv_importance_workspace_bytes(a) > 0  # the split path takes the call
    x = attn.double().cpu().numpy()
    imp = (x.sum((0, 1)) / (B * H))[M - W if W and W < M else 0:].sum(0)
    if ks > 1 and N > ks:
        pad = np.concatenate([np.zeros(ks // 2), imp, np.zeros(ks)])
        imp = np.array([pad[n:n + ks].sum() / ks for n in range(N)])
    full = np.zeros(ns)
    full[:min(ns, N)] = imp[:ns]
    exp = s0.double().cpu().numpy() * np.float64(np.float32(0.9)) + full
    for _ in range(2):
        got = accumulate(s0.clone(), attn, 0.9, q_window=W, pool_kernel=ks).cpu().numpy()
        # every term is non-negative: B*H + M + ks + 6 fp32 roundings at most, each 2^-24 relative
        np.testing.assert_allclose(got, exp, rtol=(B * H + M + ks + 6) * 2.0 ** -24, atol=1e-30)
    # a first score that is not finite stays in its own key
    attn[0, 0, -1, N // 2] = float("inf")
    got = accumulate(torch.zeros(N, device="cuda"), attn, 0.0, q_window=W, pool_kernel=1)
    assert torch.isinf(got[N // 2]) and int(torch.isfinite(got).sum()) == N - 1
