"""The prefill's scratch: per (batch, kv head), 16-row chunk and split, as many rows as there are, of
D + 4 floats."""
import ctypes

import pytest


@pytest.mark.parametrize("M,g,rows", [(1, 1, 1), (1, 8, 8), (5, 3, 15), (2, 8, 16), (9, 3, 32)])
@pytest.mark.parametrize("splits", [2, 8, 40])
def test_rows_of_short_chunks(M, g, rows, splits):
    from akv import _native as nat
    lib = nat.load()
    a = nat.PrefillArgs()
    a.abi_version, a.B, a.Hq, a.Hkv, a.M, a.D, a.q_dtype = nat.ABI_VERSION, 3, 2 * g, 2, M, 128, nat.DT_F16
    a.q = a.out = a.k_hot = a.v_hot = 0x10000  # planning only
    a.n_hot, a.sm_scale, a.num_splits = 32 * 400, 128 ** -0.5, splits
    a.warm.kind = nat.WARM_NONE
    assert lib.akv_prefill_workspace_bytes(ctypes.byref(a)) == -(-(6 * splits * rows * 132 * 4) // 256) * 256
