"""Which decode kernel a tier goes to, read from the plan without a GPU: decode_fast_kernel takes
at most 256 workgroups' partials, decode_split_kernel four per compute unit, so the workspace of a
long context tells them apart."""
import ctypes

import pytest


def _workspace(kind="affine", B=3, Hq=28, Hkv=4, M=3, n_warm=9001, group=64, n_out=0, stride=0, odata=0x30000):
    from akv import _native as nat
    lib = nat.load()
    a = nat.DecodeArgs()
    a.abi_version = nat.ABI_VERSION
    a.q_dtype = nat.DT_F16
    a.B, a.Hq, a.Hkv, a.M, a.D = B, Hq, Hkv, M, 128
    a.q = a.out = a.k_hot = a.v_hot = 0x10000  # planning only: never dereferenced
    a.n_hot = 333
    a.sm_scale = 128 ** -0.5
    w = a.warm
    w.n_warm, w.token_stride = n_warm, stride
    w.k_codes = w.v_codes = w.k_scale = w.k_zero = w.v_scale = w.v_zero = 0x20000
    if kind == "affine":
        w.kind, w.bits_k, w.bits_v, w.block_t, w.group_v, w.n_out = nat.WARM_AFFINE, 2, 2, 32, group, n_out
        if n_out:
            w.k_oidx = w.v_oidx = 0x30000
            w.k_odata = w.v_odata = odata
    else:
        w.kind, w.bits_k, w.bits_v, w.group_size = nat.WARM_LEGACY, 4, 4, group
        w.meta_dtype, w.legacy_sym, w.warm_heads = nat.DT_F16, 0, B * Hkv
    nbytes = lib.akv_decode_workspace_bytes(ctypes.byref(a))
    assert nbytes > 0, lib.akv_last_error()
    return nbytes


def _fast(**kw):
    """Whether the call's workspace is of the size of the same call that surely is on the fast kernel."""
    ref = _workspace(**{**kw, "n_warm": 9008, "group": 32, "n_out": 0, "stride": 0})
    return _workspace(**kw) < 2 * ref


@pytest.mark.parametrize("kind", ["affine", "legacy"])
@pytest.mark.parametrize("group,n,fast", [(32, 9001, True), (64, 9000, True), (64, 9001, False), (64, 9002, False),
                                          (128, 9000, True), (128, 9004, False), (128, 9001, False)])
def test_meta_rows_off_16_bytes_leave_the_fast_kernel(kind, group, n, fast):
    assert _fast(kind=kind, group=group, n_warm=n) == fast
    if kind == "legacy":  # a tier's rows are `stride` apart whatever its length
        assert _fast(kind=kind, group=group, n_warm=9001, stride=n + 8) == fast


@pytest.mark.parametrize("n_out", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [9000, 9001])
def test_outlier_values_off_a_dword_leave_the_fast_kernel(n_out, n):
    """Odd lengths and counts stay (every second head's values start half a dword in, which the
    kernel straightens); tensors that start half a dword in do not."""
    kw = dict(B=3, Hq=4, Hkv=4, M=1, n_warm=n, group=32, n_out=n_out)
    assert _fast(**kw)
    assert not _fast(**kw, odata=0x30002)
