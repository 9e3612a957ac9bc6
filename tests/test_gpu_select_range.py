"""Demote selection at the sizes where its storage of the keys changes (registers, LDS,
memory) and on the score distributions that drive its histogram: exact index lists."""
import numpy as np
import pytest
import torch

from gpu_util import announce, to_dev
from oracle import selection as osel

pytestmark = pytest.mark.gpu


def _scores(kind, rows, n, rng):
    if kind == "uniform":
        return rng.random((rows, n)).astype(np.float32)
    if kind == "equal":
        return np.full((rows, n), 0.3, np.float32)
    if kind == "recency":  # decayed ones: a few values, long runs of each
        return (0.3 ** (np.arange(n)[::-1] * 5 // n)).astype(np.float32)[None].repeat(rows, 0)
    if kind == "close":  # one binade, two levels of bins and more keys in a bin than the list holds
        return np.where(rng.random((rows, n)) < 0.5, 1.0 + rng.integers(0, 9, (rows, n)) * 2.0 ** -23,
                        rng.random((rows, n)) * 1e30).astype(np.float32)
    x = rng.standard_normal((rows, n)).astype(np.float32) * np.float32(1e-38)  # wide: denormals to the extremes
    x[rng.random((rows, n)) < 0.2] = -np.inf
    x[rng.random((rows, n)) < 0.2] = np.inf
    x[rng.random((rows, n)) < 0.2] = np.nan
    x[rng.random((rows, n)) < 0.1] = -np.finfo(np.float32).max
    x[rng.random((rows, n)) < 0.1] = -0.0
    return x


@pytest.mark.parametrize("kind", ["uniform", "equal", "recency", "close", "wide"])
@pytest.mark.parametrize("rows,n", [(3, 1), (2, 63), (2, 1025), (2, 2048), (2, 2049), (3, 8192), (2, 8193),
                                    (2, 16383), (1, 32768), (2, 32769), (1, 65535), (1, 65537), (1, 131071)])
def test_select_storage_and_distributions(kind, rows, n):
    from akv.drop_in import select_demote_indices
    announce(f"select {kind} {rows}x{n}")
    imp = _scores(kind, rows, n, np.random.default_rng(n))
    for take in sorted({1, n // 3, n // 2, n - min(n, 40), n - 1, n} - {0}):
        got = select_demote_indices(to_dev(imp), take, n, 64).cpu().numpy().reshape(rows, take)
        for r in range(rows):
            assert np.array_equal(got[r], osel.select_demote_indices(imp[r], take, n, 64)), (r, take)
