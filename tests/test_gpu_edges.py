"""Kernels at the sizes where their tiles, remainders and dispatch rules turn:
each compared with float64 under a bound that follows from its arithmetic.
"""
import numpy as np
import pytest

from slate_amd import DeviceBuffer as DB
from slate_amd import check

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def host(buf, shape, dtype=np.float32):
    return buf.to_array(dtype, shape)


# Rows 1 / 16 / 17 / 32 / 33 / 64 / 65 (the row tiles of the kernel), K around
# its 16-element units and its rounds of 64 units, N around the 16-, 32- and
# 64-column groups and the two lines of the column rule (4096, 8192).
@pytest.mark.parametrize("B,K,N", [(1, 1, 1), (2, 15, 3), (16, 16, 16), (17, 17, 17), (3, 255, 33), (16, 1031, 100),
                                   (32, 257, 4095), (33, 64, 4097), (5, 130, 8191), (16, 48, 8193), (64, 271, 8200),
                                   (65, 33, 31), (64, 1030, 4100), (20, 515, 8195), (16, 2100, 4099)])
def test_linear_batch_tiles(hip, B, K, N):
    rng = np.random.default_rng(B * 7919 + K * 31 + N)
    X = rng.normal(0, 1, (B, K)).astype(np.float32)
    W = rng.normal(0, 0.5, (K, N)).astype(np.float32)
    C = DB(B * N * 4 + 64)
    C.upload(np.full(B * N + 16, 7.0, np.float32))
    hip.linear_batch(C.p, DB.from_array(X).p, DB.from_array(W).p, B, K, N)
    got = host(C, (B * N + 16,))
    check(0, "linear_batch")
    assert np.all(got[B * N:] == 7.0)                       # nothing past the result is written
    X6, W6 = X.astype(np.float64), W.astype(np.float64)
    # K products and sums of f32, in any order: K roundings of the absolute sum
    bound = (K + 2) * EPS * (np.abs(X6) @ np.abs(W6))
    assert np.all(np.abs(got[:B * N].reshape(B, N) - X6 @ W6) <= bound)


def test_linear_batch_special_values(hip):
    """Infinities and NaN stay in their own rows and columns, also in the
    last, partly filled unit of K; subnormal products are kept."""
    B, K, N = 3, 19, 21
    rng = np.random.default_rng(3)
    X = rng.normal(0, 1, (B, K)).astype(np.float32)
    W = rng.normal(0, 1, (K, N)).astype(np.float32)
    X[0] = 1e-20
    W[:, 0] = 1e-20
    W[18, 5] = np.inf
    X[1, 17] = np.nan
    C = DB(B * N * 4)
    hip.linear_batch(C.p, DB.from_array(X).p, DB.from_array(W).p, B, K, N)
    got = host(C, (B, N))
    assert np.all(np.isnan(got[1])) and np.all(np.isinf(got[[0, 2], 5]))
    keep = [c for c in range(N) if c != 5]
    want = X.astype(np.float64) @ np.where(np.isinf(W), 0, W).astype(np.float64)
    assert np.all(np.isfinite(got[[0, 2]][:, keep]))
    assert abs(got[0, 0] - want[0, 0]) <= (K + 2) * 2.0 ** -149
    np.testing.assert_allclose(got[2, keep], want[2, keep], atol=(K + 2) * EPS * float(np.abs(X[2]).sum() * 4))
