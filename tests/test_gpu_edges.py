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


def _q8(rng, M, K):
    """Q8_0 bytes (34-byte blocks) and the weights in float64."""
    d = rng.uniform(1e-4, 2e-2, (M, K // 32, 1)).astype(np.float16)
    d[rng.random(d.shape) < 0.1] *= -1
    q = rng.integers(-128, 128, (M, K // 32, 32)).astype(np.int8)
    raw = np.concatenate([d.view(np.uint8).reshape(M, K // 32, 2), q.view(np.uint8)], -1)
    return np.ascontiguousarray(raw.reshape(-1)), (d.astype(np.float64) * q).reshape(M, K)


# One row: the four / eight rows a workgroup owns and the line between them
# (4096 rows), half blocks below a wave, 512 half blocks (K 8192) and one more
# block (two passes).  More rows: the regrouping pass at partly filled groups
# (K % 256), one to five groups (K 32 .. 1056), row tiles (M % 16) and blocks
# that start on any even byte.
@pytest.mark.parametrize("B,M,K", [(1, 1, 32), (1, 3, 64), (1, 5, 1024), (1, 4095, 96), (1, 4097, 288), (1, 9, 8192),
                                   (1, 7, 8224), (1, 17, 14336), (2, 1, 32), (3, 15, 288), (16, 33, 224),
                                   (17, 100, 800), (64, 47, 544), (65, 260, 1056)])
def test_q8_row_layout_edges(hip, B, M, K):
    rng = np.random.default_rng(B * 131 + M * 17 + K)
    raw, w = _q8(rng, M, K)
    X = rng.normal(0, 1, (B, K)).astype(np.float32)
    X[0, :32] *= 1e3
    A = DB(raw.size + 16)
    A.upload(np.concatenate([np.zeros(2, np.uint8), raw]))   # blocks start on any even byte
    T, R0 = DB(hip.lib.slate_hip_q8_0_tiled_bytes(M, K)), DB.from_array(raw)
    check(hip.lib.slate_hip_q8_0_tile(T.p, R0.p, M, K), "q8_0_tile")
    Xd, Y, Yt = DB.from_array(X), DB(B * M * 4), DB(B * M * 4)
    check(hip.lib.slate_hip_matmul_q8_0(Y.p, A.ptr + 2, Xd.p, B, M, K), "matmul_q8_0")
    check(hip.lib.slate_hip_matmul_q8_0_tiled(Yt.p, T.p, Xd.p, B, M, K), "matmul_q8_0_tiled")
    got, tiled = host(Y, (B, M)), host(Yt, (B, M))
    assert np.array_equal(got.view(np.uint32), tiled.view(np.uint32))
    X6 = X.astype(np.float64)
    # one row: 8 products, their sum, d, at most two passes, 6 + 8 sums: under
    # 32 roundings of the absolute sum.  More rows: x as two f16 (2^-22 of the
    # group's largest value each) and a rounding per MFMA, d and group sum.
    size = np.abs(X6) @ np.abs(w).T
    if B == 1:
        bound = 32 * EPS * size
    else:
        xmax = np.repeat(np.abs(np.pad(X6, ((0, 0), (0, -K % 256)))).reshape(B, -1, 256).max(-1), 256, 1)[:, :K]
        bound = (K // 32 * 18 + 32) * EPS * size + 2.0 ** -22 * (xmax @ np.abs(w).T)
    assert np.all(np.abs(got - X6 @ w.T) <= bound)
