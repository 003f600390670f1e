"""Kernels at the sizes where their tiles, remainders and dispatch rules turn:
each compared with float64 under a bound that follows from its arithmetic.
"""
import numpy as np
import pytest

import slate_amd
from oracle.pyoracle import OracleModel
from slate_amd import DeviceBuffer as DB
from slate_amd import check
from slate_amd.synth import make_llama
from tests.helpers import Q4, Q4_SEED, relerr

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


# One row into its own memory (whole, or its second half): every result is
# made from the row as it came, as where the results go elsewhere.
@pytest.mark.parametrize("M,K,off", [(4096, 4096, 0), (14336, 4096, 2048), (2048, 8192, 4096)])
def test_q8_matvec_over_its_own_row(hip, M, K, off):
    rng = np.random.default_rng(M + K)
    raw, w = _q8(rng, M, K)
    x = rng.normal(0, 1, K).astype(np.float32)
    A, T = DB.from_array(raw), DB(hip.lib.slate_hip_q8_0_tiled_bytes(M, K))
    check(hip.lib.slate_hip_q8_0_tile(T.p, A.p, M, K), "q8_0_tile")
    x6 = x.astype(np.float64)
    # (the bound of test_q8_row_layout_edges for more than one row)
    xmax = np.repeat(np.abs(x6).reshape(-1, 256).max(-1), 256)
    bound = (K // 32 * 18 + 32) * EPS * (np.abs(w) @ np.abs(x6)) + 2.0 ** -22 * (np.abs(w) @ xmax)
    for fn, weights in ((hip.lib.slate_hip_matmul_q8_0, A), (hip.lib.slate_hip_matmul_q8_0_tiled, T)):
        for _ in range(3):
            buf = DB((K + M) * 4)
            buf.upload(x)
            check(fn(buf.ptr + 4 * off, weights.p, buf.p, 1, M, K), "matmul_q8_0")
            got = host(buf, (K + M,))[off:off + M]
            assert np.all(np.abs(got - w @ x6) <= bound)


# Widths around the one-, two- and four-float4 forms (4096, 8192, 16384), odd
# widths and rows that start off 16 bytes (the plain form); y may be x.
@pytest.mark.parametrize("D,off", [(1, 0), (3, 0), (4, 0), (256, 1), (260, 0), (4096, 0), (4100, 0), (8192, 0),
                                   (8196, 0), (12289, 0), (16384, 0), (16388, 0), (4096, 3)])
def test_rmsnorm_rows_widths(hip, D, off):
    rng = np.random.default_rng(D + off)
    B, eps = 3, 1e-5
    x = rng.normal(0, 2, (B, D)).astype(np.float32)
    w = rng.normal(1, 0.2, D).astype(np.float32)
    xb = DB(B * D * 4 + 32)
    pad = np.zeros(off, np.float32)
    xb.upload(np.concatenate([pad, x.reshape(-1), np.full(4, 9, np.float32)]))
    y, wd = DB(B * D * 4), DB.from_array(w)
    check(hip.rmsnorm_rows(y.p, xb.ptr + 4 * off, wd.p, B, D, eps), "rmsnorm_rows")
    check(hip.rmsnorm_rows(xb.ptr + 4 * off, xb.ptr + 4 * off, wd.p, B, D, eps), "rmsnorm_rows in place")
    x6 = x.astype(np.float64)
    want = x6 * w / np.sqrt((x6 * x6).mean(-1, keepdims=True) + np.float64(np.float32(eps)))
    raw = host(xb, (off + B * D + 4,))
    assert np.all(raw[-4:] == 9)
    for got in (host(y, (B, D)), raw[off:off + B * D].reshape(B, D)):
        # at most 17 squares per thread in f32 (half of their roundings under
        # the root), then eight roundings to the product
        assert np.all(np.abs(got - want) <= 20 * EPS * np.abs(want))


def test_rope_rows_counts_bad_rows_of_each_call(hip):
    x = np.ones((6, 8), np.float32)
    for bad in (2, 1, 0, 3, 0):
        pos = np.array([5] * (6 - bad) + [9, -9, 8][:bad], np.int32)
        xb = DB.from_array(x)
        hip.lib.slate_hip_clear_error()
        rc = hip.rope_rows(xb.p, DB.from_array(pos).p, 6, 1, 8, 10000.0, 8)
        err = hip.lib.slate_hip_last_error()
        hip.lib.slate_hip_clear_error()
        assert rc == (-1 if bad else 0)
        assert (b"%d rows" % bad in err) if bad else err is None
        got = host(xb, (6, 8))
        assert np.array_equal(got[6 - bad:], x[6 - bad:]) and not np.any(np.all(got[:6 - bad] == 1, -1))


def _q4k(rng, M, K):
    """Q4_K bytes, the weights in float64 and the size of their two terms
    (d sc q and dmin mn)."""
    raw = rng.integers(0, 256, (M * K // 256, 144), dtype=np.uint8)
    head = rng.uniform(1e-5, 1e-3, (raw.shape[0], 2)).astype(np.float16)
    raw[:, :4] = head.view(np.uint8).reshape(-1, 4)
    s = raw[:, 4:16].astype(np.int64)
    sc = np.concatenate([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1)
    mn = np.concatenate([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
    q = raw[:, 16:].reshape(-1, 8, 16)
    q = np.concatenate([q & 15, q >> 4], 2).astype(np.float64)
    a = (head[:, 0:1].astype(np.float64) * sc)[..., None] * q
    b = (head[:, 1:2].astype(np.float64) * mn)[..., None] * np.ones(32)
    return raw.reshape(-1), (a - b).reshape(M, K), (a + b).reshape(M, K)


# Unsplit plans write the caller's rows themselves: row counts inside and at
# the end of 16-row tiles on the decode kernel (one and two tiles) and the
# prompt kernel (groups of two and four tiles and a shorter last one); and
# the line between the two forms for at most 16 rows (8000 x 256: split).
@pytest.mark.parametrize("B,M,K", [(2, 49163, 256), (13, 49163, 256), (16, 50001, 512), (17, 49163, 256),
                                   (32, 49163, 256), (33, 40007, 512), (63, 40007, 256), (65, 40007, 256),
                                   (9, 8000, 512), (13, 3000, 19968)])
@pytest.mark.parametrize("form", ["row", "tiled", "noalloc"])
def test_q4k_rows_of_the_output(hip, B, M, K, form):
    if form == "noalloc" and B * M > 1.5e6:
        pytest.skip("one split of partials is over that entry's fixed scratch")
    rng = np.random.default_rng(B + M + K)
    raw, w, size = _q4k(rng, M, K)
    X = rng.normal(0, 1, (B, K)).astype(np.float32)
    A, Xd, Y = DB.from_array(raw), DB.from_array(X), DB((B * M + 64) * 4)
    Y.upload(np.full(B * M + 64, 7.0, np.float32))
    if form == "tiled":
        T = DB(hip.lib.slate_hip_q4k_tiled_bytes(M, K))
        check(hip.lib.slate_hip_q4k_tile(T.p, A.p, M, K), "q4k_tile")
        check(hip.lib.slate_hip_matmul_q4k_tiled(Y.p, T.p, Xd.p, B, M, K), "matmul_q4k_tiled")
    elif form == "row":
        check(hip.matmul_q4k(Y.p, A.p, Xd.p, B, M, K), "matmul_q4k")
    else:
        check(hip.lib.slate_hip_matmul_q4k_noalloc(Y.p, A.p, Xd.p, B, M, K), "matmul_q4k_noalloc")
    got = host(Y, (B * M + 64,))
    assert np.all(got[B * M:] == 7.0)
    X6 = X.astype(np.float64)
    # x and its sub-block sums as two f16 (2^-22 of the block's largest value,
    # 32 of them to a sum), then at most 24 roundings per 256-element block
    xmax = np.repeat(np.abs(X6).reshape(B, -1, 256).max(-1), 256, 1)
    bound = (K // 256 * 24 + 32) * EPS * (np.abs(X6) @ size.T) + 2.0 ** -21 * (xmax @ size.T)
    assert np.all(np.abs(got[:B * M].reshape(B, M) - X6 @ w.T) <= bound)


# 13-16 rows of a long matmul go over an operand, fewer through the converting
# kernel: at these shapes both add up the same values in the same splits, so
# a row's result has the same bits either way.
@pytest.mark.parametrize("M,K", [(14336, 4096), (18944, 3584), (13000, 4352)])
def test_q4k_rows_the_same_over_operand_and_conversion(hip, M, K):
    rng = np.random.default_rng(M + K)
    raw, _, _ = _q4k(rng, M, K)
    X = rng.normal(0, 1, (16, K)).astype(np.float32)
    A, Xd, Y = DB.from_array(raw), DB.from_array(X), DB(16 * M * 4)
    T = DB(hip.lib.slate_hip_q4k_tiled_bytes(M, K))
    check(hip.lib.slate_hip_q4k_tile(T.p, A.p, M, K), "q4k_tile")
    for fn, w in ((hip.lib.slate_hip_matmul_q4k, A), (hip.lib.slate_hip_matmul_q4k_tiled, T)):
        got = {}
        for B in (7, 12, 13, 16):
            check(fn(Y.p, w.p, Xd.p, B, M, K), "matmul_q4k")
            got[B] = host(Y, (16, M))[:B].view(np.uint32).copy()
        for B in (7, 12, 13):
            assert np.array_equal(got[B], got[16][:B]), B


# One row: x handed out through LDS (from 6M weights on) and loaded directly,
# with whole and partly filled waves of blocks, one and two passes over K, and
# the 16-row workgroups of long rows.
@pytest.mark.parametrize("M,K", [(1535, 4096), (1537, 4096), (6145, 1024), (6143, 1024), (3001, 2304), (455, 14336),
                                 (330, 19968), (25000, 256)])
def test_q4k_matvec_activation_paths(hip, M, K):
    rng = np.random.default_rng(M + K)
    raw, w, size = _q4k(rng, M, K)
    x = rng.normal(0, 1, K).astype(np.float32)
    y = DB((M + 16) * 4)
    y.upload(np.full(M + 16, 7.0, np.float32))
    hip.matvec_q4k(y.p, DB.from_array(raw).p, DB.from_array(x).p, M, K)
    check(0, "matvec_q4k")
    got = host(y, (M + 16,))
    assert np.all(got[M:] == 7.0)
    # per sub-block 16 products twice and the sum of 32 x, their scales, then
    # up to three passes, 4 + 32 sums: under 80 roundings of the absolute sum
    x6 = x.astype(np.float64)
    assert np.all(np.abs(got[:M] - w @ x6) <= 80 * EPS * (size @ np.abs(x6)))


@pytest.mark.parametrize("lens", [(100, 27), (101, 27), (64, 65), (1, 120, 3, 90)])
def test_prompt_steps_around_the_shared_row_factor(orc, lens):
    """Prompt steps of 127 rows (each consumer sums a row's squares itself), 128
    and more (one kernel does), the last rows alone normalised for the LM
    head; then a decode step.  Against the oracle token by token; 1e-4 is the
    bound between any two orders of the engine's sums in this suite."""
    t = make_llama(Q4, Q4_SEED, quant="q4k")
    m = slate_amd.Llama.from_tensors(Q4, t, max_slots=len(lens), max_tokens=sum(lens))
    om = OracleModel(orc, Q4, t)
    rng = np.random.default_rng(sum(lens))
    prompts = [rng.integers(0, Q4.vocab, n).astype(np.int32) for n in lens]
    ss = [m.session() for _ in lens]
    rc, lg, _ = m.step(ss, lens, np.concatenate(prompts))
    check(rc, "prompt step")
    rc, lg2, _ = m.step(ss, [1] * len(lens), np.full(len(lens), 5, np.int32))
    check(rc, "decode step")
    for i, p in enumerate(prompts):
        o = om.session()
        _, want = o.prefill(p)
        assert relerr(lg[i], want) < 1e-4, i
        _, want = o.decode(5)
        assert relerr(lg2[i], want) < 1e-4, i


def _ragged_case(rng, order):
    """(sequence, position) per token: runs of several lengths around the
    units of 16 / G tokens and the chunks of 256 keys, joined, broken, or in
    an order in which hardly any token follows another."""
    runs = [(0, 0, 33), (1, 250, 9), (2, 0, 1), (2, 1, 4), (3, 511, 2), (4, 700, 17), (0, 33, 2), (5, 3, 1)]
    tok = [(s, p0 + i) for s, p0, n in runs for i in range(n)]
    tok += [(6, 40), (6, 40), (6, 39), (6, 38)]             # repeated and falling positions
    if order == "shuffled":
        tok = [tok[i] for i in rng.permutation(len(tok))]
    elif order == "reversed":
        tok = tok[::-1]
    elif order == "long":                                   # runs over the list kernel's 1024 entries
        tok = tok + [(7, i) for i in range(720)] + [(4, i) for i in range(250)] + [(1, 5)]
    return tok


@pytest.mark.parametrize("hd,Hq,Hkv,order", [(128, 8, 2, "joined"), (128, 2, 2, "joined"), (128, 8, 1, "shuffled"),
                                             (64, 4, 2, "joined"), (64, 8, 2, "reversed"), (32, 8, 8, "joined"),
                                             (32, 16, 2, "long"), (32, 3, 3, "long"), (64, 24, 3, "joined")])
def test_attention_runs(hip, hd, Hq, Hkv, order):
    """More than 64 query tokens: runs share their K/V rows, whatever order
    the tokens come in.  Every cache row that no token may see is NaN."""
    rng = np.random.default_rng(hd * Hq + len(order))
    S, nslot = 768, 8
    tok = _ragged_case(rng, order)
    T = len(tok)
    seq = np.array([s for s, _ in tok], np.int32)
    pos = np.array([p for _, p in tok], np.int32)
    last = [max([p for s, p in tok if s == b], default=-1) for b in range(nslot)]
    K = rng.normal(0, 1, (nslot, Hkv, S, hd)).astype(np.float32)
    V = rng.normal(0, 1, (nslot, Hkv, S, hd)).astype(np.float32)
    for b in range(nslot):
        K[b, :, last[b] + 1:] = np.nan
        V[b, :, last[b] + 1:] = np.nan
    base = np.arange(nslot, dtype=np.int64)[::-1] * (Hkv * S * hd)
    q = rng.normal(0, 1, (T, Hq, hd)).astype(np.float32)

    def call(Kc, Vc):
        out = DB((T * Hq * hd + 64) * 4)
        out.upload(np.full(T * Hq * hd + 64, 7.0, np.float32))
        check(hip.lib.slate_hip_attention_ragged(
            out.p, DB.from_array(q).p, DB.from_array(Kc[::-1].copy()).p, DB.from_array(Vc[::-1].copy()).p,
            DB.from_array(seq).p, DB.from_array(pos).p, DB.from_array(base.copy()).p, T, Hq, Hkv, hd, S * hd, S),
            "attention_ragged")
        got = host(out, (T * Hq * hd + 64,))
        assert np.all(got[T * Hq * hd:] == 7.0)
        return got[:T * Hq * hd].reshape(T, Hq, hd)

    got = call(K, V)
    G = Hq // Hkv
    q6, K6, V6 = q.astype(np.float64), K.astype(np.float64), V.astype(np.float64)
    for t in range(T):
        L = pos[t] + 1
        k, v = K6[seq[t], :, :L].repeat(G, 0), V6[seq[t], :, :L].repeat(G, 0)
        s = np.einsum("hd,hld->hl", q6[t], k) / np.sqrt(hd)
        mag = np.einsum("hd,hld->hl", np.abs(q6[t]), np.abs(k)).max() / np.sqrt(hd)
        p = np.exp(s - s.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        # a score is hd products and sums; its error moves a weight by that
        # much twice (numerator and sum); then at most 256 + 64 roundings
        bound = (2 * (hd + 8) * EPS * mag + (min(L, 256) + 64) * EPS) * np.einsum("hl,hld->hd", p, np.abs(v))
        assert np.all(np.abs(got[t] - np.einsum("hl,hld->hd", p, v)) <= bound), (t, tok[t])

    # an infinite V row reaches the tokens that see it and no others, with
    # every other token's bits as they were but for the order of its sums
    V[1, :, 255] = np.inf
    V[0, :, 17, 3] = np.nan
    again = call(K, V)
    for t in range(T):
        if seq[t] == 1 and pos[t] >= 255:
            assert not np.any(np.isfinite(again[t])), (t, tok[t])
        elif seq[t] == 0 and pos[t] >= 17:
            assert np.all(np.isnan(again[t][:, 3])) and np.all(np.isfinite(np.delete(again[t], 3, -1)))
        else:
            # (the last tokens of a run take the exact path of their unit)
            assert np.allclose(again[t], got[t], rtol=0, atol=64 * EPS * 8), (t, tok[t])


def _check_attention(hip, rng, tok, hd, Hq, Hkv, stride, offs, off=(0, 0, 0)):
    """attention_ragged of tokens (sequence, position) against float64: kv
    heads `stride` floats apart, sequence b's base offs[b] floats off, the
    pointers of q, K and V off[i] floats off 16 bytes."""
    S, nslot, T = 768, len(offs), len(tok)
    seq = np.array([s for s, _ in tok], np.int32)
    pos = np.array([p for _, p in tok], np.int32)
    base = np.arange(nslot, dtype=np.int64) * (Hkv * stride + 4) + np.array(offs)
    pool = int(base[-1]) + Hkv * stride + 4
    K, V = (rng.normal(0, 1, pool).astype(np.float32) for _ in range(2))
    q = rng.normal(0, 1, (T, Hq, hd)).astype(np.float32)
    bufs = []
    for a, o in zip((q, K, V), off):
        bufs.append(DB((a.size + 4) * 4))
        bufs[-1].upload(np.concatenate([np.zeros(o, np.float32), a.reshape(-1), np.zeros(4 - o, np.float32)]))
    out = DB((T * Hq * hd + 64) * 4)
    out.upload(np.full(T * Hq * hd + 64, 7.0, np.float32))
    check(hip.lib.slate_hip_attention_ragged(
        out.p, *[b.ptr + 4 * o for b, o in zip(bufs, off)], DB.from_array(seq).p, DB.from_array(pos).p,
        DB.from_array(base).p, T, Hq, Hkv, hd, stride, S), "attention_ragged")
    got = host(out, (T * Hq * hd + 64,))
    assert np.all(got[T * Hq * hd:] == 7.0)
    got = got[:T * Hq * hd].reshape(T, Hkv, Hq // Hkv, hd)
    q6 = q.astype(np.float64).reshape(got.shape)
    for t in range(T):
        L = pos[t] + 1
        for h in range(Hkv):
            b = int(base[seq[t]]) + h * stride
            k, v = (a[b:b + L * hd].astype(np.float64).reshape(L, hd) for a in (K, V))
            s = q6[t, h] @ k.T / np.sqrt(hd)
            mag = (np.abs(q6[t, h]) @ np.abs(k).T).max() / np.sqrt(hd)
            p = np.exp(s - s.max(-1, keepdims=True))
            p /= p.sum(-1, keepdims=True)
            # (the bound of test_attention_runs)
            bound = (2 * (hd + 8) * EPS * mag + (min(L, 256) + 64) * EPS) * (p @ np.abs(v))
            assert np.all(np.abs(got[t, h] - p @ v) <= bound), (t, tok[t], h)


# More than 64 tokens: rows that start on 16 bytes only in some sequences
# (kv_base takes any offset), and q, K, V or the heads off 16 bytes.
@pytest.mark.parametrize("hd,Hq,Hkv", [(128, 8, 2), (64, 8, 8), (32, 8, 1)])
@pytest.mark.parametrize("form", ["base", "q", "K", "V", "stride"])
def test_attention_of_unaligned_rows(hip, hd, Hq, Hkv, form):
    offs = (1, 0, 3, 0, 2, 0, 1) if form == "base" else (0,) * 7
    off = {"q": (1, 0, 0), "K": (0, 3, 0), "V": (0, 0, 2)}.get(form, (0, 0, 0))
    _check_attention(hip, np.random.default_rng(hd + len(form)), _ragged_case(None, "joined"), hd, Hq, Hkv,
                     768 * hd + (1 if form == "stride" else 0), offs, off)


# More than 64 tokens that hardly share keys (each workgroup of the token kernel
# numbers them for itself) and calls of several passes of 1024 tokens: all
# alone, short and long; alone but for a pair; a pass alone, then runs that
# begin before the pass does and end in it; an unaligned sequence in one pass.
@pytest.mark.parametrize("hd,Hq,Hkv", [(128, 4, 1), (128, 2, 2), (64, 8, 1), (32, 6, 3)])
@pytest.mark.parametrize("form", ["short", "long", "pair", "passes", "unaligned pass"])
def test_attention_of_lone_tokens(hip, hd, Hq, Hkv, form):
    rng = np.random.default_rng(hd * Hq + len(form))
    offs = [0] * 7
    tok = [(i % 6, int(p)) for i, p in enumerate(rng.integers(0, 700 if form == "long" else 90, 65))]
    if form == "pair":
        tok += [(6, 255), (6, 256)]
    if form in ("passes", "unaligned pass"):
        tok = [(i % 6, (37 * i) % 41) for i in range(1020)] + [(6, i) for i in range(200)]
        tok += [(i % 3, 700 - i) for i in range(700)] + [(4, i) for i in range(228)]
    if form == "unaligned pass":
        offs[2] = 3
        tok = tok[:1024] + [(6, 4 + i) for i in range(300)]
    _check_attention(hip, rng, tok, hd, Hq, Hkv, 768 * hd, tuple(offs))
