"""Measured cases: what a program that serves LLaMA models through this
library asks of it, from single entry points of the C ABI up to steps of the
device engine.

Kinds of cases:

  q4k      one Q4_K matmul, Y = X W^T (matvec_q4k / matmul_q4k on slate's
           row layout, matmul_q4k_tiled on weights regrouped once at load)
  q8       one Q8_0 matmul (q8_0_matvec / matmul_q8_0 / matmul_q8_0_tiled)
  linear   one f32 linear layer, C = X W (linear_batch, the toy engine's)
  layer    one token through one decoder layer, one entry at a time, as an
           engine that knows only the backend's entries runs it
  attn     ragged GQA attention of decode tokens and prompt chunks
  head     final norm, LM head and greedy argmax of a batch
  engine   the device engine: fresh sessions take their prompts in one
           ragged step, then decode together

Weights are N(0, 0.02) quantised to their format, activations N(0, 1).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import slate_amd
from slate_amd.synth import LlamaShape

DEV = "cuda"
EPS = 1e-5
THETA = 10000.0
STD = 0.02


def _lib():
    slate_amd.Backend()                      # raises where there is no device
    return slate_amd.load_library()


def _ok(rc, what):
    if rc:
        slate_amd.check(rc, what)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32) * std


def _ready(state):
    torch.cuda.synchronize()                 # inputs are complete before the backend's stream reads them
    return state


# -- weights ------------------------------------------------------------------
def _q4k_row(lib, M, K, seed):
    w = torch.empty(M * (K // 256) * 144, dtype=torch.uint8, device=DEV)
    _ok(lib.slate_hip_synth_q4k(w.data_ptr(), M, K, seed, STD), "synth_q4k")
    return w


def _q4k_tile(lib, row, M, K):
    t = torch.empty(lib.slate_hip_q4k_tiled_bytes(M, K), dtype=torch.uint8, device=DEV)
    _ok(lib.slate_hip_q4k_tile(t.data_ptr(), row.data_ptr(), M, K), "q4k_tile")
    return t


def _q4k_dense(raw, M, K):
    """Q4_K bytes in slate's row layout as [M, K] float64."""
    b = raw.view(M * (K // 256), 144)
    head = b[:, :4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].to(torch.int32)
    lo, hi, mix = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([lo & 63, (mix & 15) | ((lo >> 6) << 4)], 1).double()
    mn = torch.cat([hi & 63, (mix >> 4) | ((hi >> 6) << 4)], 1).double()
    q = b[:, 16:].reshape(-1, 8, 16)
    q = torch.cat([q & 15, q >> 4], 2).double()
    return ((head[:, 0:1] * sc).unsqueeze(2) * q - (head[:, 1:2] * mn).unsqueeze(2)).reshape(M, K)


def _q8_row(g, M, K):
    """Q8_0 bytes of N(0, STD) weights: 34-byte blocks of f16 d and 32 int8."""
    w = _normal(g, M * (K // 32), 32, std=STD)
    d = (w.abs().amax(1, keepdim=True) / 127.0).half()
    q = torch.where(d > 0, torch.round(w / d.float()), torch.zeros_like(w)).clamp(-127, 127).to(torch.int8)
    return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], 1).reshape(-1)


def _q8_dense(raw, M, K):
    b = raw.view(M * (K // 32), 34)
    return (b[:, :2].contiguous().view(torch.float16).double() *
            b[:, 2:].contiguous().view(torch.int8).double()).reshape(M, K)


# -- one quantised matmul -----------------------------------------------------
def _mm_prepare(c, seed):
    lib, g = _lib(), _gen(seed)
    B, M, K = c["B"], c["M"], c["K"]
    st = {"lib": lib, "B": B, "M": M, "K": K, "X": _normal(g, B, K), "Y": torch.empty(B, M, device=DEV)}
    if c["kind"] == "q4k":
        st["row"] = _q4k_row(lib, M, K, seed)
        st["W"] = _q4k_tile(lib, st["row"], M, K) if c["tiled"] else st["row"]
        st["fn"] = lib.slate_hip_matmul_q4k_tiled if c["tiled"] else lib.slate_hip_matmul_q4k
        st["vec"] = lib.slate_hip_matvec_q4k
    else:
        st["row"] = st["W"] = _q8_row(g, M, K)
        if c["tiled"]:
            st["W"] = torch.empty(lib.slate_hip_q8_0_tiled_bytes(M, K), dtype=torch.uint8, device=DEV)
            torch.cuda.synchronize()
            _ok(lib.slate_hip_q8_0_tile(st["W"].data_ptr(), st["row"].data_ptr(), M, K), "q8_0_tile")
        st["fn"] = lib.slate_hip_matmul_q8_0_tiled if c["tiled"] else lib.slate_hip_matmul_q8_0
        st["vec"] = lib.slate_hip_q8_0_matvec
    st["is_vec"] = B == 1 and not c["tiled"]
    return _ready(st)


def _mm_run(st):
    y, w, x = st["Y"].data_ptr(), st["W"].data_ptr(), st["X"].data_ptr()
    if st["is_vec"]:
        st["vec"](y, w, x, st["M"], st["K"])
    else:
        _ok(st["fn"](y, w, x, st["B"], st["M"], st["K"]), "matmul")
    return st["Y"]


def _mm_exact(c, seed):
    st = _mm_prepare(c, seed)
    dense = _q4k_dense if c["kind"] == "q4k" else _q8_dense
    return st["X"].double() @ dense(st["row"], c["M"], c["K"]).t().contiguous()


def _mm_work(c):
    B, M, K = c["B"], c["M"], c["K"]
    w = M * K * (144 / 256 if c["kind"] == "q4k" else 34 / 32)
    return {"bytes": w + 4 * B * (M + K), "flops": 2 * B * M * K}


# -- f32 linear layer ---------------------------------------------------------
def _lin_prepare(c, seed):
    g = _gen(seed)
    return _ready({"lib": _lib(), "c": c, "X": _normal(g, c["B"], c["K"]), "W": _normal(g, c["K"], c["N"], std=STD),
                   "C": torch.empty(c["B"], c["N"], device=DEV)})


def _lin_run(st):
    c = st["c"]
    st["lib"].slate_hip_linear_batch(st["C"].data_ptr(), st["X"].data_ptr(), st["W"].data_ptr(), c["B"], c["K"], c["N"])
    return st["C"]


def _lin_exact(c, seed):
    st = _lin_prepare(c, seed)
    return st["X"].double() @ st["W"].double()


def _lin_work(c):
    B, K, N = c["B"], c["K"], c["N"]
    return {"bytes": 4 * (B * K + K * N + B * N), "flops": 2 * B * K * N}


# -- one token through one decoder layer --------------------------------------
def _layer_dims(c):
    D, hd = c["d"], c["hd"]
    return D, c["heads"], c["kv_heads"], hd, c["kv_heads"] * hd, c["ffn"], c["ctx"]


def _layer_prepare(c, seed):
    lib, g = _lib(), _gen(seed)
    D, Hq, Hkv, hd, kvd, F, L = _layer_dims(c)
    shapes = {"q": (D, D), "k": (kvd, D), "v": (kvd, D), "o": (D, D), "gate": (F, D), "up": (F, D), "down": (D, F)}
    st = {"lib": lib, "c": c, "shapes": shapes}
    for i, (n, (m, k)) in enumerate(shapes.items()):
        st["w_" + n] = _q4k_row(lib, m, k, seed * 8 + i)
        st["y_" + n] = torch.empty(m, device=DEV)
    st["embd"] = _normal(g, 256, D)
    st["token"] = seed % 256
    st["n1"] = 1 + _normal(g, D, std=0.1)
    st["n2"] = 1 + _normal(g, D, std=0.1)
    for n, w in (("x", D), ("xn", D), ("att", D), ("h", F)):
        st[n] = torch.empty(w, device=DEV)
    st["K"] = _normal(g, Hkv, L, hd)
    st["V"] = _normal(g, Hkv, L, hd)
    st["pos"] = torch.tensor([L - 1], dtype=torch.int32, device=DEV)
    st["seq"] = torch.zeros(1, dtype=torch.int32, device=DEV)
    st["base"] = torch.zeros(1, dtype=torch.int64, device=DEV)
    st["p"] = {n: t.data_ptr() for n, t in st.items() if isinstance(t, torch.Tensor)}
    return _ready(st)


def _layer_run(st):
    lib, p = st["lib"], st["p"]
    D, Hq, Hkv, hd, kvd, F, L = _layer_dims(st["c"])
    mv = lib.slate_hip_matvec_q4k
    lib.slate_hip_embed_lookup(p["x"], p["embd"], st["token"], D)
    lib.slate_hip_rmsnorm_row(p["xn"], p["x"], p["n1"], D, EPS)
    mv(p["y_q"], p["w_q"], p["xn"], D, D)
    mv(p["y_k"], p["w_k"], p["xn"], kvd, D)
    mv(p["y_v"], p["w_v"], p["xn"], kvd, D)
    _ok(lib.slate_hip_rope_rows(p["y_q"], p["pos"], 1, Hq, hd, THETA, L), "rope_rows")
    _ok(lib.slate_hip_rope_rows(p["y_k"], p["pos"], 1, Hkv, hd, THETA, L), "rope_rows")
    _ok(lib.slate_hip_attention_ragged(p["att"], p["y_q"], p["K"], p["V"], p["seq"], p["pos"], p["base"], 1, Hq, Hkv,
                                       hd, L * hd, L), "attention_ragged")
    mv(p["y_o"], p["w_o"], p["att"], D, D)
    lib.slate_hip_add_inplace(p["x"], p["y_o"], D)
    lib.slate_hip_rmsnorm_row(p["xn"], p["x"], p["n2"], D, EPS)
    mv(p["y_gate"], p["w_gate"], p["xn"], F, D)
    mv(p["y_up"], p["w_up"], p["xn"], F, D)
    lib.slate_hip_silu_mul(p["h"], p["y_gate"], p["y_up"], F)
    mv(p["y_down"], p["w_down"], p["h"], D, F)
    lib.slate_hip_add_inplace(p["x"], p["y_down"], D)
    return {"x": st["x"], "k": st["y_k"], "v": st["y_v"], "att": st["att"]}


def _rope(x, pos):
    """x [..., heads, hd] f64 rotated at pos [...]; the angles are f32, as the model defines them."""
    hd = x.shape[-1]
    i = np.arange(hd // 2, dtype=np.float32)
    inv = np.power(float(np.float32(THETA)), (np.float32(-2.0) * i / np.float32(hd)).astype(np.float64)).astype(np.float32)
    ang = torch.from_numpy(np.asarray(pos, np.float32)[..., None] * inv).double().to(x.device)
    c, s = ang.cos().unsqueeze(-2), ang.sin().unsqueeze(-2)
    a, b = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _norm(x, w):
    return x * w / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _silu(g):
    return g / (1 + torch.exp(-g))


def _attend(q, K, V, p0):
    """q [n, Hq, hd] at positions p0.., K/V [Hkv, L, hd], f64 -> [n, Hq, hd]."""
    n, Hq, hd = q.shape
    Hkv = K.shape[0]
    G = Hq // Hkv
    L = p0 + n
    qs = q.reshape(n, Hkv, G, hd).permute(1, 0, 2, 3).reshape(Hkv, n * G, hd).contiguous()
    s = torch.matmul(qs, K[:, :L].transpose(1, 2).contiguous()) / math.sqrt(hd)
    if n > 1:
        last = torch.arange(p0, L, device=q.device).repeat_interleave(G)
        s = s.masked_fill(torch.arange(L, device=q.device)[None] > last[:, None], -math.inf)
    o = torch.matmul(torch.softmax(s, -1), V[:, :L].contiguous())
    return o.reshape(Hkv, n, G, hd).permute(1, 0, 2, 3).reshape(n, Hq, hd)


def _layer_exact(c, seed):
    st = _layer_prepare(c, seed)
    D, Hq, Hkv, hd, kvd, F, L = _layer_dims(c)
    w = {n: _q4k_dense(st["w_" + n], *s) for n, s in st["shapes"].items()}
    x = st["embd"][st["token"]].double()
    xn = _norm(x, st["n1"].double())
    q = _rope((w["q"] @ xn).reshape(1, Hq, hd), [L - 1])
    k = _rope((w["k"] @ xn).reshape(1, Hkv, hd), [L - 1])
    v = w["v"] @ xn
    att = _attend(q, st["K"].double(), st["V"].double(), L - 1).reshape(D)
    x = x + w["o"] @ att
    xn = _norm(x, st["n2"].double())
    x = x + w["down"] @ (_silu(w["gate"] @ xn) * (w["up"] @ xn))
    return {"x": x, "k": k.reshape(-1), "v": v, "att": att}


def _layer_work(c):
    D, Hq, Hkv, hd, kvd, F, L = _layer_dims(c)
    n = 2 * D * D + 2 * kvd * D + 3 * D * F
    return {"bytes": n * 144 / 256 + 8 * L * kvd + 4 * (4 * D + 2 * kvd), "flops": 2 * n + 4 * L * Hq * hd}


# -- ragged attention ---------------------------------------------------------
def _attn_batch(c):
    """Per sequence: positions already cached and new tokens.  Decode tokens
    come first, then the prompt chunks; contexts are log-normal around
    `ctx`, chunk lengths within a factor of two below `chunk` (lengths belong
    to the case, values to the seed)."""
    r = np.random.default_rng(c["ctx"])
    n_dec, n_pre = c["decode"], c["chunks"]
    ctx = np.clip(np.exp(r.normal(math.log(c["ctx"]), 0.8, n_dec + n_pre)), 16, c["max_pos"] - c["chunk"]).astype(int)
    n_new = [1] * n_dec + [int(v) for v in r.integers((c["chunk"] + 1) // 2, c["chunk"] + 1, n_pre)]
    p0 = [int(v) for v in ctx[:n_dec]] + [int(v) * (i % 2) for i, v in enumerate(ctx[n_dec:])]
    return p0, n_new


def _attn_prepare(c, seed):
    g = _gen(seed)
    Hq, Hkv, hd, S = c["heads"], c["kv_heads"], c["hd"], c["max_pos"]
    p0, n_new = _attn_batch(c)
    n, T = len(p0), sum(n_new)
    i32 = dict(dtype=torch.int32, device=DEV)
    seq = [i for i in range(n) for _ in range(n_new[i])]
    pos = [p0[i] + j for i in range(n) for j in range(n_new[i])]
    return _ready({"lib": _lib(), "c": c, "T": T, "p0": p0, "n_new": n_new, "q": _normal(g, T, Hq, hd),
                   "K": _normal(g, n, Hkv, S, hd), "V": _normal(g, n, Hkv, S, hd),
                   "seq": torch.tensor(seq, **i32), "pos": torch.tensor(pos, **i32),
                   "base": torch.arange(n, dtype=torch.int64, device=DEV) * (Hkv * S * hd),
                   "out": torch.empty(T, Hq, hd, device=DEV)})


def _attn_run(st):
    c = st["c"]
    _ok(st["lib"].slate_hip_attention_ragged(
        st["out"].data_ptr(), st["q"].data_ptr(), st["K"].data_ptr(), st["V"].data_ptr(), st["seq"].data_ptr(),
        st["pos"].data_ptr(), st["base"].data_ptr(), st["T"], c["heads"], c["kv_heads"], c["hd"],
        c["max_pos"] * c["hd"], c["max_pos"]), "attention_ragged")
    return st["out"]


def _attn_exact(c, seed):
    st = _attn_prepare(c, seed)
    out, t = [], 0
    for i, (p, n) in enumerate(zip(st["p0"], st["n_new"])):
        L = p + n
        out.append(_attend(st["q"][t:t + n].double(), st["K"][i, :, :L].double(), st["V"][i, :, :L].double(), p))
        t += n
    return torch.cat(out)


def _attn_work(c):
    p0, n_new = _attn_batch(c)
    kv = c["kv_heads"] * c["hd"]
    D = c["heads"] * c["hd"]
    keys = sum(p + n for p, n in zip(p0, n_new))
    pairs = sum(n * p + n * (n + 1) // 2 for p, n in zip(p0, n_new))
    return {"bytes": 8 * keys * kv + 8 * sum(n_new) * D, "flops": 4 * pairs * D}


# -- final norm, LM head, greedy argmax ---------------------------------------
def _head_prepare(c, seed):
    lib, g = _lib(), _gen(seed)
    B, D, V = c["B"], c["d"], c["vocab"]
    row = _q4k_row(lib, V, D, seed)
    return _ready({"lib": lib, "c": c, "row": row, "W": _q4k_tile(lib, row, V, D), "x": _normal(g, B, D),
                   "n": 1 + _normal(g, D, std=0.1), "xn": torch.empty(B, D, device=DEV),
                   "logits": torch.empty(B, V, device=DEV), "next": torch.empty(B, dtype=torch.int32, device=DEV)})


def _head_run(st):
    lib, c = st["lib"], st["c"]
    B, D, V = c["B"], c["d"], c["vocab"]
    xn, lg = st["xn"].data_ptr(), st["logits"].data_ptr()
    _ok(lib.slate_hip_rmsnorm_rows(xn, st["x"].data_ptr(), st["n"].data_ptr(), B, D, EPS), "rmsnorm_rows")
    _ok(lib.slate_hip_matmul_q4k_tiled(lg, st["W"].data_ptr(), xn, B, V, D), "matmul_q4k_tiled")
    _ok(lib.slate_hip_argmax_rows(st["next"].data_ptr(), lg, B, V), "argmax_rows")
    return {"logits": st["logits"], "next": st["next"]}


def _head_exact(c, seed):
    st = _head_prepare(c, seed)
    xn = _norm(st["x"].double(), st["n"].double())
    return {"logits": xn @ _q4k_dense(st["row"], c["vocab"], c["d"]).t().contiguous(), "next": None}


def _head_work(c):
    B, D, V = c["B"], c["d"], c["vocab"]
    return {"bytes": V * D * 144 / 256 + 4 * B * (D + V) + 4 * D, "flops": 2 * B * D * V}


# -- the device engine --------------------------------------------------------
def _engine_shape(c):
    longest = c["prompt"] + c["steps"] + 1
    return LlamaShape(n_layers=c["layers"], d_model=c["d"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                      ffn=c["ffn"], vocab=c["vocab"], max_seq=(longest + 255) // 256 * 256)


def _engine_tokens(c, seed):
    lens = np.random.default_rng(c["prompt"]).integers((c["prompt"] + 3) // 4, c["prompt"] + 1, c["seqs"])
    r = np.random.default_rng(seed)
    prompts = [r.integers(0, c["vocab"], n).astype(np.int32) for n in lens]
    return prompts, r.integers(0, c["vocab"], (c["steps"], c["seqs"])).astype(np.int32)


def _engine_prepare(c, seed):
    _lib()
    prompts, cont = _engine_tokens(c, seed)
    m = slate_amd.Llama.synthetic(_engine_shape(c), seed, c["quant"], max_slots=c["seqs"],
                                  max_tokens=max(16, sum(len(p) for p in prompts)))
    return _ready({"m": m, "sessions": [m.session() for _ in prompts], "n_new": [len(p) for p in prompts],
                   "packed": np.concatenate(prompts), "cont": cont, "one": [1] * len(prompts)})


def _engine_run(st):
    m, ss = st["m"], st["sessions"]
    for s in ss:
        m.lib.slate_hip_llama_session_reset(s.h)
    rc, first, _ = m.step(ss, st["n_new"], st["packed"])
    _ok(rc, "llama_step")
    last = None
    for i, toks in enumerate(st["cont"]):
        end = i + 1 == len(st["cont"])       # a greedy program asks for logits only where it looks at them
        rc, last, _ = m.step(ss, st["one"], toks, want_logits=end)
        _ok(rc, "llama_step")
    return {"prompt": first} if last is None else {"prompt": first, "decode": last}


def _engine_exact(c, seed):
    st = _engine_prepare(c, seed)
    m, s = st["m"], _engine_shape(c)
    D, hd, kvd = s.d_model, s.head_dim, s.kv_dim
    prompts, cont = _engine_tokens(c, seed)

    def get(name, rows, cols):
        raw, dt = m.get_tensor(name)
        t = torch.from_numpy(raw).to(DEV)
        return {0: lambda: t.view(torch.float32).double().reshape(rows, cols), 16: lambda: _q8_dense(t, rows, cols),
                18: lambda: _q4k_dense(t, rows, cols)}[dt]()

    seqs = [np.concatenate([p, cont[:, i]]) for i, p in enumerate(prompts)]
    ends = np.cumsum([len(t) for t in seqs])
    emb = get("token_embd", s.vocab, D)
    x = emb[torch.from_numpy(np.concatenate(seqs).astype(np.int64)).to(DEV)]
    del emb
    pos = np.concatenate([np.arange(len(t)) for t in seqs])
    for i in range(s.n_layers):
        w = lambda n, r, k: get("blk.%d.%s" % (i, n), r, k).t().contiguous()  # noqa: E731
        xn = _norm(x, get("blk.%d.attn_norm" % i, 1, D))
        q = _rope((xn @ w("attn_q", D, D)).reshape(-1, s.n_heads, hd), pos)
        k = _rope((xn @ w("attn_k", kvd, D)).reshape(-1, s.n_kv_heads, hd), pos)
        v = (xn @ w("attn_v", kvd, D)).reshape(-1, s.n_kv_heads, hd)
        att = []
        for e, t in zip(ends, seqs):
            a = e - len(t)
            att.append(_attend(q[a:e], k[a:e].transpose(0, 1).contiguous(), v[a:e].transpose(0, 1).contiguous(), 0))
        x = x + torch.cat(att).reshape(-1, D) @ w("attn_output", D, D)
        xn = _norm(x, get("blk.%d.ffn_norm" % i, 1, D))
        x = x + (_silu(xn @ w("ffn_gate", s.ffn, D)) * (xn @ w("ffn_up", s.ffn, D))) @ w("ffn_down", D, s.ffn)
    x = _norm(x, get("output_norm", 1, D))
    wo = get("output", s.vocab, D).t().contiguous()
    starts = np.concatenate([[0], ends[:-1]])
    pr = x[torch.from_numpy(starts + [len(p) - 1 for p in prompts]).to(DEV)] @ wo
    if not len(cont):
        return {"prompt": pr}
    return {"prompt": pr, "decode": x[torch.from_numpy(ends - 1).to(DEV)] @ wo}


def _engine_work(c):
    s = _engine_shape(c)
    prompts, cont = _engine_tokens(c, 1)
    D, kvd, B, n = s.d_model, s.kv_dim, len(prompts), c["steps"]
    per = 2 * D * D + 2 * kvd * D + 3 * D * s.ffn
    wb = {18: 144 / 256, 16: 34 / 32, 0: 4}[c["quant"]]
    pt = sum(len(p) for p in prompts)
    rows = pt + B * n                                    # tokens through the layers
    kv = sum(len(p) for p in prompts) + sum(len(p) + j + 1 for p in prompts for j in range(n))
    pairs = sum(len(p) * (len(p) + 1) // 2 for p in prompts) + sum(len(p) + j + 1 for p in prompts for j in range(n))
    return {"bytes": (1 + n) * wb * (s.n_layers * per + s.vocab * D) + 8 * s.n_layers * kvd * kv +
                     4 * rows * D + 4 * 2 * B * s.vocab,
            "flops": 2 * rows * s.n_layers * per + 2 * B * (1 + n) * s.vocab * D + 4 * s.n_layers * pairs * D}


# -----------------------------------------------------------------------------
_KINDS = {
    "q4k": (_mm_prepare, _mm_run, _mm_exact, _mm_work),
    "q8": (_mm_prepare, _mm_run, _mm_exact, _mm_work),
    "linear": (_lin_prepare, _lin_run, _lin_exact, _lin_work),
    "layer": (_layer_prepare, _layer_run, _layer_exact, _layer_work),
    "attn": (_attn_prepare, _attn_run, _attn_exact, _attn_work),
    "head": (_head_prepare, _head_run, _head_exact, _head_work),
    "engine": (_engine_prepare, _engine_run, _engine_exact, _engine_work),
}

# Relative errors that a correct implementation with f32 sums shows: about four
# times the largest that the kinds show against 64 bits (4.3e-7 for the matmuls,
# 2.5e-7 for attention, 6.3e-7 for a layer, 2.4e-6 for the engine's logits).
_REL = {"q4k": 2e-6, "q8": 2e-6, "linear": 2e-6, "layer": 3e-6, "attn": 1e-6, "head": 2e-6, "engine": 1e-5}


def listed():
    return [
        # one token of one sequence through one attention projection: slate's matvec_q4k on the bytes of the file
        {"name": "q4k matvec", "kind": "q4k", "B": 1, "M": 4096, "K": 4096, "tiled": False},
        # a decode batch through an FFN projection, weights as loaded
        {"name": "q4k batch 16", "kind": "q4k", "B": 16, "M": 14336, "K": 4096, "tiled": False},
        # an arriving prompt through the down projection, weights regrouped at load
        {"name": "q4k prompt 301", "kind": "q4k", "B": 301, "M": 4096, "K": 14336, "tiled": True},
        # the same for models stored as Q8_0: one token on the bytes of the file, a batch on regrouped weights
        {"name": "q8 matvec", "kind": "q8", "B": 1, "M": 4096, "K": 4096, "tiled": False},
        {"name": "q8 batch 16", "kind": "q8", "B": 16, "M": 14336, "K": 4096, "tiled": True},
        # the toy engine's f32 head (vocabulary 4096) and FFN at a batch of 16
        {"name": "f32 linear 16", "kind": "linear", "B": 16, "K": 1024, "N": 4096},
        # one token through an 8B layer by the backend's entries, as slate's own decode loop calls them
        {"name": "vtable layer", "kind": "layer", "d": 4096, "heads": 32, "kv_heads": 8, "hd": 128, "ffn": 14336,
         "ctx": 1000},
        # decode attention of 64 sequences with long-tailed contexts
        {"name": "attn decode 64", "kind": "attn", "heads": 32, "kv_heads": 8, "hd": 128, "decode": 64, "chunks": 0,
         "chunk": 1, "ctx": 1024, "max_pos": 16384},
        # a step's attention with prompt chunks beside decode tokens
        {"name": "attn chunks", "kind": "attn", "heads": 32, "kv_heads": 8, "hd": 128, "decode": 13, "chunks": 3,
         "chunk": 200, "ctx": 700, "max_pos": 4096},
        # the end of a decode step: final norm, LM head, greedy token
        {"name": "head 16", "kind": "head", "B": 16, "d": 4096, "vocab": 128256},
        # continuous batching: 16 sequences take short prompts, then decode together
        {"name": "engine decode", "kind": "engine", "layers": 2, "d": 4096, "heads": 32, "kv_heads": 8, "ffn": 14336,
         "vocab": 32000, "quant": 18, "seqs": 16, "prompt": 40, "steps": 16},
        # prompts of up to 512 tokens prefilled in one ragged step
        {"name": "engine prefill", "kind": "engine", "layers": 2, "d": 4096, "heads": 32, "kv_heads": 8, "ffn": 14336,
         "vocab": 32000, "quant": 18, "seqs": 6, "prompt": 512, "steps": 0},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(sorted(_KINDS))
    if kind in ("q4k", "q8"):
        one = rng.random() < 0.3
        unit = 256 if kind == "q4k" else 32
        return {"kind": kind, "B": 1 if one else _log(rng, 2, 400 if kind == "q4k" else 64), "M": _log(rng, 256, 14336),
                "K": unit * _log(rng, 256 // unit, 14336 // unit), "tiled": rng.random() < 0.5}
    if kind == "linear":
        return {"kind": kind, "B": _log(rng, 1, 64), "K": _log(rng, 64, 4096), "N": _log(rng, 64, 8192)}
    # head counts and sizes as the models of this family have them
    heads, kv, hd = rng.choice([(32, 8, 128), (32, 32, 128), (16, 4, 64), (32, 4, 64), (16, 8, 128), (64, 8, 128)])
    if kind == "layer":
        heads, kv, hd = rng.choice([(32, 8, 128), (32, 32, 128), (16, 4, 64), (16, 8, 128)])
        return {"kind": kind, "d": heads * hd, "heads": heads, "kv_heads": kv, "hd": hd, "ffn": 256 * _log(rng, 8, 56),
                "ctx": _log(rng, 16, 8000)}
    if kind == "attn":
        chunks = rng.choice([0, 0, 1, 2, 4])
        dec = _log(rng, 1, 64) if chunks == 0 or rng.random() < 0.7 else 0
        return {"kind": kind, "heads": heads, "kv_heads": kv, "hd": hd, "decode": dec, "chunks": chunks,
                "chunk": _log(rng, 8, 256) if chunks else 1, "ctx": _log(rng, 64, 1500),
                "max_pos": rng.choice([2048, 4096])}
    if kind == "head":
        return {"kind": kind, "B": _log(rng, 1, 32), "d": 256 * _log(rng, 4, 16), "vocab": _log(rng, 4000, 128256)}
    heads, kv, hd = rng.choice([(32, 8, 128), (16, 4, 64), (32, 4, 64), (16, 8, 128)])
    return {"kind": kind, "layers": rng.choice([1, 2]), "d": heads * hd, "heads": heads, "kv_heads": kv,
            "ffn": 256 * _log(rng, 8, 56), "vocab": _log(rng, 256, 32000), "quant": rng.choice([18, 18, 18, 16]),
            "seqs": _log(rng, 1, 24), "prompt": _log(rng, 4, 64), "steps": rng.randint(0, 12)}


def prepare(case, seed):
    return dict(_KINDS[case["kind"]][0](case, seed), kind=case["kind"])


def run(state):
    return _KINDS[state["kind"]][1](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    return {"rel": _REL[case["kind"]]}
