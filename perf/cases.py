"""What the speed of this engine is measured on.

Each case is one call, or one short sequence of calls, that a program using
the engine makes: the two whole-model calls (decode steps and a chunked
prefill) and the single layers and products behind them, each through its own
public entry point of the C ABI on buffers that are already in HBM
(sg_gpu_wrap_device). Shapes are this repository's: the 2B and 27B model
configurations (surge_amd.CFG_2B, CFG_27B; the 27B's layers repeat with a
period of four, so four of them stand for all) and the per-kernel ones of
bench.py --micro.

Inputs are made from the seed alone with the distributions the path meets:
Q8_0 blocks of uniform int8 with f16 scales |N(0, 0.02)| / 127, unit-variance
activations, norm weights near 1, gates in their useful range.
"""
import ctypes as C
import math

import numpy as np
import torch

import surge_amd as S

KINDS = ("decode", "prefill", "attn_decode", "attn_chunk", "gdn_step", "gdn_chunk", "matvec", "matmul")
EPS = 1e-6
THETA = 1e7
VOCAB = S.CFG_2B["vocab"]

# (query heads, kv heads, head dim): the 27B's, the 2B's and the micro config's attention.
HEADS = ((24, 4, 256), (8, 2, 256), (16, 4, 256))
# (rows, cols) of the projections of both models, gate and up as the file holds them.
WEIGHTS_2B = ((8192, 2048), (6144, 2048), (2048, 6144), (4096, 2048), (2048, 2048))
WEIGHTS_27B = ((12288, 5120), (10240, 5120), (6144, 5120), (17408, 5120), (5120, 17408), (5120, 6144))


def listed():
    return [
        # One user's turn fed to the 2B model token by token (sg_gpu_prefill starts a new
        # sequence, so whatever continues one goes through the decode step): the smallest
        # kernels, where launches and latency count. The logits of the last token are read.
        {"name": "decode_2b", "kind": "decode", "shape": "2b", "layers": 24, "steps": 8},
        # A prompt into the 27B shape in the benchmark's 512-token chunks, the last one ragged
        # (1100 = 512 + 512 + 76), four of its layers and the head.
        {"name": "prefill_27b", "kind": "prefill", "shape": "27b", "layers": 4, "tokens": 1100, "chunk": 512},
        # Decode attention early in a conversation (the micro configuration's heads).
        {"name": "attn_decode_512", "kind": "attn_decode", "heads": 16, "kv_heads": 4, "head_dim": 256, "keys": 512},
        # Decode attention of the 27B deep in a document, at a length no tile divides.
        {"name": "attn_decode_32k", "kind": "attn_decode", "heads": 24, "kv_heads": 4, "head_dim": 256, "keys": 32771},
        # The 27B's attention layer over the last 512-token chunk of a 32k prompt.
        {"name": "attn_chunk_32k", "kind": "attn_chunk", "heads": 24, "kv_heads": 4, "head_dim": 256, "base": 32256,
         "tokens": 512},
        # The 2B's attention layer over the ragged end of a short prompt.
        {"name": "attn_chunk_ragged", "kind": "attn_chunk", "heads": 8, "kv_heads": 2, "head_dim": 256, "base": 1024,
         "tokens": 77},
        # One token through the 2B's DeltaNet layer (the micro configuration).
        {"name": "gdn_step_16", "kind": "gdn_step", "k_heads": 16, "v_heads": 16, "dim": 128},
        # The 27B's DeltaNet layer over a full chunk.
        {"name": "gdn_chunk_48", "kind": "gdn_chunk", "k_heads": 16, "v_heads": 48, "dim": 128, "tokens": 512, "first": 0},
        # The 2B's DeltaNet layer over a short prompt that no block divides, starting off the ring's origin.
        {"name": "gdn_chunk_ragged", "kind": "gdn_chunk", "k_heads": 16, "v_heads": 16, "dim": 128, "tokens": 45, "first": 3},
        # One quantised linear layer on one token (the micro configuration).
        {"name": "matvec_4096", "kind": "matvec", "rows": 4096, "cols": 4096},
        # The 27B's gate projection over a full chunk: the largest product of a prefill.
        {"name": "matmul_gate_512", "kind": "matmul", "tokens": 512, "rows": 17408, "cols": 5120},
        # The 27B's down projection over a short prompt.
        {"name": "matmul_down_40", "kind": "matmul", "tokens": 40, "rows": 5120, "cols": 17408},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    if kind == "decode":
        shape = rng.choice(("2b", "27b"))
        layers = 4 * rng.randint(1, 6) if shape == "2b" else 4
        return {"kind": kind, "shape": shape, "layers": layers, "steps": rng.randint(1, 8)}
    if kind == "prefill":
        shape = rng.choice(("2b", "27b"))
        layers = 4 * rng.randint(1, 3) if shape == "2b" else 4
        return {"kind": kind, "shape": shape, "layers": layers, "tokens": _log(rng, 6, 1100),
                "chunk": rng.choice((256, 512, 1024))}
    if kind in ("attn_decode", "attn_chunk"):
        nh, nkv, hd = rng.choice(HEADS)
        c = {"kind": kind, "heads": nh, "kv_heads": nkv, "head_dim": hd}
        if kind == "attn_decode":
            c["keys"] = _log(rng, 24, 200000)
        else:
            c["base"] = 0 if rng.random() < 0.25 else _log(rng, 16, 32000)
            c["tokens"] = _log(rng, 6, 512)
        return c
    if kind in ("gdn_step", "gdn_chunk"):
        nk = rng.choice((4, 8, 12, 16, 16, 16))     # 16 in both models; less is a shard or a small model
        c = {"kind": kind, "k_heads": nk, "v_heads": nk * rng.randint(1, 3), "dim": rng.choice((64, 128, 128))}
        if kind == "gdn_chunk":
            c["tokens"] = _log(rng, 6, 1024)
            c["first"] = rng.randint(0, 3)
        return c
    rows, cols = rng.choice(WEIGHTS_2B + WEIGHTS_27B)
    if rng.random() < 0.5:      # generic sizes: any row count, whole Q8_0 blocks
        rows, cols = _log(rng, 500, 17408), 32 * _log(rng, 16, 544)
    if kind == "matvec":
        if rng.random() < 0.2:
            rows, cols = VOCAB, 2048      # the 2B's head
        return {"kind": kind, "rows": rows, "cols": cols}
    most = 512 * 17408 * 5120 // (rows * cols)
    return {"kind": kind, "tokens": min(_log(rng, 2, 1024), max(2, most)), "rows": rows, "cols": cols}


# ---------------------------------------------------------------- what a program holds

class _Dev:
    """A tensor's memory as a buffer handle."""

    def __init__(self, gpu, t):
        self.t = t
        h = C.c_void_p()
        S.check(S.lib().sg_gpu_wrap_device(gpu.handle, t.data_ptr(), t.numel() * t.element_size(), C.byref(h)))
        self.handle = h

    def __del__(self):
        S.lib().sg_gpu_buf_free(self.handle)


class _Model:
    """A model on the GPU with a decode state, as Gpu and Synth give it."""

    def __init__(self, cfg, seed, max_ctx):
        self.syn = S.Synth(cfg, S.SG_T_Q8_0, seed=seed)
        self.gpu = S.Gpu()
        self.gpu.load_model(self.syn.model)
        self.gpu.state_new(max_ctx)

    def __del__(self):
        if getattr(self, "gpu", None) is not None:
            self.gpu.close()
        self.syn.close()


_one_gpu = None


def _gpu():
    """The one handle that all single-layer calls of the program go through."""
    global _one_gpu
    if _one_gpu is None:
        _one_gpu = S.Gpu()
    return _one_gpu


def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) % (1 << 62))


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _q8(g, rows, cols):
    """A Q8_0 matrix as a file holds it: [rows][cols/32] blocks of an f16 scale and 32 int8."""
    nb = cols // 32
    q = torch.randint(-127, 128, (rows, nb, 32), generator=g, device="cuda", dtype=torch.int8)
    d = (torch.randn((rows, nb, 1), generator=g, device="cuda").abs() * (0.02 / 127)).half()
    return torch.cat([d.view(torch.uint8), q.view(torch.uint8)], dim=2).contiguous()


def _cfg(case):
    return dict(S.CFG_2B if case["shape"] == "2b" else S.CFG_27B, n_layers=case["layers"])


def _tokens(case, seed, n):
    return np.random.default_rng(seed).integers(0, VOCAB, n).astype(np.int32)


def _inputs(case, seed):
    """The input tensors of a single-layer case, by name."""
    g, k = _rng(seed), case["kind"]
    if k == "attn_decode":
        nh, nkv, hd, n = case["heads"], case["kv_heads"], case["head_dim"], case["keys"]
        return {"q": _normal(g, nh, hd), "k": _normal(g, n, nkv, hd).half(), "v": _normal(g, n, nkv, hd).half()}
    if k == "attn_chunk":
        nh, nkv, hd, base, n = (case[x] for x in ("heads", "kv_heads", "head_dim", "base", "tokens"))
        kv = _normal(g, 2, base + n, nkv, hd).half()
        kv[:, base:] = 0
        return {"in": _normal(g, n, 2 * nh * hd + 2 * nkv * hd), "w": _uniform(g, 0.9, 1.1, 2 * hd), "kv": kv}
    if k in ("gdn_step", "gdn_chunk"):
        nk, nv, n, d = case["k_heads"], case["v_heads"], case.get("tokens", 1), case["dim"]
        cd, vd = (2 * nk + nv) * d, nv * d
        w = torch.cat([_uniform(g, -0.5, 0.5, cd * 4), -torch.exp(_uniform(g, -1, 1, nv)), _uniform(g, -0.5, 0.5, nv),
                       _uniform(g, 0.9, 1.1, d)])
        state = torch.cat([_normal(g, 3 * cd), _normal(g, vd * d) * 0.05])
        return {"in": _normal(g, n, cd + vd + 2 * nv), "w": w, "state": state}
    w = _q8(g, case["rows"], case["cols"])
    return {"w": w, "x": _normal(g, case.get("tokens", 1), case["cols"])}


def prepare(case, seed):
    k = case["kind"]
    if k in ("decode", "prefill"):
        n = case["steps"] if k == "decode" else case["tokens"]
        return {"case": case, "model": _Model(_cfg(case), seed, 4096), "tokens": _tokens(case, seed, n)}
    gpu, t = _gpu(), _inputs(case, seed)
    if k == "attn_decode":
        nh, nkv, hd, n = case["heads"], case["kv_heads"], case["head_dim"], case["keys"]
        t["out"] = torch.empty(nh, hd, device="cuda")
        p = [nh, nkv, hd, n, hd, S.fbits(1 / math.sqrt(hd))]
    elif k == "attn_chunk":
        nh, nkv, hd, base, n = (case[x] for x in ("heads", "kv_heads", "head_dim", "base", "tokens"))
        t["out"] = torch.empty(n, nh, hd, device="cuda")
        p = [nh, nkv, hd, 64, base, n, S.fbits(THETA), S.fbits(EPS)]
    elif k in ("gdn_step", "gdn_chunk"):
        nk, nv, n, d = case["k_heads"], case["v_heads"], case.get("tokens", 1), case["dim"]
        t["out"] = torch.empty(n, nv * d, device="cuda")
        p = [d, d, nv, nk, 4, 1, 1, S.fbits(EPS)]
        if k == "gdn_chunk":
            p = [d, d, nv, nk, 4, 3 | case["first"] << 2, n, S.fbits(EPS)]
    elif k == "matvec":
        t["out"] = torch.empty(case["rows"], device="cuda")
        p = [case["rows"], case["cols"]]
    else:
        t["out"] = torch.empty(case["tokens"], case["rows"], device="cuda")
        p = [case["tokens"], case["rows"], case["cols"]]
    return {"case": case, "gpu": gpu, "p": S.params(p), "t": t, "b": {n: _Dev(gpu, x) for n, x in t.items()}}


def run(state):
    k = state["case"]["kind"]
    if k == "decode":
        gpu, tokens = state["model"].gpu, state["tokens"]
        gpu.state_reset()
        for pos, tok in enumerate(tokens[:-1]):
            gpu.forward_nosync(int(tok), pos)
        return gpu.forward(int(tokens[-1]), len(tokens) - 1)
    if k == "prefill":
        return state["model"].gpu.prefill(state["tokens"], state["case"]["chunk"])
    L, g, b, t, p = S.lib(), state["gpu"].handle, state["b"], state["t"], state["p"]
    out = t["out"]
    if k == "attn_decode":
        S.check(L.sg_gpu_run_attn_decode_f16(g, b["q"].handle, b["k"].handle, b["v"].handle, b["out"].handle, p))
        return out
    if k == "attn_chunk":
        S.check(L.sg_gpu_run_attn_chunk(g, b["in"].handle, b["w"].handle, b["kv"].handle, b["out"].handle, p))
        return {"out": out, "kv": t["kv"]}
    if k in ("gdn_step", "gdn_chunk"):
        f = L.sg_gpu_run_gdn_step if k == "gdn_step" else L.sg_gpu_run_gdn_chunk
        S.check(f(g, b["in"].handle, b["w"].handle, b["state"].handle, b["out"].handle, p))
        return {"out": out, "state": t["state"]}
    if k == "matvec":
        S.check(L.sg_gpu_run_op(g, b"k_matvec_q8", b["w"].handle, b["x"].handle, b["out"].handle, p))
    else:
        S.check(L.sg_gpu_run_op(g, b"k_matmul_q8", b["x"].handle, b["w"].handle, b["out"].handle, p))
    return out


# ---------------------------------------------------------------- the work of one pass

def _mats(c, i):
    """(rows, cols) of layer i's matrices: input projection, output projection, gate/up, down."""
    h, f, hd = c["hidden"], c["ffn_hidden"], c["head_dim"]
    if (i + 1) % c["full_attn_interval"] == 0:
        aw = c["n_heads"] * hd
        a = [(2 * aw + 2 * c["n_kv_heads"] * hd, h), (h, aw)]
    else:
        vd = c["n_v_heads"] * c["head_v_dim"]
        a = [(2 * c["n_k_heads"] * c["head_k_dim"] + 2 * vd + 2 * c["n_v_heads"], h), (h, vd)]
    return a + [(2 * f, h), (h, f)]


def work(case):
    k = case["kind"]
    if k in ("decode", "prefill"):
        c = _cfg(case)
        body = sum(r * n for i in range(c["n_layers"]) for r, n in _mats(c, i))
        head = c["vocab"] * c["hidden"]
        n_gdn = c["n_layers"] * 3 // 4
        s = 4 * c["n_v_heads"] * c["head_v_dim"] * c["head_k_dim"]
        pairs = c["n_layers"] // 4 * c["n_heads"] * c["head_dim"]
        if k == "decode":       # every step reads every weight and reads and writes the DeltaNet state
            n = case["steps"]
            return {"bytes": n * ((body + head) * 34 // 32 + 2 * n_gdn * s + 4 * c["vocab"]),
                    "flops": n * 2 * (body + head)}
        n = case["tokens"]
        chunks = -(-n // case["chunk"])
        return {"bytes": (chunks * body + head) * 34 // 32 + 2 * chunks * n_gdn * s,
                "flops": 2 * n * body + 2 * head + 2 * n * n * pairs + 6 * n * n_gdn * s / 4}
    if k == "attn_decode":
        nh, nkv, hd, n = case["heads"], case["kv_heads"], case["head_dim"], case["keys"]
        return {"bytes": 4 * n * nkv * hd + 8 * nh * hd, "flops": 4 * n * nh * hd}
    if k == "attn_chunk":
        nh, nkv, hd, base, n = (case[x] for x in ("heads", "kv_heads", "head_dim", "base", "tokens"))
        return {"bytes": 4 * (base + n) * nkv * hd + 4 * n * (3 * nh + 2 * nkv) * hd,
                "flops": 4 * nh * hd * (n * base + n * (n + 1) / 2)}
    if k in ("gdn_step", "gdn_chunk"):
        nk, nv, n, d = case["k_heads"], case["v_heads"], case.get("tokens", 1), case["dim"]
        cd, vd = (2 * nk + nv) * d, nv * d
        return {"bytes": 4 * (n * (cd + 2 * vd + 2 * nv) + 4 * cd + 2 * (3 * cd + vd * d)), "flops": n * 6 * vd * d}
    n, rows, cols = case.get("tokens", 1), case["rows"], case["cols"]
    return {"bytes": rows * cols * 34 // 32 + 4 * n * (rows + cols), "flops": 2 * n * rows * cols}


# About four times the distance from exact() measured over the ranges above. 32-bit sums give
# 1e-7 to 3e-7; the products split x into two bf16 (2^-16 per element); what passes through the
# f16 K/V cache moves further where a value falls on the other side of a rounding (one cached
# element by 2^-11, which a whole model then carries through its layers to the logits).
TOLERANCE = {
    "decode": {"rel": 2.5e-4, "max": 1.3e-3},
    "prefill": {"rel": 2.2e-4, "max": 1.2e-3},
    "attn_decode": {"rel": 1.3e-6, "max": 6e-6},
    "attn_chunk": {"rel": 1e-4, "max": 4e-3},
    "gdn_step": {"rel": 8e-7, "max": 4e-6},
    "gdn_chunk": {"rel": 8e-7, "max": 4e-5},
    "matvec": {"rel": 4e-7, "max": 2e-6},
    "matmul": {"rel": 1e-5, "max": 6e-5},
}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# ---------------------------------------------------------------- the same in 64 bits

def _dequant(raw, rows, cols):
    b = raw.reshape(rows, cols // 32, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).reshape(rows, cols)


def _rms(x, w, eps):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _rope(x, pos, rd):
    """x [n][heads][hd], the first rd dims rotated in half-split pairs."""
    h = rd // 2
    inv = torch.tensor([THETA ** (-2.0 * i / rd) for i in range(h)], dtype=torch.float64, device=x.device)
    ang = pos.double()[:, None] * inv
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :h], x[..., h:rd]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., rd:]], dim=-1)


def _attn(q, k, v, base):
    """Causal attention of q [n][nh][hd] at positions base.. over k, v [base+n][nkv][hd]."""
    n, nh, hd = q.shape
    keys, nkv, _ = k.shape
    mask = torch.arange(keys, device=q.device)[None, :] > base + torch.arange(n, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(nh):
        kh, vh = k[:, h * nkv // nh].contiguous(), v[:, h * nkv // nh].contiguous()
        s = (q[:, h] @ kh.T.contiguous()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), dim=-1) @ vh
    return out


def _attn_layer(rows, qn, kn, k_old, v_old, nh, nkv, hd, eps):
    """An attention layer's core on projection rows [n][q|gate per head, k, v]: the gated
    output, and K and V of the new positions. The cache keeps 16-bit floats."""
    n, base = rows.shape[0], k_old.shape[0]
    qg = rows[:, :2 * nh * hd].reshape(n, nh, 2 * hd)
    k = rows[:, 2 * nh * hd:(2 * nh + nkv) * hd].reshape(n, nkv, hd)
    v = rows[:, (2 * nh + nkv) * hd:].reshape(n, nkv, hd)
    pos = torch.arange(base, base + n, device=rows.device)
    q, k = _rope(_rms(qg[..., :hd], qn, eps), pos, 64), _rope(_rms(k, kn, eps), pos, 64)
    o = _attn(q, torch.cat([k_old, k.float().half().double()]), torch.cat([v_old, v.float().half().double()]), base)
    return o * torch.sigmoid(qg[..., hd:]), k, v


def _gdn_layer(rows, conv_w, ssm_a, dt_bias, norm_w, tail, st, nk, nv, eps):
    """A DeltaNet layer's core on projection rows [n][qkv, z, b, a]: outputs, new conv tail,
    new state. Value heads are tiled over the key heads; ssm_a holds -exp(A_log)."""
    n, d = rows.shape[0], norm_w.numel()
    cd, vd = (2 * nk + nv) * d, nv * d
    x = torch.cat([tail, rows[:, :cd]])
    y = sum(x[j:j + n] * conv_w[:, j] for j in range(4))
    y = y * torch.sigmoid(y)
    q = _rms(y[:, :nk * d].reshape(n, nk, d), None, 1e-6) / d
    k = _rms(y[:, nk * d:2 * nk * d].reshape(n, nk, d), None, 1e-6) / math.sqrt(d)
    v = y[:, 2 * nk * d:].reshape(n, nv, d)
    z, b, a = rows[:, cd:cd + vd].reshape(n, nv, d), rows[:, cd + vd:cd + vd + nv], rows[:, cd + vd + nv:]
    beta, decay = torch.sigmoid(b), torch.exp(ssm_a * torch.nn.functional.softplus(a + dt_bias, threshold=1e9))
    hk = torch.arange(nv, device=rows.device) % nk
    q, k = q[:, hk], k[:, hk]
    out = torch.empty(n, nv, d, dtype=torch.float64, device=rows.device)
    st = st.clone()
    for t in range(n):
        st *= decay[t][:, None, None]
        delta = (v[t] - (st * k[t][:, None, :]).sum(-1)) * beta[t][:, None]
        st += delta[:, :, None] * k[t][:, None, :]
        out[t] = (st * q[t][:, None, :]).sum(-1)
    out = _rms(out, norm_w, eps) * z * torch.sigmoid(z)
    return out.reshape(n, vd), x[n:], st


def _host(ptr, nbytes):
    return torch.from_numpy(np.ctypeslib.as_array(C.cast(ptr, C.POINTER(C.c_uint8)), shape=(nbytes,))).cuda()


def _exact_model(case, seed):
    c, eps = _cfg(case), EPS
    syn = S.Synth(c, S.SG_T_Q8_0, seed=seed)
    m = syn.model.contents
    tokens = torch.from_numpy(_tokens(case, seed, case.get("steps") or case["tokens"])).long().cuda()
    h, f, nh, nkv, hd = c["hidden"], c["ffn_hidden"], c["n_heads"], c["n_kv_heads"], c["head_dim"]
    nk, nv, d = c["n_k_heads"], c["n_v_heads"], c["head_k_dim"]
    cd, vd, aw = (2 * nk + nv) * d, nv * d, nh * hd

    def mat(ptr, rows, cols):
        return _dequant(_host(ptr, rows * cols // 32 * 34), rows, cols)

    def small(ptr, n):
        return _host(ptr, 4 * n).view(torch.float32).double()

    def times(x, ptr, rows, cols):
        return x @ mat(ptr, rows, cols).T

    emb = _host(m.tok_emb, c["vocab"] * h // 32 * 34).reshape(c["vocab"], -1)[tokens].contiguous()
    x = _dequant(emb, len(tokens), h)
    for i in range(c["n_layers"]):
        w = m.layers[i]
        y = _rms(x, small(w.ln1, h), eps)
        if w.q_proj:
            rows = torch.cat([times(y, w.q_proj, 2 * aw, h), times(y, w.k_proj, nkv * hd, h),
                              times(y, w.v_proj, nkv * hd, h)], dim=1)
            none = torch.empty(0, nkv, hd, dtype=torch.float64, device="cuda")
            o, _, _ = _attn_layer(rows, small(w.q_norm, hd), small(w.k_norm, hd), none, none, nh, nkv, hd, eps)
            x = x + times(o.reshape(-1, aw), w.o_proj, h, aw)
        else:
            rows = torch.cat([times(y, w.ssm_in_qkv, cd, h), times(y, w.ssm_in_z, vd, h), times(y, w.ssm_in_b, nv, h),
                              times(y, w.ssm_in_a, nv, h)], dim=1)
            o, _, _ = _gdn_layer(rows, small(w.ssm_conv1d, cd * 4).reshape(cd, 4), small(w.ssm_a, nv),
                                 small(w.ssm_dt_bias, nv), small(w.ssm_norm, d),
                                 torch.zeros(3, cd, dtype=torch.float64, device="cuda"),
                                 torch.zeros(nv, d, d, dtype=torch.float64, device="cuda"), nk, nv, eps)
            x = x + times(o, w.ssm_out, h, vd)
        y = _rms(x, small(w.ln2, h), eps)
        g = times(y, w.gate_proj, f, h)
        x = x + times(g * torch.sigmoid(g) * times(y, w.up_proj, f, h), w.down_proj, h, f)
    y = _rms(x[-1:], small(m.out_norm, h), eps)
    out = times(y, m.lm_head, c["vocab"], h).reshape(-1)
    syn.close()
    return out


def exact(case, seed):
    k = case["kind"]
    if k in ("decode", "prefill"):
        return _exact_model(case, seed)
    t = _inputs(case, seed)
    if k == "attn_decode":
        return _attn(t["q"].double()[None], t["k"].double(), t["v"].double(), case["keys"] - 1)[0]
    if k == "attn_chunk":
        nh, nkv, hd, base = (case[x] for x in ("heads", "kv_heads", "head_dim", "base"))
        w, old = t["w"].double(), t["kv"][:, :base].double()
        o, kn, vn = _attn_layer(t["in"].double(), w[:hd], w[hd:], old[0], old[1], nh, nkv, hd, EPS)
        return {"out": o, "kv": torch.stack([torch.cat([old[0], kn]), torch.cat([old[1], vn])])}
    if k in ("gdn_step", "gdn_chunk"):
        nk, nv, d = case["k_heads"], case["v_heads"], case["dim"]
        cd, vd = (2 * nk + nv) * d, nv * d
        w, st = t["w"].double(), t["state"].double()
        o, tail, s = _gdn_layer(t["in"].double(), w[:4 * cd].reshape(cd, 4), w[4 * cd:4 * cd + nv],
                                w[4 * cd + nv:4 * cd + 2 * nv], w[4 * cd + 2 * nv:], st[:3 * cd].reshape(3, cd),
                                st[3 * cd:].reshape(nv, d, d), nk, nv, EPS)
        return {"out": o, "state": torch.cat([tail.reshape(-1), s.reshape(-1)])}
    y = t["x"].double() @ _dequant(t["w"], case["rows"], case["cols"]).T
    return y[0] if k == "matvec" else y
