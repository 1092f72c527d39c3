"""The calls whose speed is followed, as a program makes them through g2hip.

Six kinds of case:
  matvec     one decode matvec of the reference operator surface (bias, residual, GELU)
  splitk     the split-K matvec: strided partials, then the ordered reduction
  attention  single-query attention over the K/V cache: the three reference operators, or the fused call
  matmul     one prompt GEMM
  mlp        the MLP block of a prompt, operator by operator: LayerNorm, matmul, GELU, matmul, add
  model      a whole model: a prompt, then decode steps with given tokens, every forward's logits read

Sizes are the GPT-2 configurations' (n_embd 768..1600, ffn 4 n_embd, vocabulary 50257, head dim 64, context
1024) and ragged ones in between; a prompt has any length.  Activations are N(0, 1), weights N(0, 0.02), as the
random-init models have them.  Device buffers are torch tensors given to the library as pointers.
"""
import math
import os
import sys
from collections import OrderedDict

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpt2-opencl-1.1_amd"))
import g2hip  # noqa: E402

DEV = "cuda:0"
VOCAB, CTX = 50257, 1024
STD = 0.02
SHAPES = {"small": (12, 768, 12), "medium": (24, 1024, 16), "large": (36, 1280, 20), "xl": (48, 1600, 25)}


def listed():
    return [
        # a decode step's smallest matrix: the attention projection of the 124M model, added to the residual stream
        {"name": "matvec_proj", "kind": "matvec", "N": 768, "K": 768, "f16": False, "gelu": False, "residual": True},
        # the first MLP matrix of the 1.5B model with fp16 weights, GELU behind it
        {"name": "matvec_ffn_f16", "kind": "matvec", "N": 6400, "K": 1600, "f16": True, "gelu": True, "residual": False},
        # the vocabulary head of the 124M model: the longest matvec of a step, an odd number of columns
        {"name": "matvec_head", "kind": "matvec", "N": VOCAB, "K": 768, "f16": False, "gelu": False, "residual": False},
        # the second MLP matrix of the 124M model in the reference's split-K form, with its default four slices
        {"name": "splitk_ffn2", "kind": "splitk", "N": 768, "K": 3072, "slices": 4, "f16": False},
        # a decode step's attention by the three reference operators, 124M model, in the middle of a conversation
        {"name": "attention_ops", "kind": "attention", "heads": 12, "T": 700, "fused": False},
        # the same at the 1.5B model's width with the context full, by the fused call
        {"name": "attention_fused", "kind": "attention", "heads": 25, "T": CTX, "fused": True},
        # a short prompt's q/k/v matrix, 124M model
        {"name": "matmul_prompt", "kind": "matmul", "M": 64, "N": 2304, "K": 768, "f16": False},
        # a prompt of no round length through the 1.5B model's first MLP matrix, fp16 weights
        {"name": "matmul_ragged_f16", "kind": "matmul", "M": 333, "N": 6400, "K": 1600, "f16": True},
        # logits of every position of a full context: the largest product of the operator sweep
        {"name": "matmul_vocab", "kind": "matmul", "M": CTX, "N": VOCAB, "K": 1600, "f16": False},
        # the MLP block of the 774M model over a 256-token prompt, operator by operator
        {"name": "mlp_block", "kind": "mlp", "rows": 256, "E": 1280, "F": 5120},
        # prompt processing alone: the 774M model in fp32, 256 tokens to the first logits
        {"name": "prefill_large", "kind": "model", "size": "large", "f16": False, "fused": True, "prompt": 256, "steps": 0},
        # a request to the 1.5B model with fp16 weights: a 512-token prompt, then one token after another
        {"name": "request_xl_f16", "kind": "model", "size": "xl", "f16": True, "fused": True, "prompt": 512, "steps": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "splitk", "attention", "attention", "matmul", "matmul", "matmul", "mlp", "model"])
    f16 = rng.random() < 0.5
    if kind == "matvec":
        return {"kind": kind, "N": _log(rng, 512, VOCAB), "K": _log(rng, 256, 6400) if rng.random() < 0.5 else rng.choice([768, 1024, 1280, 1600]),
                "f16": f16, "gelu": rng.random() < 0.5, "residual": rng.random() < 0.5}
    if kind == "splitk":
        return {"kind": kind, "N": 4 * _log(rng, 128, 1600), "K": _log(rng, 256, 6400), "slices": rng.randint(1, 8), "f16": f16}
    if kind == "attention":
        return {"kind": kind, "heads": rng.choice([12, 16, 20, 25]), "T": _log(rng, 16, CTX), "fused": f16}
    if kind == "matmul":
        M, K = _log(rng, 8, CTX), _log(rng, 256, 6400)
        return {"kind": kind, "M": M, "N": min(_log(rng, 256, VOCAB), CTX * VOCAB * 1600 // (M * K)), "K": K, "f16": f16}
    if kind == "mlp":
        E = SHAPES[rng.choice(list(SHAPES))][1]
        return {"kind": kind, "rows": _log(rng, 8, CTX), "E": E, "F": 4 * E}
    if rng.random() < 0.3:  # the reference's own sequence of operators: fp32, short prompts
        return {"kind": kind, "size": "small", "f16": False, "fused": False, "prompt": _log(rng, 4, 96), "steps": rng.randint(0, 8)}
    size = rng.choice(["small", "medium", "large"])
    return {"kind": kind, "size": size, "f16": f16, "fused": True, "prompt": _log(rng, 4, 512), "steps": rng.randint(0, 8)}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _inputs(c, seed):
    """The case's random inputs on the GPU, by name: what exact() works from too."""
    g = _gen(seed)

    def acts(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    def weights(*shape, f16=False):
        w = torch.randn(shape, generator=g, device=DEV) * STD
        return w.half() if f16 else w

    k = c["kind"]
    if k in ("matvec", "splitk"):
        return {"A": acts(c["K"]), "B": weights(c["K"], c["N"], f16=c["f16"]), "bias": weights(c["N"]), "res": acts(c["N"])}
    if k == "attention":
        D = 64 * c["heads"]
        return {"qkv": acts(3 * D), "kc": acts(D, CTX), "vc": acts(CTX, D)}
    if k == "matmul":
        return {"A": acts(c["M"], c["K"]), "B": weights(c["K"], c["N"], f16=c["f16"]), "bias": weights(c["N"])}
    if k == "mlp":
        R, E, F = c["rows"], c["E"], c["F"]
        return {"x": acts(R, E), "g": 1 + 5 * weights(E), "b": 5 * weights(E), "w1": weights(E, F), "b1": weights(F),
                "w2": weights(F, E), "b2": weights(E)}
    ids = torch.randint(0, VOCAB, (c["prompt"] + c["steps"],), generator=g, device=DEV, dtype=torch.int32)
    return {"ids": ids.cpu().numpy()}


def _model_weights(size, f16):
    """Yields the tensors of a random-init model, the same for every seed of a case: a served model stays as it is
    loaded, its prompts change.  fp16 weights are given as the values that fp16 holds."""
    L, E, _ = SHAPES[size]
    g = _gen(20240 + E)

    def mat(*shape):
        w = torch.randn(shape, generator=g, device=DEV) * STD
        return w.half().float() if f16 else w

    yield mat(VOCAB, E), mat(CTX, E)
    for _ in range(L):
        yield mat(E, 3 * E), mat(E, E), mat(E, 4 * E), mat(4 * E, E)


_models = OrderedDict()  # loaded models, the last three: a program keeps the model that it serves


def _model(c):
    key = (c["size"], c["f16"], c["fused"])
    if key in _models:
        _models.move_to_end(key)
        return _models[key]
    L, E, H = SHAPES[c["size"]]
    it = _model_weights(c["size"], c["f16"])
    one, zero = torch.ones(E).numpy(), torch.zeros(4 * E).numpy()
    wte, wpe = (t.cpu().numpy() for t in next(it))
    layers = []
    for mats in it:
        qkv, proj, fc, fc2 = (t.cpu().numpy() for t in mats)
        layers.append((one, zero[:E], qkv, zero[:3 * E], proj, zero[:E], one, zero[:E], fc, zero, fc2, zero[:E]))
    cfg = g2hip.make_config(L, E, H)
    m = g2hip.Model.from_host(cfg, {"wte": wte, "wpe": wpe, "lnf_w": one, "lnf_b": zero[:E], "layers": layers},
                              g2hip.F16 if c["f16"] else g2hip.F32, g2hip.PATH_FUSED if c["fused"] else g2hip.PATH_REFERENCE)
    while len(_models) >= 3:
        _models.popitem(last=False)
    _models[key] = m
    return m


def prepare(case, seed):
    g2hip.init(0)
    s = {"c": case, **_inputs(case, seed)}

    def out(*shape):
        return torch.zeros(shape, device=DEV)

    k = case["kind"]
    if k in ("matvec", "splitk"):
        s["C"] = out(case["N"])
        if k == "splitk":
            s["partial"] = out(case["slices"], case["N"])
    elif k == "attention":
        s["out"] = out(64 * case["heads"])
        s["scores"] = out(case["heads"], CTX)
    elif k == "matmul":
        s["C"] = out(case["M"], case["N"])
    elif k == "mlp":
        s["ln"], s["h"], s["y"] = out(case["rows"], case["E"]), out(case["rows"], case["F"]), out(case["rows"], case["E"])
    else:
        s["model"] = _model(case)
    s["p"] = {n: t.data_ptr() for n, t in s.items() if isinstance(t, torch.Tensor)}
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    c, p = s["c"], s["p"]
    k = c["kind"]
    if k == "matvec":
        g2hip.matvec(p["A"], p["B"], p["bias"], p["res"] if c["residual"] else None, p["C"], c["N"], c["K"], c["gelu"], f16=c["f16"])
        return s["C"]
    if k == "splitk":
        g2hip.matvec_sk(p["A"], p["B"], p["partial"], c["N"], c["K"], c["slices"], f16=c["f16"])
        g2hip.reduce_partial(p["partial"], p["bias"], p["res"], p["C"], c["N"], c["slices"])
        return s["partial"], s["C"]
    if k == "attention":
        NH, T = c["heads"], c["T"]
        D = 64 * NH
        if c["fused"]:
            g2hip.attn_1q(p["qkv"], p["kc"], p["vc"], p["out"], 0, T, D, NH, CTX, 0, 0.125)
            return s["out"]
        g2hip.attn_scores_1q(p["qkv"], p["kc"], p["scores"], 0, T, D, 64, NH, CTX, 0.125)
        g2hip.attn_softmax_1q(p["scores"], T, NH)
        g2hip.attn_out_1q(p["scores"], p["vc"], p["out"], T, D, 64, 0)
        return s["scores"], s["out"]
    if k == "matmul":
        g2hip.matmul(p["A"], p["B"], p["bias"], p["C"], c["M"], c["N"], c["K"], f16=c["f16"])
        return s["C"]
    if k == "mlp":
        R, E, F = c["rows"], c["E"], c["F"]
        g2hip.layernorm(p["x"], p["ln"], p["g"], p["b"], E, R)
        g2hip.matmul(p["ln"], p["w1"], p["b1"], p["h"], R, F, E)
        g2hip.gelu(p["h"], R * F)
        g2hip.matmul(p["h"], p["w2"], p["b2"], p["y"], R, E, F)
        g2hip.add(p["y"], p["x"], R * E)
        return s["ln"], s["h"], s["y"]
    m, P = s["model"], c["prompt"]
    m.prefill(s["ids"][:P])
    logits = [m.logits()]
    for i in range(c["steps"]):
        m.decode(s["ids"][P + i], P + i)
        logits.append(m.logits())
    return logits


# ------------------------------------------------------------------ what a pass needs

def work(c):
    k = c["kind"]
    w = 2 if c.get("f16") else 4
    if k == "matvec":
        N, K = c["N"], c["K"]
        return {"bytes": w * N * K + 4 * K + 4 * N * (3 if c["residual"] else 2), "flops": 2 * N * K}
    if k == "splitk":
        N, K = c["N"], c["K"]
        return {"bytes": w * N * K + 4 * K + 4 * N * (3 + c["slices"]), "flops": 2 * N * K}
    if k == "attention":
        NH, T = c["heads"], c["T"]
        return {"bytes": 4 * 64 * NH * (2 * T + 2) + (0 if c["fused"] else 4 * NH * T), "flops": 4 * 64 * NH * T}
    if k == "matmul":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 4 * (M * K + M * N + N) + w * N * K, "flops": 2 * M * N * K}
    if k == "mlp":
        R, E, F = c["rows"], c["E"], c["F"]
        return {"bytes": 4 * (2 * E * F + F + 3 * E + R * (3 * E + F)), "flops": 4 * R * E * F}
    L, E, _ = SHAPES[c["size"]]
    P, S = c["prompt"], c["steps"]
    mats, kv = L * 12 * E * E, 2 * L * E
    cached = sum(P + i + 1 for i in range(S))  # positions that the decode steps read
    return {"bytes": (1 + S) * (w * (mats + E * VOCAB) + 4 * VOCAB) + 4 * kv * (P + S + cached),
            "flops": 2 * mats * (P + S) + 2 * (1 + S) * E * VOCAB + 2 * kv * (P * (P + 1) // 2 + cached)}


def tolerance(c):
    """About four times what the start shows against 64 bits: fp32 sums of a few thousand terms, in any order."""
    return {"rel": 8e-6 if c["kind"] == "model" else 4e-6}


# ------------------------------------------------------------------ the same in 64 bits

def _gelu(v):
    return 0.5 * v * (1 + torch.tanh(0.7978845608 * (v + 0.044715 * v ** 3)))


def _norm(x, g=1.0, b=0.0):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + 1e-5) * g + b


def _exact_model(c, ids):
    L, E, H = SHAPES[c["size"]]
    P, S = c["prompt"], c["steps"]
    it = _model_weights(c["size"], c["f16"])
    wte, wpe = (t.double() for t in next(it))
    t = torch.as_tensor(ids, device=DEV).long()
    n = P + S
    x = wte[t] + wpe[:n]
    mask = torch.triu(torch.full((n, n), -math.inf, dtype=torch.float64, device=DEV), 1)
    for mats in it:
        qkv, proj, fc, fc2 = (t.double() for t in mats)
        q, kk, v = (_norm(x) @ qkv).split(E, 1)
        heads = []
        for h in range(H):
            r = slice(64 * h, 64 * h + 64)
            heads.append(torch.softmax(q[:, r] @ kk[:, r].T.contiguous() * 0.125 + mask, 1) @ v[:, r].contiguous())
        x = x + torch.cat(heads, 1) @ proj
        x = x + _gelu(_norm(x) @ fc) @ fc2
    out = _norm(x[P - 1:]) @ wte.T.contiguous()
    return [row for row in out]


def exact(c, seed):
    s = {n: t.double() if isinstance(t, torch.Tensor) else t for n, t in _inputs(c, seed).items()}
    k = c["kind"]
    if k == "matvec":
        y = s["A"] @ s["B"] + s["bias"]
        y = y + s["res"] if c["residual"] else y
        return _gelu(y) if c["gelu"] else y
    if k == "splitk":
        n = c["slices"]
        partial = torch.stack([s["A"][i::n] @ s["B"][i::n] for i in range(n)])
        return partial, partial.sum(0) + s["bias"] + s["res"]
    if k == "attention":
        NH, T = c["heads"], c["T"]
        q = s["qkv"][: 64 * NH].view(NH, 64, 1)
        scores = torch.zeros(NH, CTX, dtype=torch.float64, device=DEV)
        scores[:, :T] = torch.softmax((q * s["kc"].view(NH, 64, CTX)[:, :, :T]).sum(1) * 0.125, 1)
        out = (scores[:, :T].T.reshape(T, NH, 1) * s["vc"][:T].view(T, NH, 64)).sum(0).reshape(-1)
        return out if c["fused"] else (scores, out)
    if k == "matmul":
        return s["A"] @ s["B"] + s["bias"]
    if k == "mlp":
        ln = _norm(s["x"], s["g"], s["b"])
        h = _gelu(ln @ s["w1"] + s["b1"])
        return ln, h, h @ s["w2"] + s["b2"] + s["x"]
    return _exact_model(c, s["ids"])
