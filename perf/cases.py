"""The work that users of this framework run on one GPU, as timed cases: MoE layers on
device buffers (decode and batches, every device form of the experts), the host-buffer
hook that glm.c's C host calls, and the whole model's batched prefill and decode.

A case's checkpoint (weights, seeded by its shape alone) is what a program loads once;
its inputs (activations, prompt tokens, the latent cache they fill) come from the seed
given to prepare(). Weights are drawn as the framework's benchmark draws them: int8
uniform in [-127, 127], scales |N(0, 1)| times a constant (held by fp16 at group size 32,
fp32 otherwise), router N(0, 0.02), selection bias N(0, 0.01) or Zipf(1.2), norms N(1, 0.1).
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "glm.c_amd"))

import gmoe  # noqa: E402

DEV = "cuda"
EPS = 1e-5
MOE_SCALE = 0.002  # of the expert weights, as the benchmark's layers
ATT_SCALE = 0.001  # of the dense side: attention scores of standard deviation 2 to 3
ROUTED_SCALE = 1.8
MIN_DENOM = 6.103515625e-5  # glm.c's least denominator of the top-k weights
# GLM-4.7-Flash's MoE shape; a case names what differs from it
MOE = {"D": 2048, "F": 1536, "E": 64, "K": 4, "gs": 32, "zipf": False}
# and its dense side
DENSE = {"dim": 2048, "hidden_dim": 10240, "vocab_size": 154880, "q_lora_rank": 768, "kv_lora_rank": 512,
         "rope_dim": 64, "qk_nope_dim": 192, "head_k_dim": 256, "v_head_dim": 256}
PREFILL_BATCH = 1024


def listed():
    return [
        # one decode step through all MoE layers of GLM-4.7-Flash, as a serving loop runs it
        {"name": "decode_46_layers", "op": "moe", "T": 1, "layers": 46},
        # the same step on a pipeline stage's layers in the form glm.c's exporter writes
        {"name": "decode_16_layers_gs16", "op": "moe", "T": 1, "layers": 16, "gs": 16},
        # glm.c's own token loop: each MoE layer called on activations in host memory
        {"name": "hook_4_layers", "op": "hook", "T": 1, "layers": 4},
        # a few sequences decoded together, or a prompt's short tail
        {"name": "batch_8", "op": "moe", "T": 8, "layers": 4},
        # a ragged small batch in the exporter's form
        {"name": "batch_37_gs16", "op": "moe", "T": 37, "layers": 2, "gs": 16},
        # skewed routing: four experts take about two fifths of the assignments
        {"name": "batch_128_zipf", "op": "moe", "T": 128, "layers": 1, "zipf": True},
        # a prompt batch through one layer
        {"name": "batch_512", "op": "moe", "T": 512, "layers": 1},
        # the default prefill batch in the exporter's form
        {"name": "batch_1024_gs16", "op": "moe", "T": 1024, "layers": 1, "gs": 16},
        # a checkpoint of another group size: glm.c's own layout on the device
        {"name": "batch_64_gs64", "op": "moe", "T": 64, "layers": 1, "gs": 64},
        # the last batch of a 4096-token prompt: the longest attention of its prefill
        {"name": "prefill_1024_at_3072", "op": "prefill", "n": 1024, "pos": 3072, "layers": 3},
        # a short prompt of odd length in the exporter's form
        {"name": "prefill_201_gs16", "op": "prefill", "n": 201, "pos": 0, "layers": 3, "gs": 16},
        # one token of the whole model's forward after a 4096-token prompt
        {"name": "decode_at_4096", "op": "decode", "pos": 4096, "layers": 6},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["moe", "moe", "moe", "moe", "hook", "prefill", "prefill", "decode"])
    gs = rng.choice([32, 32, 16, 16, 64])
    if op in ("moe", "hook"):
        T = _log(rng, 1, 1024) if op == "moe" else _log(rng, 1, 64)
        c = {"op": op, "T": T, "layers": rng.randint(1, 8) if T <= 8 else rng.randint(1, 2), "gs": gs}
        if rng.random() < 0.5:  # other shapes that the framework's tests run
            c.update(D=rng.choice([1024, 2048]), F=rng.choice([768, 1024, 1536]), E=rng.choice([32, 64, 128]),
                     K=rng.choice([2, 4, 6, 8]))
        if rng.random() < 0.25:
            c["zipf"] = True
        return c
    c = {"op": op, "layers": rng.randint(2, 3), "gs": rng.choice([32, 16]), "n_heads": rng.choice([4, 20, 20])}
    if op == "prefill":
        c["n"] = _log(rng, 1, 1024)
        c["pos"] = rng.choice([0, rng.randint(1, 3072)])
    else:
        c["pos"] = _log(rng, 16, 4096)
    return c


def _moe(case):
    return {k: case.get(k, v) for k, v in MOE.items()}


def _dense(case):
    L = case["layers"]
    return dict(DENSE, n_layers=L, attn_layers=L, has_l0_ffn=1, n_heads=case.get("n_heads", 20),
                group_size=case.get("gs", 32))


# ---- the checkpoint ------------------------------------------------------------------------


def _gen(*key):
    s = 17
    for k in key:
        s = (s * 1000003 + int(k) + 1) % (1 << 62)
    g = torch.Generator(device=DEV)
    g.manual_seed(s)
    return g


def _q8(g, rows, cols, gs, scale, lead=()):
    """int8 values and fp32 scales per group (values that fp16 holds at group size 32)."""
    q = torch.randint(-127, 128, (*lead, rows, cols), generator=g, device=DEV, dtype=torch.int8)
    s = torch.randn((*lead, rows, cols // gs), generator=g, device=DEV).abs_() * scale
    return q, (s.half().float() if gs == 32 else s)


def _norm(g, n):
    return 1 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _experts(m):
    """One layer's expert matrices; every layer of a case holds a copy of them in memory of its own."""
    D, F, E, gs = m["D"], m["F"], m["E"], m["gs"]
    g = _gen(1, D, F, E, gs)
    w = {}
    for name, rows, cols in (("gate", F, D), ("up", F, D), ("down", D, F)):
        w[name + "_q"], w[name + "_s"] = _q8(g, rows, cols, gs, MOE_SCALE, (E,))
        w[name + "_sh_q"], w[name + "_sh_s"] = _q8(g, rows, cols, gs, MOE_SCALE)
    return w


def _router(m, layer):
    D, E = m["D"], m["E"]
    g = _gen(2, D, E, m["K"], m["zipf"], layer)
    w = {"ffn_norm": _norm(g, D), "gate_inp": 0.02 * torch.randn(E, D, generator=g, device=DEV)}
    b = 0.01 * torch.randn(E, generator=g, device=DEV)
    if m["zipf"]:  # popularity falls as rank^-1.2 over a seeded order of the experts
        rank = torch.randperm(E, generator=g, device=DEV) + 1
        pop = rank.float() ** -gmoe.ZIPF_S
        b = gmoe.ZIPF_BETA * torch.log(pop / pop.mean())
    w["exp_probs_b"] = b
    return w


class _Layer:
    """A layer's host arrays, as gmoe.Context.upload takes them."""

    def __init__(self, arrays):
        self.arrays = arrays

    def weights(self):
        return gmoe.LayerWeights(*[gmoe.ptr(self.arrays[n]) for n, _ in gmoe.LayerWeights._fields_])


def _host(w):
    return {k: v.cpu().numpy() for k, v in w.items()}


def _dense_weights(c):
    """The model-wide tensors and each attention layer's, on the GPU."""
    D, gs, H, V, F = c["dim"], c["group_size"], c["n_heads"], c["vocab_size"], c["hidden_dim"]
    kv, rope, ql = c["kv_lora_rank"], c["rope_dim"], c["q_lora_rank"]
    g = _gen(3, D, H, gs)

    def q8(w, name, rows, cols):
        w[name + "_q"], w[name + "_s"] = _q8(g, rows, cols, gs, ATT_SCALE)

    top = {"output_norm": _norm(g, D), "l0_ffn_norm": _norm(g, D)}
    q8(top, "tok", V, D)
    q8(top, "out", V, D)
    q8(top, "l0_ffn_gate", F, D)
    q8(top, "l0_ffn_up", F, D)
    q8(top, "l0_ffn_down", D, F)
    layers = []
    for _ in range(c["n_layers"]):
        a = {"attn_norm": _norm(g, D), "q_a_norm": _norm(g, ql), "kv_a_norm": _norm(g, kv)}
        q8(a, "q_a", ql, D)
        q8(a, "q_b", H * c["head_k_dim"], ql)
        q8(a, "kv_a", kv + rope, D)
        q8(a, "k_b", H * kv, c["qk_nope_dim"])
        q8(a, "v_b", H * c["v_head_dim"], kv)
        q8(a, "attn_out", D, H * c["v_head_dim"])
        layers.append(a)
    return top, layers


_loaded = {}  # what the program has loaded: the checkpoint of the most recent shape


def _load(kind, key, make):
    if _loaded.get(kind, (None,))[0] != key:
        _loaded.pop(kind, None)
        _loaded[kind] = (key, make())
    return _loaded[kind][1]


def _context(m, layers, max_tokens):
    """A gmoe.Context with `layers` MoE layers resident."""
    def make():
        shape = gmoe.Shape(m["D"], m["F"], m["E"], m["K"], m["gs"])
        ctx = gmoe.Context(shape, n_layers=layers + 1, max_tokens=max_tokens)
        experts = _host(_experts(m))
        for layer in range(1, layers + 1):
            ctx.upload(layer, _Layer({**experts, **_host(_router(m, layer))}))
        return ctx

    return _load("moe", (tuple(m.items()), layers, max_tokens), make)


def _model(c, m, cap):
    """A gmoe.Model (a latent cache of its own) around the shared MoE layers, and those."""
    batch = PREFILL_BATCH
    ctx = _context(m, c["n_layers"] - 1, batch)

    def make():
        top, layers = _dense_weights(c)
        return _host(top), [_host(a) for a in layers]

    top, layers = _load("dense", tuple(c.items()), make)
    model = gmoe.Model(dict(c, cache_cap=cap, max_batch=batch))
    model.upload(top)
    for layer, a in enumerate(layers):
        model.upload_attn(layer, a)
    model.set_moe(ctx, range(1, c["n_layers"]))
    return model, ctx


def _activations(case, m, seed):
    return torch.randn(case["T"], m["D"], generator=_gen(4, seed), device=DEV)


def _tokens(n, vocab, seed):
    return torch.randint(3, vocab, (n,), generator=_gen(5, seed), device=DEV, dtype=torch.int32).cpu().numpy()


# ---- the cases -----------------------------------------------------------------------------


def prepare(case, seed):
    m = _moe(case)
    if case["op"] in ("moe", "hook"):
        ctx = _context(m, case["layers"], case["T"])
        x = _activations(case, m, seed)
        if case["op"] == "hook":
            return {"case": case, "ctx": ctx, "x": x.cpu().numpy()}
        return {"case": case, "ctx": ctx, "x": x, "out": torch.empty_like(x)}
    c = _dense(case)
    n = case["n"] if case["op"] == "prefill" else 1
    tokens = _tokens(case["pos"] + n, c["vocab_size"], seed)
    model, ctx = _model(c, m, case["pos"] + n)
    for p in range(0, case["pos"], PREFILL_BATCH):  # the prompt before the call
        model.prefill(tokens[p:min(p + PREFILL_BATCH, case["pos"])], p)
    return {"case": case, "ctx": ctx, "model": model, "tokens": tokens}


def run(state):
    case = state["case"]
    if case["op"] == "moe":
        x, out = state["x"], state["out"]
        state["ctx"].forward_layers(1, case["layers"], case["T"], x.data_ptr(), out.data_ptr(),
                                    stream=torch.cuda.current_stream().cuda_stream)
        return out
    if case["op"] == "hook":
        x, outs = state["x"], []
        for layer in range(1, case["layers"] + 1):
            x, st = gmoe.forward_host(state["ctx"], layer, x)
            outs.append({"x": x, **{k: st[k] for k in ("xn", "router_prob", "topk_idx", "topk_w", "shared_out",
                                                        "routed_out")}})
        return outs
    if case["op"] == "prefill":
        return state["model"].prefill(state["tokens"][case["pos"]:], case["pos"])
    return state["model"].forward_token(state["tokens"][case["pos"]], case["pos"])


def _touched(m, T):
    """Distinct routed experts that T tokens of K assignments are expected to touch."""
    E, K = m["E"], m["K"]
    p = [1.0 / E] * E
    if m["zipf"]:
        p = [r ** -gmoe.ZIPF_S for r in range(1, E + 1)]
        p = [v / sum(p) for v in p]
    return sum(1 - (1 - min(1.0, K * v)) ** T for v in p)


def _q8_bytes(rows, cols, gs, scale_bytes=4):
    return rows * cols * (1 + scale_bytes / gs)


def work(case):
    """Each touched weight, the cache and the activations once; multiply-adds as two."""
    m = _moe(case)
    D, F, E, K, gs = m["D"], m["F"], m["E"], m["K"], m["gs"]
    expert = 3 * _q8_bytes(F, D, gs, 2 if gs == 32 else 4)

    def moe(T):
        return (_touched(m, T) + 1) * expert + 4 * E * D + 8 * T * D, 2 * T * (3 * F * D * (K + 1) + E * D)

    if case["op"] in ("moe", "hook"):
        b, f = moe(case["T"])
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    c = _dense(case)
    H, kv, rope, ql, V = c["n_heads"], c["kv_lora_rank"], c["rope_dim"], c["q_lora_rank"], c["vocab_size"]
    n, pos = (case["n"], case["pos"]) if case["op"] == "prefill" else (1, case["pos"])
    mats = [(ql, D), (kv + rope, D), (H * c["head_k_dim"], ql), (H * kv, c["qk_nope_dim"]),
            (H * c["v_head_dim"], kv), (D, H * c["v_head_dim"])]
    pairs = n * pos + n * (n + 1) // 2  # (token, position) pairs of the causal attention
    b = sum(_q8_bytes(r, k, gs) for r, k in mats) + 4 * (pos + n) * (kv + rope)
    f = 2 * n * sum(r * k for r, k in mats) + 2 * pairs * H * (2 * kv + rope)
    mb, mf = moe(n)
    b, f = b * c["n_layers"] + mb * (c["n_layers"] - 1), f * c["n_layers"] + mf * (c["n_layers"] - 1)
    l0 = 3 * c["hidden_dim"] * D
    return {"bytes": b + _q8_bytes(3 * c["hidden_dim"], D, gs) + _q8_bytes(V, D, gs) + 4 * V,
            "flops": f + 2 * n * l0 + 2 * V * D}


def tolerance(case):
    # fp32 sums and 22-bit splits of the inputs: up to 2.3e-6 against 64 bits over 46 layers
    # (largest 1e-5 of the root mean square); a model at 4096 positions, whose softmax widens
    # its scores' rounding, up to 5e-5 (largest 2.5e-4). Four times these.
    if case["op"] in ("moe", "hook"):
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2e-4, "max": 1e-3}


# ---- the same in 64 bits -------------------------------------------------------------------


def _deq(q, s):
    return (q.double().unflatten(-1, (s.shape[-1], -1)) * s.double().unsqueeze(-1)).flatten(-2)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _ffn(x, gate, up, down):
    g, u = x @ _deq(*gate).T, x @ _deq(*up).T
    return (g * torch.sigmoid(g) * u) @ _deq(*down).T


def _moe_exact(x, m, ex, ro):
    xn = _rms(x, ro["ffn_norm"])
    p = torch.sigmoid(xn @ ro["gate_inp"].double().T)
    idx = torch.topk(p + ro["exp_probs_b"].double(), m["K"], -1).indices
    w = p.gather(1, idx)
    w = w / w.sum(-1, keepdim=True).clamp_min(MIN_DENOM)
    routed = torch.zeros_like(x)
    for e in idx.unique().tolist():
        t, k = (idx == e).nonzero(as_tuple=True)
        y = _ffn(xn[t], *[(ex[n + "_q"][e], ex[n + "_s"][e]) for n in ("gate", "up", "down")])
        routed.index_add_(0, t, ROUTED_SCALE * w[t, k].unsqueeze(1) * y)
    shared = _ffn(xn, *[(ex[n + "_sh_q"], ex[n + "_sh_s"]) for n in ("gate", "up", "down")])
    return {"x": x + (shared + routed), "xn": xn, "router_prob": p, "topk_idx": None, "topk_w": w,
            "shared_out": shared, "routed_out": routed}


def _rope(x, pos, rope):
    """Pairs (2i, 2i + 1) turned by glm.c's angles, which are defined in fp32."""
    i = np.arange(0, rope, 2, dtype=np.float32)
    freq = np.power(np.float32(1e6), -(i / np.float32(rope)))
    ang = torch.from_numpy(pos.astype(np.float32)[:, None] * freq[None, :]).to(DEV).double()
    c, s = ang.cos(), ang.sin()
    while c.dim() < x.dim():
        c, s = c.unsqueeze(1), s.unsqueeze(1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)


def _attention_exact(x, c, a):
    n, H, kv, rope, nope = x.shape[0], c["n_heads"], c["kv_lora_rank"], c["rope_dim"], c["qk_nope_dim"]
    w = {k: _deq(a[k + "_q"], a[k + "_s"]) for k in ("q_a", "q_b", "kv_a", "k_b", "v_b", "attn_out")}
    xn, pos = _rms(x, a["attn_norm"]), np.arange(n)
    kva = xn @ w["kv_a"].T
    comp, pe = _rms(kva[:, :kv], a["kv_a_norm"]), _rope(kva[:, kv:], pos, rope)
    q = (_rms(xn @ w["q_a"].T, a["q_a_norm"]) @ w["q_b"].T).unflatten(1, (H, -1))
    q_pe = _rope(q[..., nope:], pos, rope)
    k_b, v_b = w["k_b"].unflatten(0, (H, kv)), w["v_b"].unflatten(0, (H, -1))
    heads = []
    for h in range(H):
        parts = []
        for t in range(0, n, 1024):
            u = min(n, t + 1024)
            s = (q[t:u, h, :nope] @ k_b[h].T) @ comp[:u].T + q_pe[t:u, h] @ pe[:u].T
            later = torch.arange(u, device=DEV)[None, :] > torch.arange(t, u, device=DEV)[:, None]
            s = (s / math.sqrt(c["head_k_dim"])).masked_fill(later, -math.inf).softmax(-1)
            parts.append((s @ comp[:u]) @ v_b[h].T)
        heads.append(torch.cat(parts))
    return x + torch.cat(heads, 1) @ w["attn_out"].T


def exact(case, seed):
    m = _moe(case)
    ex = _experts(m)
    if case["op"] in ("moe", "hook"):
        x, outs = _activations(case, m, seed).double(), []
        for layer in range(1, case["layers"] + 1):
            outs.append(_moe_exact(x, m, ex, _router(m, layer)))
            x = outs[-1]["x"]
        return x if case["op"] == "moe" else outs
    c = _dense(case)
    n = case["pos"] + (case["n"] if case["op"] == "prefill" else 1)
    top, layers = _dense_weights(c)
    t = torch.from_numpy(_tokens(n, c["vocab_size"], seed)).to(DEV).long()
    x = _deq(top["tok_q"][t], top["tok_s"][t])
    for layer, a in enumerate(layers):
        x = _attention_exact(x, c, a)
        if layer == 0:
            mats = [(top["l0_ffn_" + k + "_q"], top["l0_ffn_" + k + "_s"]) for k in ("gate", "up", "down")]
            x = x + _ffn(_rms(x, top["l0_ffn_norm"]), *mats)
        else:
            x = _moe_exact(x, m, ex, _router(m, layer))["x"]
    x = _rms(x[-1:], top["output_norm"])
    return torch.cat([x @ _deq(top["out_q"][r:r + 16384], top["out_s"][r:r + 16384]).T
                      for r in range(0, c["vocab_size"], 16384)], 1)[0]
