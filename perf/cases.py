"""What is measured: the MoE block and the calls around it, as a host program makes them.

A case is one call (or the one short sequence of calls) of a user's program through the public entry
points, on inputs that are in place before it:

  layer     rbt_hip_moe_dev on device pointers: one MoE block over T tokens. A decode step has T = 1, a
            step of several sequences T = their number, a prompt chunk T = its length.
  seam      rbt_hip_moe on host pointers: the call that the patched engine makes per token and layer.
  prompt    rbt_hip_generate over a prompt without generated tokens, then rbt_hip_forward of the
            prompt's last token: a prompt read in, up to the logits that follow it.
  generate  rbt_hip_generate of a short answer, then one rbt_hip_forward behind it: a whole greedy call.

The full layer shape is the one the benchmark runs (dim 2048, 64 experts, top-8, hidden 1024, 16 layers,
vocabulary 50304); the odd shapes are generic. Weights are N(0, 0.02) as in the benchmark, except where
small dims would leave no signal (scaled by the fan-in); activations N(0, 1) in f32, as an RMSNorm leaves
them. Skewed calls add 2.0 to the router logits of eight experts, as the benchmark's skewed leg does.
"""
import ctypes as C
import math

import numpy as np
import torch

from rabbitm2_amd import hip

FULL = {"D": 2048, "E": 64, "K": 8, "H": 1024}
MODEL = {"layers": 16, "heads": 16, "hd": 128, "vocab": 50304, "eps": 1e-5, "theta": 10000.0}
_handle = []


def listed():
    layer = dict(FULL, kind="layer", dtype="bf16", order="avx2", skew=False, renorm=True)
    return [
        # one token of one sequence: the call of every decode step, the smallest one on the full shape
        dict(layer, name="decode-1", T=1),
        # a handful of tokens: a few sequences stepped together, or drafted tokens checked at once
        dict(layer, name="few-5", T=5),
        # one step of a batch of sequences
        dict(layer, name="batch-32", T=32),
        # a prompt chunk, evenly routed
        dict(layer, name="prefill-512", T=512),
        # a ragged prompt whose tokens crowd onto eight experts, weights not renormalised
        dict(layer, name="skewed-777", T=777, skew=True, renorm=False),
        # the longest prompt that the model's positions allow, in one call
        dict(layer, name="prefill-4096", T=4096),
        # a prompt in the engine's default arithmetic: its scalar summation order, f32 weights
        dict(layer, name="f32-prefill-200", T=200, dtype="f32", order="scalar"),
        # one token in the same arithmetic
        dict(layer, name="f32-decode-1", T=1, dtype="f32", order="scalar"),
        # a small model with sizes that no tile divides
        dict(layer, name="odd-50", T=50, D=1000, E=20, K=3, H=330, renorm=False),
        # the engine's own call: one token, host pointers, waits for its result
        {"name": "seam-1", "kind": "seam", "T": 1},
        # a prompt through the whole model to the logits behind it
        {"name": "prompt-400", "kind": "prompt", "n": 400},
        # a short prompt and a short greedy answer
        {"name": "generate-24+40", "kind": "generate", "n": 24, "gen": 40},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choices(["full", "f32", "odd", "seam", "prompt", "generate"], [8, 3, 3, 1, 2, 1])[0]
    if kind == "seam":
        return {"kind": "seam", "T": _log(rng, 1, 64)}
    if kind == "prompt":
        return {"kind": "prompt", "n": _log(rng, 20, 400)}
    if kind == "generate":
        return {"kind": "generate", "n": rng.randint(8, 40), "gen": rng.randint(8, 40)}
    c = dict(FULL, kind="layer", dtype="bf16", order=rng.choice(["avx2", "avx2", "avx2", "scalar"]),
             skew=rng.random() < 0.3, renorm=rng.random() < 0.5)
    if kind == "full":
        c["T"] = _log(rng, 1, 4096)
    elif kind == "f32":
        c.update(T=_log(rng, 1, 200), dtype="f32", order=rng.choice(["avx2", "scalar"]))
    else:
        E = rng.randint(8, 64)
        c.update(D=4 * _log(rng, 16, 500), E=E, K=rng.randint(1, 8), H=_log(rng, 40, 1000), T=_log(rng, 1, 1000),
                 dtype=rng.choice(["bf16", "bf16", "f32"]))
    return c


# ---- inputs
_DT = {"bf16": (hip.DT_BF16, torch.bfloat16, 2), "f32": (hip.DT_F32, torch.float32, 4)}


def _normal(seed, stream, shape, scale, dtype=torch.float32):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + stream) % (1 << 62))
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, scale, generator=g)


def _layer_weights(case, seed, base=0):
    """(router [E][D], expert blobs [E][stride in elements]) of one layer in the file's layout."""
    D, E, H = case["D"], case["E"], case["H"]
    _, dt, esz = _DT[case["dtype"]]
    full = D == FULL["D"] and H == FULL["H"]
    stride = (3 * H * D * esz + 4095) // 4096 * 4096
    router = _normal(seed, base + 1, (E, D), 0.02 if full else 1.0 / math.sqrt(D), dt)
    experts = _normal(seed, base + 2, (E, stride // esz), 0.02 if full else 1.0 / math.sqrt(D), dt)
    return router, experts, stride


def _bias(case):
    if not case["skew"]:
        return None
    b = torch.zeros(case["E"], device="cuda")
    b[:8] = 2.0
    return b


def _layer_x(case, seed):
    return _normal(seed, 3, (case["T"], case["D"]), 1.0)


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _prepare_layer(case, seed):
    if not _handle:
        _handle.append(hip.Device(0))  # one handle per program, as the engine has
    dev = _handle[0]
    T, D, K = case["T"], case["D"], case["K"]
    router, experts, stride = _layer_weights(case, seed)
    bias, x = _bias(case), _layer_x(case, seed)
    desc = hip.moe_layer_desc(D, case["E"], K, case["H"], _DT[case["dtype"]][0], int(case["renorm"]), _ptr(router),
                              _ptr(experts), stride, None if bias is None else _ptr(bias))
    dev.reserve(desc, T)
    out = (torch.empty((T, D), device="cuda"), torch.empty((T, K), dtype=torch.int32, device="cuda"),
           torch.empty((T, K), device="cuda"))
    torch.cuda.synchronize()  # the handle has a stream of its own
    order = hip.ORDER_SCALAR if case["order"] == "scalar" else hip.ORDER_AVX2
    return {"kind": "layer", "dev": dev, "order": order, "desc": desc, "keep": (router, experts, bias, x), "T": T,
            "ptr": [_ptr(x)] + [_ptr(o) for o in out], "out": out}


class _Image:
    """The model image of a handle as a tensor of bytes."""

    def __init__(self, ptr, nbytes):
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 2}


class _Model:
    """A handle that holds a random model; the handle goes with it."""

    def __init__(self, layers, vocab, seed):
        m, f = MODEL, FULL
        cfg = hip.Config(vocab=vocab, dim=f["D"], n_layers=layers, n_heads=m["heads"], n_kv_heads=m["heads"],
                         head_dim=m["hd"], n_experts=f["E"], top_k=f["K"], expert_hidden=f["H"], max_seq=4096,
                         dtype=hip.DT_BF16, qk_norm=1, norm_topk=0, rope_theta=m["theta"], rms_eps=m["eps"])
        self.dev = hip.Device(0)
        base = self.dev.model_create(cfg)
        last, n = self.dev.tensor("lm_head")
        image = torch.as_tensor(_Image(base.value, last + n), device="cuda")
        for name, layer, t in _model_weights(layers, vocab, seed):
            off, n = self.dev.tensor(name, layer)
            image[off:off + n].view(t.dtype).copy_(t.reshape(-1))
        torch.cuda.synchronize()

    def __del__(self):
        if getattr(self, "dev", None) is not None:
            self.dev.close()


def _model_weights(layers, vocab, seed):
    """(name, layer, values) of every tensor; norms are ones."""
    D, qd = FULL["D"], MODEL["heads"] * MODEL["hd"]
    case = dict(FULL, dtype="bf16")
    yield "tok_emb", 0, _normal(seed, 11, (vocab, D), 0.02, torch.bfloat16)
    for l in range(layers):
        for name, n in (("attn_norm", D), ("q_norm", qd), ("k_norm", qd), ("ffn_norm", D)):
            yield name, l, torch.ones(n, device="cuda")
        for i, (name, shape) in enumerate((("wq", (qd, D)), ("wk", (qd, D)), ("wv", (qd, D)), ("wo", (D, qd)))):
            yield name, l, _normal(seed, 100 * (l + 1) + i, shape, 0.02, torch.bfloat16)
        router, experts, _ = _layer_weights(case, seed, 100 * (l + 1) + 10)
        yield "router", l, router
        yield "experts", l, experts
    yield "final_norm", 0, torch.ones(D, device="cuda")
    yield "lm_head", 0, _normal(seed, 12, (vocab, D), 0.02, torch.bfloat16)


def _tokens(n, seed):
    return np.random.RandomState(seed % (1 << 31)).randint(0, MODEL["vocab"], n).astype(np.int32)


def prepare(case, seed):
    if case["kind"] == "layer":
        return _prepare_layer(case, seed)
    if case["kind"] == "seam":
        r = np.random.RandomState(seed % (1 << 31))
        xb, x = (r.standard_normal((case["T"], FULL["D"])).astype(np.float32) for _ in range(2))
        return {"kind": "seam", "model": _Model(1, 256, seed), "xb": xb, "x": x}
    m = _Model(MODEL["layers"], MODEL["vocab"], seed)
    m.dev.state_init(512)  # the engine's default context
    return dict(case, model=m, tokens=_tokens(case["n"], seed))


# ---- the calls
def run(state):
    kind = state["kind"]
    if kind == "layer":
        dev, p = state["dev"], state["ptr"]
        dev.set_router_order(state["order"])
        dev.moe_dev(state["desc"], p[0], state["T"], moe=p[1], routing=p[2], weights=p[3])
        return state["out"]
    dev = state["model"].dev
    if kind == "seam":
        return dev.moe(0, state["xb"], state["x"])
    tokens, n = state["tokens"], state["n"]
    if kind == "prompt":
        dev.generate(tokens, 0)
        logits, routing = dev.forward(tokens[-1], n - 1, MODEL["vocab"], MODEL["layers"], FULL["K"])
        return logits, routing
    ids, _ = dev.generate(tokens, state["gen"])
    logits, _ = dev.forward(ids[-1], n + state["gen"] - 1, MODEL["vocab"], MODEL["layers"], FULL["K"])
    return np.array(ids, np.int32), logits


# ---- what a pass cannot do without
def _touched(case, T):
    """Experts that T tokens are expected to select (each weight read once)."""
    E, K = case["E"], case["K"]
    p = [K / E] * E
    if case.get("skew") and E > 8:
        hot = 8 * 7.39 / (8 * 7.39 + E - 8)  # the eight experts' share of a softmax with +2.0
        p = [min(1.0, K * hot / 8)] * 8 + [min(1.0, max(K - 8 * min(1.0, K * hot / 8), K * (1 - hot)) / (E - 8))] * (E - 8)
    return sum(1.0 - (1.0 - q) ** T for q in p)


def _layer_work(case, T):
    D, E, K, H = (case[k] for k in "DEKH")
    esz = _DT[case["dtype"]][2]
    return {"bytes": E * D * esz + _touched(case, T) * 3 * H * D * esz + 8.0 * T * D + 8.0 * T * K,
            "flops": 2.0 * T * (E * D + 3.0 * K * H * D)}


def _model_work(n, steps):
    """n positions read in as one block, then `steps` tokens one after the other, each with its logits."""
    D, qd, V, L = FULL["D"], MODEL["heads"] * MODEL["hd"], MODEL["vocab"], MODEL["layers"]
    case = dict(FULL, dtype="bf16")
    dense, one, many = 4 * D * qd, _layer_work(case, 1), _layer_work(case, max(n, 1))
    by = fl = 0.0
    if n:
        by += L * (2 * dense + many["bytes"] + 16 * n * qd)
        fl += L * (2.0 * dense * n + many["flops"] + 2.0 * n * n * qd)
    by += steps * (L * (2 * dense + one["bytes"] + 8.0 * (n + steps / 2) * qd) + 2.0 * V * D)
    fl += steps * (L * (2.0 * dense + one["flops"] + 4.0 * (n + steps / 2) * qd) + 2.0 * V * D)
    return {"bytes": by, "flops": fl}


def work(case):
    if case["kind"] == "layer":
        return _layer_work(case, case["T"])
    if case["kind"] == "seam":
        w = _layer_work(dict(FULL, dtype="bf16"), case["T"])
        return {"bytes": w["bytes"] + 4.0 * case["T"] * FULL["D"], "flops": w["flops"]}
    if case["kind"] == "prompt":
        return _model_work(case["n"] - 1, 1)
    return _model_work(case["n"] - 1, case["gen"] + 1)


def tolerance(case):
    """Four times the distance seen between the path and its value in 64 bits: 4.4e-6 where a batch's
    activations are multiplied as two bf16 parts (bf16 weights), 4.9e-7 with f32 products, 3.1e-8 of the
    residual rows. The whole calls are 2.7e-7 away, but a rounding there can swap two nearly equal
    experts of one of several thousand (token, layer) choices, which moves the last logits by up to
    about 1e-4."""
    if case["kind"] == "layer":
        return {"rel": 2e-5, "max": 4e-4} if case["dtype"] == "bf16" else {"rel": 2e-6, "max": 1e-4}
    if case["kind"] == "seam":
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 1e-4, "max": 2e-3, "differ": 0.01}


# ---- the same in 64 bits
def _moe64(x, router, experts, bias, D, H, K, renorm):
    """(moe [T][D], routing [T][K], weights [T][K]) for f64 rows x."""
    logits = x @ router.double().T
    if bias is not None:
        logits = logits + bias.double()
    p = torch.softmax(logits, 1)
    w, idx = torch.sort(p, dim=1, descending=True, stable=True)
    w, idx = w[:, :K], idx[:, :K]
    if renorm:
        w = w / w.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, k = torch.nonzero(idx == e, as_tuple=True)
        b = experts[e].double()
        w1, w3, w2 = b[:H * D].view(H, D), b[H * D:2 * H * D].view(H, D), b[2 * H * D:3 * H * D].view(D, H)
        g = x[t] @ w1.T
        h = g / (1.0 + torch.exp(-g)) * (x[t] @ w3.T)
        out.index_add_(0, t, w[t, k].unsqueeze(1) * (h @ w2.T))
    return out, idx.to(torch.int32), w


def _norm64(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


class _Model64:
    """The whole forward pass in 64 bits over blocks of new positions, with its own cache."""

    def __init__(self, seed):
        self.w = {(name, l): t for name, l, t in _model_weights(MODEL["layers"], MODEL["vocab"], seed)}
        self.k, self.v = [[] for _ in range(MODEL["layers"])], [[] for _ in range(MODEL["layers"])]
        self.pos = 0

    def _rope(self, x, pos):
        hd = MODEL["hd"]
        f = MODEL["theta"] ** (-2.0 * torch.arange(hd // 2, dtype=torch.float64, device="cuda") / hd)
        a = pos.double().unsqueeze(1) * f
        c, s = torch.cos(a).unsqueeze(1), torch.sin(a).unsqueeze(1)
        lo, hi = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat((lo * c - hi * s, hi * c + lo * s), -1)

    def step(self, tokens):
        """Runs the tokens at the next positions; the last one's (logits, routing [layers][K])."""
        n, nh, hd, eps, w = len(tokens), MODEL["heads"], MODEL["hd"], MODEL["eps"], self.w
        pos = torch.arange(self.pos, self.pos + n, device="cuda")
        x = w["tok_emb", 0][torch.as_tensor(tokens, device="cuda").long()].double()
        routing = []
        for l in range(MODEL["layers"]):
            xb = _norm64(x, eps)
            q, k, v = (xb @ w[name, l].double().T for name in ("wq", "wk", "wv"))
            q, k = (self._rope(_norm64(t, eps).view(n, nh, hd), pos) for t in (q, k))
            self.k[l].append(k)
            self.v[l].append(v.view(n, nh, hd))
            ks, vs = torch.cat(self.k[l]), torch.cat(self.v[l])
            s = torch.matmul(q.transpose(0, 1), ks.permute(1, 2, 0).contiguous()) / math.sqrt(hd)
            s = s.masked_fill(torch.arange(len(ks), device="cuda") > pos.view(-1, 1), -math.inf)
            ao = torch.matmul(torch.softmax(s, -1), vs.transpose(0, 1).contiguous()).transpose(0, 1).reshape(n, nh * hd)
            x = x + ao @ w["wo", l].double().T
            moe, idx, _ = _moe64(_norm64(x, eps), w["router", l], w["experts", l], None, FULL["D"], FULL["H"],
                                 FULL["K"], False)
            x = x + moe
            routing.append(idx[-1])
        self.pos += n
        return w["lm_head", 0].double() @ _norm64(x[-1], eps), torch.stack(routing)


def exact(case, seed):
    if case["kind"] == "layer":
        router, experts, _ = _layer_weights(case, seed)
        return _moe64(_layer_x(case, seed).double(), router, experts, _bias(case), case["D"], case["H"], case["K"],
                      case["renorm"])
    if case["kind"] == "seam":
        r = np.random.RandomState(seed % (1 << 31))
        xb, x = (r.standard_normal((case["T"], FULL["D"])).astype(np.float32) for _ in range(2))
        router, experts = (t for name, _, t in _model_weights(1, 256, seed) if name in ("router", "experts"))
        moe, idx, _ = _moe64(torch.as_tensor(xb, device="cuda").double(), router, experts, None, FULL["D"], FULL["H"],
                             FULL["K"], False)
        return torch.as_tensor(x, device="cuda").double() + moe, idx
    tokens, m = _tokens(case["n"], seed), _Model64(seed)
    logits, routing = m.step(tokens)
    if case["kind"] == "prompt":
        return logits, routing
    ids = [int(logits.argmax())]
    while len(ids) < case["gen"]:
        ids.append(int(m.step(ids[-1:])[0].argmax()))
    return np.array(ids, np.int32), m.step(ids[-1:])[0]
