"""Performance cases of the CIS-2 forward pass: what programs ask of it
through the package's Python interface, from one matrix-vector product to a
4096-token prompt.

Every result is pinned bit for bit by the CIS-2 arithmetic, so every
tolerance is "exact".  Shapes are the SmolLM2-135M, llama-160m and
Qwen3-0.6B configurations; weights are random bf16 of those shapes, norm
weights near one.  A case is one of

  gemv    a strict-order matrix-vector product on host vectors (batch > 0:
          that many products of independent matrices in one call)
  token   one position for each of `seqs` sequences whose caches hold `pos`
          earlier positions: logits and greedy ids
  decode  one sequence: prompt, then `gen` tokens (greedy, or drawn with a
          seed where temperature > 0) with the witness, and the logits at
          the last position
  batch   `seqs` ragged prompts decoded together for `gen` tokens, and
          each sequence's logits at its last position
  verify  the teacher-forced check of a claimed continuation: its logits,
          ids and digests
"""
import hashlib
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cis2-lab-archive_amd"))

from cis2amd import Cis2Model, GemvPlan  # noqa: E402
from cis2amd.artifacts import ModelSpec  # noqa: E402

# hidden, inter, layers, heads, kv heads, head_dim, vocab, eps, theta, tied, qk norm
SHAPES = {
    "smollm2": (576, 1536, 30, 9, 3, 64, 49152, 1e-5, 100000.0, True, False),
    "llama160m": (768, 3072, 12, 12, 12, 64, 32000, 1e-6, 10000.0, False, False),
    "qwen3": (1024, 3072, 28, 16, 8, 128, 151936, 1e-6, 1000000.0, True, True),
}


def gemv(name, m, k, batch=0):
    return {"name": name, "kind": "gemv", "m": m, "k": k, "batch": batch}


def token(name, model, seqs, pos, tree=False):
    return {"name": name, "kind": "token", "model": model, "seqs": seqs, "pos": pos, "tree": tree}


def decode(name, model, prompt, gen, tree=False, temperature=0.0, top_k=0, top_p=1.0):
    return {"name": name, "kind": "decode", "model": model, "prompt": prompt, "gen": gen,
            "tree": tree, "temperature": temperature, "top_k": top_k, "top_p": top_p}


def batch(name, model, seqs, lo, hi, gen, tree=False):
    return {"name": name, "kind": "batch", "model": model, "seqs": seqs, "lo": lo, "hi": hi,
            "gen": gen, "tree": tree}


def verify(name, model, prompt, gen, tree=False):
    return {"name": name, "kind": "verify", "model": model, "prompt": prompt, "gen": gen,
            "tree": tree}


def listed():
    return [
        # one pinned-order product, the unit the kernel labs measure: launch and copies count
        gemv("gemv", 1536, 576),
        # a vocabulary projection by itself: HBM counts
        gemv("gemv_head", 49152, 576),
        # a host that drives the model one position at a time and does its own sampling
        token("token", "smollm2", 1, 160),
        # a short chat answer with its receipt
        decode("decode", "smollm2", 32, 64),
        # the same answer in the tree order
        decode("decode_tree", "smollm2", 32, 64, tree=True),
        # the same answer drawn with a seed at the settings the sampling draft gives
        decode("decode_sampled", "smollm2", 32, 32, temperature=0.8, top_k=40, top_p=0.95),
        # a few users served together
        batch("batch8", "smollm2", 8, 16, 64, 32),
        # a full serving batch with ragged prompts
        batch("batch64", "smollm2", 64, 16, 512, 32),
        # a prompt set of the second model run as one batch
        batch("batch_set", "llama160m", 300, 8, 64, 16),
        # a receipt checked in one pass: a long prompt and a short claimed answer
        verify("verify", "smollm2", 512, 33),
        # a receipt of the tree order
        verify("verify_tree", "smollm2", 61, 64, tree=True),
        # a long context: a 4096-token prompt, then its first tokens
        decode("long_context", "qwen3", 4096, 32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    case = _drawn(rng)
    del case["name"]
    return case


def _drawn(rng):
    kind = rng.choice(["gemv", "token", "decode", "batch", "verify"])
    if kind == "gemv":
        m, k = _log(rng, 16, 49152), 4 * _log(rng, 16, 560)
        most = max(1, 64_000_000 // (m * k))
        return gemv("", m, k, rng.choice([0, min(most, _log(rng, 2, 128))]))
    tree = rng.random() < 0.3
    model = rng.choice(["smollm2", "smollm2", "llama160m", "qwen3"])
    if kind == "token":
        n = _log(rng, 1, 64)
        return token("", model, n, _log(rng, 4, min(500, 8192 // n)), tree)
    if kind == "decode":
        if rng.random() < 0.3:
            return decode("", model, _log(rng, 4, 512), _log(rng, 4, 32), tree,
                          round(rng.uniform(0.5, 1.5), 2), rng.choice([0, 40, 1000]),
                          round(rng.uniform(0.5, 0.99), 2))
        long = model == "qwen3" and not tree
        return decode("", model, _log(rng, 1, 4000 if long else 512), _log(rng, 4, 48), tree)
    if kind == "batch":
        lo = _log(rng, 2, 64)
        model = rng.choice(["smollm2", "llama160m"])
        return batch("", model, _log(rng, 2, 300 if model == "llama160m" else 64), lo,
                     lo + _log(rng, 1, 128), _log(rng, 2, 24), tree)
    return verify("", model, _log(rng, 1, 2000 if model == "qwen3" and not tree else 700),
                  _log(rng, 1, 64), tree)


# ---- inputs ----------------------------------------------------------------

def _tensors(model):
    """(name, shape) of a shape's checkpoint tensors."""
    h, inter, layers, nh, nkv, hd, vocab, _, _, tied, qk = SHAPES[model]
    out = [("model.embed_tokens.weight", (vocab, h))]
    for i in range(layers):
        p = "model.layers.%d." % i
        out += [(p + "input_layernorm.weight", (h,)), (p + "post_attention_layernorm.weight", (h,)),
                (p + "self_attn.q_proj.weight", (nh * hd, h)),
                (p + "self_attn.k_proj.weight", (nkv * hd, h)),
                (p + "self_attn.v_proj.weight", (nkv * hd, h)),
                (p + "self_attn.o_proj.weight", (h, nh * hd)),
                (p + "mlp.gate_proj.weight", (inter, h)), (p + "mlp.up_proj.weight", (inter, h)),
                (p + "mlp.down_proj.weight", (h, inter))]
        if qk:
            out += [(p + "self_attn.q_norm.weight", (hd,)), (p + "self_attn.k_norm.weight", (hd,))]
    out.append(("model.norm.weight", (h,)))
    if not tied:
        out.append(("lm_head.weight", (vocab, h)))
    return out


def _weights(model, seed):
    """{name: bf16 tensor on the GPU}: N(0, 0.02), norm weights 1 + N(0, 0.1)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    shapes = _tensors(model)
    flat = torch.empty(sum(math.prod(s) for _, s in shapes), dtype=torch.bfloat16, device="cuda")
    flat.normal_(0.0, 0.02, generator=g)
    out, at = {}, 0
    for name, shape in shapes:
        n = math.prod(shape)
        t = flat[at:at + n]
        if name.endswith("norm.weight"):
            t.copy_(1.0 + 5.0 * t.float())
        out[name] = t.view(shape)
        at += n
    return out, flat


class Checkpoint:
    """What Cis2Model reads of a checkpoint: bf16 tensors and file digests."""

    def __init__(self, model, seed):
        named, flat = _weights(model, seed)
        host = flat.view(torch.int16).cpu().numpy().view(np.uint16)
        self.tensors, at = [], 0
        for name, t in named.items():
            self.tensors.append((name, tuple(t.shape), host[at:at + t.numel()]))
            at += t.numel()
        self.digest = hashlib.sha256(("%s %d" % (model, seed)).encode()).digest()

    def header_digests(self):
        return self.digest * 3


def _model(case, seed, max_pos, max_seqs=1):
    h, inter, layers, nh, nkv, hd, vocab, eps, theta, tied, qk = SHAPES[case["model"]]
    spec = ModelSpec(case["model"], h, inter, layers, nh, nkv, vocab, eps, theta, tied,
                     head_dim=hd, qk_norm=qk)
    m = Cis2Model(spec, Checkpoint(case["model"], seed), max_pos, max_seqs,
                  reduction_mode=1 if case["tree"] else 0)
    m.weights = None  # uploaded: the host copy is not needed any more
    return m


def _ids(case, seed, *shape):
    rng = np.random.default_rng([seed, 7])
    return rng.integers(0, SHAPES[case["model"]][6], shape).astype(np.uint32)


def _lengths(case):
    # the same for every seed, so that outputs keep their shapes
    return np.random.default_rng(8).integers(case["lo"], case["hi"] + 1, case["seqs"])


def _gemv_inputs(case, seed):
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((case["m"], case["k"]), dtype=np.float32) * np.float32(0.02)
    x = rng.standard_normal((max(1, case["batch"]), case["k"]), dtype=np.float32)
    return w, x


def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        w, x = _gemv_inputs(case, seed)
        return {"case": case, "plan": GemvPlan(w, copies=max(1, min(case["batch"], 8))),
                "x": x if case["batch"] else x[0]}
    if kind == "token":
        n, pos = case["seqs"], case["pos"]
        m = _model(case, seed, pos + 8, n)
        ids = _ids(case, seed, n, pos + 1)
        # the caches as a program has them after its prompts
        m.forward_rows(np.repeat(np.arange(n), pos), np.tile(np.arange(pos), n),
                       ids[:, :pos].reshape(-1)[:n * pos], want_logits=False)
        return {"case": case, "m": m, "seq": np.arange(n, dtype=np.uint32),
                "pos": np.full(n, pos, np.uint32), "tok": np.ascontiguousarray(ids[:, pos])}
    if kind == "decode":
        m = _model(case, seed, case["prompt"] + case["gen"])
        if case["temperature"] > 0:
            m.set_sampling(seed, np.float32(case["temperature"]), case["top_k"],
                           np.float32(case["top_p"]))
        return {"case": case, "m": m, "prompt": _ids(case, seed, case["prompt"])}
    if kind == "batch":
        lens = _lengths(case)
        m = _model(case, seed, int(lens.max()) + case["gen"], case["seqs"])
        ids = _ids(case, seed, int(lens.sum()))
        return {"case": case, "m": m, "lens": lens,
                "prompts": np.split(ids, np.cumsum(lens)[:-1])}
    m = _model(case, seed, case["prompt"] + case["gen"])
    ids = _ids(case, seed, case["prompt"] + case["gen"])
    return {"case": case, "m": m, "prompt": ids[:case["prompt"]], "claimed": ids[case["prompt"]:]}


def _bytes(*hexes):
    return np.frombuffer(bytes.fromhex("".join(hexes)), np.uint8)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemv":
        p = state["plan"]
        return p.run_batch(state["x"]) if case["batch"] else p(state["x"])
    m = state["m"]
    if kind == "token":
        if case["seqs"] == 1:
            logits, arg = m.forward_token(int(state["pos"][0]), int(state["tok"][0]))
            return {"logits": logits[None], "ids": np.array([arg], np.uint32)}
        logits, arg = m.forward_rows(state["seq"], state["pos"], state["tok"])
        return {"logits": logits, "ids": arg}
    if kind == "decode":
        r = m.decode(state["prompt"], case["gen"])
        last = r["ids"].size - 1
        logits, _ = m.forward_token(last, int(r["ids"][last]))
        return {"ids": r["ids"], "digests": _bytes(r["witness"], r["argmax_digest"]),
                "steps": _bytes(*r["step_digests"]), "logits": logits}
    if kind == "batch":
        rows = m.decode_batch(state["prompts"], case["gen"])
        last = state["lens"] + case["gen"] - 1
        logits, _ = m.forward_rows(np.arange(len(rows)), last, [r["ids"][-1] for r in rows])
        return {"ids": np.concatenate([r["ids"] for r in rows]),
                "digests": _bytes(*[r[k] for r in rows for k in ("witness", "argmax_digest")]),
                "logits": logits}
    r = m.verify_prefill(state["prompt"], state["claimed"], want_logits=True)
    return {"logits": r["logits"], "ids": r["generated"],
            "digests": _bytes(r["witness"], r["argmax_digest"]),
            "first": np.array([r["first_mismatch"]], np.int64)}


# ---- what a pass cannot do without -----------------------------------------

def _layer_weights(model):
    h, inter, layers, nh, nkv, hd = SHAPES[model][:6]
    return layers * (2 * h * nh * hd + 2 * h * nkv * hd + 3 * h * inter)


def _pass(model, spans, logit_rows):
    """Bytes and operations of one forward pass in f32: every weight once, the
    cached K and V rows each sequence attends to once and its new ones, the
    logits.  spans: (first position, rows) of each sequence."""
    h, _, layers, nh, nkv, hd, vocab = SHAPES[model][:7]
    rows = sum(n for _, n in spans)
    pairs = sum(n * p + n * (n + 1) // 2 for p, n in spans)
    lw, head = _layer_weights(model), (vocab * h if logit_rows else 0)
    kv = 8 * nkv * hd * layers * sum(p + n for p, n in spans)
    return (4 * (lw + head) + kv + 4 * vocab * logit_rows,
            2 * (lw * rows + head * logit_rows + 2 * nh * hd * layers * pairs))


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n, m, k = max(1, case["batch"]), case["m"], case["k"]
        return {"bytes": 4 * (min(n, 8) * m * k + n * (m + k)), "flops": 2 * n * m * k}
    model = case["model"]
    if kind == "token":
        passes = [_pass(model, [(case["pos"], 1)] * case["seqs"], case["seqs"])]
    elif kind == "decode":
        p, g = case["prompt"], case["gen"]
        passes = [_pass(model, [(0, p)], 1)] + [_pass(model, [(p + i, 1)], 1) for i in range(g)]
    elif kind == "batch":
        lens, g = [int(n) for n in _lengths(case)], case["gen"]
        passes = [_pass(model, [(0, n) for n in lens], len(lens))]
        passes += [_pass(model, [(n + i, 1) for n in lens], len(lens)) for i in range(g)]
    else:
        passes = [_pass(model, [(0, case["prompt"] + case["gen"] - 1)], case["gen"])]
    return {"bytes": sum(b for b, _ in passes), "flops": sum(f for _, f in passes)}


def tolerance(case):
    # the arithmetic pins every rounding and every order of additions, so two
    # correct implementations agree in every bit
    return "exact"


# ---- the same in 64 bits ---------------------------------------------------

def _forward64(model, seed, ids, logit_from):
    """f64 logits at positions logit_from.. of each row of ids [n][t], causal
    within the row; the arithmetic of the decoder in plain torch."""
    h, _, layers, nh, nkv, hd, vocab, eps, theta, tied, qk = SHAPES[model]
    w, _ = _weights(model, seed)
    eps = float(np.float32(eps))
    n, t = ids.shape

    def f(name):
        return w[name].double()

    def norm(x, g):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * g

    tok = torch.from_numpy(ids.astype(np.int64)).cuda()
    x = w["model.embed_tokens.weight"][tok].double()
    inv = float(np.float32(theta)) ** (-torch.arange(0, hd, 2, device="cuda").double() / hd)
    ang = torch.arange(t, device="cuda").double()[:, None] * inv
    cos, sin = ang.cos()[None, :, None], ang.sin()[None, :, None]

    def rope(v):
        a, b = v[..., :hd // 2], v[..., hd // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    mask = torch.ones(t, t, dtype=torch.bool, device="cuda").triu(1)
    for i in range(layers):
        p = "model.layers.%d." % i
        y = norm(x, f(p + "input_layernorm.weight"))
        q = (y @ f(p + "self_attn.q_proj.weight").T).view(n, t, nh, hd)
        k = (y @ f(p + "self_attn.k_proj.weight").T).view(n, t, nkv, hd)
        v = (y @ f(p + "self_attn.v_proj.weight").T).view(n, t, nkv, hd)
        if qk:
            q = norm(q, f(p + "self_attn.q_norm.weight"))
            k = norm(k, f(p + "self_attn.k_norm.weight"))
        q, k = rope(q), rope(k)
        o = torch.empty_like(q)
        for r in range(n):
            for j in range(nh):
                s = q[r, :, j] @ k[r, :, j // (nh // nkv)].T / math.sqrt(hd)
                o[r, :, j] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ \
                    v[r, :, j // (nh // nkv)]
        x = x + o.view(n, t, nh * hd) @ f(p + "self_attn.o_proj.weight").T
        y = norm(x, f(p + "post_attention_layernorm.weight"))
        g = y @ f(p + "mlp.gate_proj.weight").T
        x = x + (g * torch.sigmoid(g) * (y @ f(p + "mlp.up_proj.weight").T)) @ \
            f(p + "mlp.down_proj.weight").T
    x = norm(x[:, logit_from:], f("model.norm.weight"))
    return x @ f("model.embed_tokens.weight" if tied else "lm_head.weight").T


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        w, x = _gemv_inputs(case, seed)
        y = x.astype(np.float64) @ w.astype(np.float64).T
        return y if case["batch"] else y[0]
    if kind == "token":
        if case["seqs"] * case["pos"] > 4096:
            return None
        ids = _ids(case, seed, case["seqs"], case["pos"] + 1)
        logits = _forward64(case["model"], seed, ids, case["pos"])
        return {"logits": logits[:, 0].cpu().numpy(), "ids": None}
    if kind == "verify":
        n, g = case["prompt"], case["gen"]
        ids = _ids(case, seed, n + g)
        logits = _forward64(case["model"], seed, ids[None, :n + g - 1], n - 1)
        return {"logits": logits[0].cpu().numpy(), "ids": None, "digests": None, "first": None}
    # the logits after a decode belong to the tokens that 32-bit rounding chose
    return None
