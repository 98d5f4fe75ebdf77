"""The work that a program has this engine do, as cases to be timed and compared.

Sizes are those of the repository's own workloads (a 16-id prompt with 32 tokens, a 128-id prompt,
a 1000-id prompt, a 1920-id prompt with 128 tokens up to context 2048, the isolated lm_head and MLP
half-layer) and generic ones between them. Everything goes through the ops of qwen_megakernel_C, as
Decoder calls them, on a full 28-layer model unless a case says otherwise.

The synthetic model: fp16 weights N(0, 0.02), norm gains 1 + 0.1 N(0, 1) (q/k gains around 1.5, so
that attention is as selective as a trained model's), embeddings N(0, 1) and an lm_head whose row
perm[v] is 0.04 embedding[v]. The embedding stays visible in the last residual, so the model is sure
of its next token (perm of the last one), as a trained model mostly is, and a generation's ids do not
hang on the last bit of a logit.
"""

import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "qwen0.6b_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qwen_megakernel_C as ops  # noqa: E402
import Qwen06B_architecture as qa  # noqa: E402

H, I, HD, NQ, NKV, V = 1024, 3072, 128, 16, 8, 151936
QSZ, KVSZ = NQ * HD, NKV * HD
LAYERS, MAX_SEQ = 28, 2048
EPS = 1e-6
SCALE = 1.0 / math.sqrt(HD)
LAYER_WEIGHTS = QSZ * H + 2 * KVSZ * H + H * QSZ + 3 * I * H  # matrix entries of one layer


def listed():
    return [
        # the MLP half-layer on its own
        dict(name="mlp_block", kind="mlp"),
        # the lm_head, its logits and the greedy token
        dict(name="lm_head", kind="lm_head"),
        # one token drawn from logits a program holds: nucleus sampling
        dict(name="sample_top_p", kind="sample", n=V, temperature=0.8, top_k=0, top_p=0.95),
        # one step of a chat loop (Decoder.step), in the middle of a conversation
        dict(name="step", kind="step", layers=LAYERS, pos=700),
        # 32 greedy tokens after a 16-id prompt
        dict(name="generate_32_short", kind="generate", layers=LAYERS, start=15, steps=32),
        # 128 greedy tokens up to the full context
        dict(name="generate_128_ctx2048", kind="generate", layers=LAYERS, start=1920, steps=128),
        # 32 sampled tokens, the usual chat settings
        dict(name="sampled_32", kind="sampled", layers=LAYERS, start=500, steps=32, temperature=0.7, top_k=20,
             top_p=0.8),
        # the prompts of the workloads above, all but their last id: a short question, a paragraph, a
        # page, the longest
        dict(name="prefill_15", kind="prefill", layers=LAYERS, start=0, n=15),
        dict(name="prefill_127", kind="prefill", layers=LAYERS, start=0, n=127),
        dict(name="prefill_999", kind="prefill", layers=LAYERS, start=0, n=999),
        dict(name="prefill_1919", kind="prefill", layers=LAYERS, start=0, n=1919),
        # a user's next turn in a long conversation
        dict(name="prefill_turn", kind="prefill", layers=LAYERS, start=1400, n=61),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["prefill"] * 5 + ["generate"] * 2 + ["sampled"] * 2 + ["step", "step", "sample"])
    if kind == "prefill":
        n = _log_int(rng, 1, 2047)
        # a first prompt or a later turn; the full model mostly, a shallow one now and then
        start = rng.choice([0, 0, rng.randint(0, MAX_SEQ - n)])
        return dict(kind=kind, layers=rng.choice([LAYERS, LAYERS, LAYERS, rng.randint(1, 8)]), start=start, n=n)
    if kind == "step":
        return dict(kind=kind, layers=rng.choice([LAYERS, LAYERS, rng.randint(1, 8)]),
                    pos=_log_int(rng, 1, MAX_SEQ) - 1)
    if kind == "sample":
        return dict(kind=kind, n=rng.choice([V, V, _log_int(rng, 1000, V)]),
                    temperature=round(rng.uniform(0.5, 1.2), 3), top_k=rng.choice([0, 0, 20, 50, 200]),
                    top_p=rng.choice([1.0, 0.8, 0.9, 0.95]))
    steps = _log_int(rng, 2, 64)
    c = dict(kind=kind, layers=LAYERS, start=rng.randint(0, MAX_SEQ - steps), steps=steps)
    if kind == "sampled":
        # (with a top-p, so that a model as sure as this one draws the token the reference expects)
        c.update(temperature=round(rng.uniform(0.5, 0.9), 3), top_k=rng.choice([0, 20, 50, 200]),
                 top_p=rng.choice([0.8, 0.9, 0.95]))
    return c


# ---- inputs ---------------------------------------------------------------------------------


def _model(seed, layers):
    """The synthetic model's tensors, in the layout of load_weights."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=0.02, mean=0.0):
        t = torch.empty(shape, dtype=torch.float16, device="cuda").normal_(0.0, 1.0, generator=g)
        return t.mul_(std).add_(mean) if mean else t.mul_(std)

    embed = normal(V, H, std=1.0)
    perm = torch.randperm(V, device="cuda", generator=g)
    lm_head = torch.empty_like(embed)
    lm_head[perm] = embed * 0.04
    lw = []
    for _ in range(layers):
        lw += [normal(H, std=0.1, mean=1.0), normal(QSZ, H), normal(KVSZ, H), normal(KVSZ, H),
               normal(HD, std=0.1, mean=1.5), normal(HD, std=0.1, mean=1.5), normal(H, QSZ),
               normal(H, std=0.1, mean=1.0), normal(I, H), normal(I, H), normal(H, I)]
    cos, sin = qa.rope_tables("cuda")
    return dict(embed=embed, perm=perm, lm_head=lm_head, layer_weights=lw, cos=cos, sin=sin,
                final_norm=normal(H, std=0.1, mean=1.0), gen=g, normal=normal)


def _decoder_state(case, seed, start, n):
    """Model, K/V cache holding `start` earlier positions, and the ids of the call."""
    L = case["layers"]
    m = _model(seed, L)
    kc = torch.zeros(L, NKV, MAX_SEQ, HD, dtype=torch.float16, device="cuda")
    vc = torch.zeros_like(kc)
    if start:
        kc[:, :, :start] = m["normal"](L, NKV, start, HD, std=1.5)
        vc[:, :, :start] = m["normal"](L, NKV, start, HD, std=0.64)
    ids = torch.randint(0, V, (n,), device="cuda", generator=m["gen"], dtype=torch.int32)
    f32 = dict(dtype=torch.float32, device="cuda")
    s = dict(case=case, m=m, kc=kc, vc=vc, ids=ids, first=int(ids[0]), packed=qa._pack_layer_weights(m["layer_weights"]),
             hidden=torch.empty(H, dtype=torch.float16, device="cuda"), norm_out=torch.empty(H, **f32))
    end = start + (n if case["kind"] == "prefill" else case.get("steps", 1))
    # the cache rows a call writes
    s["k_new"], s["v_new"] = kc[:, :, start:end], vc[:, :, start:end]
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        g = torch.Generator(device="cuda").manual_seed(seed)

        def normal(*shape, std):
            return torch.empty(shape, dtype=torch.float16, device="cuda").normal_(0.0, 1.0, generator=g).mul_(std)

        return dict(case=case, x=normal(H, std=1.5), norm=normal(H, std=0.1).add_(1.0), gate=normal(I, H, std=0.02),
                    up=normal(I, H, std=0.02), down=normal(H, I, std=0.02))
    if kind == "lm_head":
        g = torch.Generator(device="cuda").manual_seed(seed)
        w = torch.empty(V, H, dtype=torch.float16, device="cuda").normal_(0.0, 1.0, generator=g).mul_(0.02)
        h = torch.empty(H, dtype=torch.float16, device="cuda").normal_(0.0, 1.0, generator=g)
        return dict(case=case, w=w, h=h, logits=torch.empty(V, dtype=torch.float32, device="cuda"))
    if kind == "sample":
        # a language model's logits: a broad bulk and a few hundred plausible tokens
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.empty(case["n"], dtype=torch.float32, device="cuda").normal_(0.0, 2.0, generator=g)
        top = torch.randint(0, case["n"], (300,), device="cuda", generator=g)
        x[top] = torch.empty(300, device="cuda").normal_(11.0, 2.0, generator=g)
        return dict(case=case, logits=x, seed=seed)
    if kind == "prefill":
        return _decoder_state(case, seed, case["start"], case["n"])
    if kind == "step":
        s = _decoder_state(case, seed, case["pos"], 1)
        f16 = dict(dtype=torch.float16, device="cuda")
        f32 = dict(dtype=torch.float32, device="cuda")
        # the reference's scratch tensors, which decode() takes
        s["scratch"] = (torch.empty(QSZ, **f32), torch.empty(H, **f32), torch.empty(QSZ, **f16), torch.empty(KVSZ, **f16),
                        torch.empty(KVSZ, **f16), torch.empty(QSZ, **f16), torch.empty(I, **f32))
        s["bmax"] = (torch.empty(4096, **f32), torch.empty(4096, dtype=torch.int32, device="cuda"))
        return s
    s = _decoder_state(case, seed, case["start"], 1)
    s["seed"] = seed
    if kind == "generate":
        s["logits"] = torch.empty(case["steps"], V, dtype=torch.float32, device="cuda")
    return s


# ---- one pass ---------------------------------------------------------------------------------


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "mlp":
        return ops.mlp_block(s["x"], s["norm"], s["gate"], s["up"], s["down"])
    if kind == "lm_head":
        tok = ops.lm_head_argmax(s["h"], s["w"], s["logits"])
        return dict(token=tok, logits=s["logits"])
    if kind == "sample":
        return ops.sample(s["logits"], c["temperature"], c["top_k"], c["top_p"], s["seed"], 7)
    m = s["m"]
    kv = dict(k=s["k_new"], v=s["v_new"], hidden=s["hidden"])
    if kind == "prefill":
        ops.prefill(s["ids"], m["embed"], s["packed"], m["cos"], m["sin"], s["kc"], s["vc"], s["hidden"], c["layers"],
                    c["start"], MAX_SEQ, SCALE)
        return kv
    kv["norm_out"] = s["norm_out"]
    if kind == "step":
        kv["token"] = ops.decode(s["first"], m["embed"], s["packed"], m["final_norm"], m["lm_head"], m["cos"], m["sin"],
                                 s["kc"], s["vc"], s["hidden"], *s["scratch"], s["norm_out"], *s["bmax"], c["layers"],
                                 c["pos"], MAX_SEQ, SCALE)
    elif kind == "generate":
        kv["tokens"] = ops.generate_ex(s["first"], c["steps"], None, m["embed"], s["packed"], m["final_norm"],
                                       m["lm_head"], m["cos"], m["sin"], s["kc"], s["vc"], s["hidden"], s["norm_out"],
                                       s["logits"], None, c["layers"], c["start"], MAX_SEQ, SCALE)
        kv["logits"] = s["logits"]
    else:
        kv["tokens"], kv["count"] = ops.generate_sampled(
            s["first"], c["steps"], -1, m["embed"], s["packed"], m["final_norm"], m["lm_head"], m["cos"], m["sin"],
            s["kc"], s["vc"], s["hidden"], s["norm_out"], c["layers"], c["start"], MAX_SEQ, SCALE, c["temperature"],
            c["top_k"], c["top_p"], s["seed"])
    return kv


# ---- what a pass cannot do without -------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        return {"bytes": 2 * 3 * I * H + 2 * 2 * H + 4 * H, "flops": 2 * 3 * I * H}
    if kind == "lm_head":
        return {"bytes": 2 * V * H + 2 * H + 4 * V + 4, "flops": 2 * V * H}
    if kind == "sample":
        return {"bytes": 4 * case["n"] + 4, "flops": 4 * case["n"]}
    L = case["layers"]
    weights = L * (2 * LAYER_WEIGHTS + 2 * (2 * H + 2 * HD))
    row = 2 * 2 * KVSZ * L  # K and V of one position
    if kind == "prefill":
        n, start = case["n"], case["start"]
        keys = n * start + n * (n + 1) // 2  # (query, key) pairs
        return {"bytes": weights + 2 * n * H + row * (start + n) + 2 * H + 4 * n,
                "flops": L * (2 * n * LAYER_WEIGHTS + 4 * NQ * HD * keys)}
    start, steps = (case["pos"], 1) if kind == "step" else (case["start"], case["steps"])
    ctx = sum(start + t + 1 for t in range(steps))  # positions attended, over the steps
    head = 2 * V * H + 2 * H + 2 * H + (4 * V if kind == "generate" else 0)
    return {"bytes": steps * (weights + head) + row * ctx + 6 * H + 4 * steps,
            "flops": steps * 2 * (L * LAYER_WEIGHTS + V * H) + L * 4 * NQ * HD * ctx}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "lm_head":  # sums in 32 bits: 9e-8 off 64 bits, 5e-7 at the worst logit
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "mlp":  # SiLU * up in 16 bits: 4e-5 off, 1.1e-4 at the worst row
        return {"rel": 2e-4, "max": 2e-3}
    # fp16 activations through every layer: 0.6 to 1.9e-3 off 64 bits (9e-3 at the worst value), and
    # prefill and decode, two implementations of the same, are 2.1e-3 apart (1.1e-2 at the worst value)
    return {"rel": 8e-3, "max": 5e-2}


# ---- the same in 64 bits ------------------------------------------------------------------------


def _rms(x, g):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * g.double()


def _forward64(s, ids, start):
    """Every position's K, V and last residual of ids at positions start .., after the cached ones."""
    m, c = s["m"], s["case"]
    n = ids.numel()
    x = m["embed"][ids.long()].double()
    cos, sin = m["cos"][start:start + n].double(), m["sin"][start:start + n].double()

    def rope(y):  # [n, heads, HD]
        lo, hi = y[..., :HD // 2], y[..., HD // 2:]
        return y * cos[:, None] + torch.cat([-hi, lo], -1) * sin[:, None]

    mask = torch.arange(start + n, device="cuda")[None, :] > (start + torch.arange(n, device="cuda"))[:, None]
    ks, vs = [], []
    for layer in range(c["layers"]):
        g1, wq, wk, wv, gq, gk, wo, g2, wg, wu, wd = m["layer_weights"][11 * layer:11 * layer + 11]
        h = _rms(x, g1)
        q = rope(_rms((h @ wq.double().T).view(n, NQ, HD), gq))
        k = rope(_rms((h @ wk.double().T).view(n, NKV, HD), gk)).transpose(0, 1).contiguous()
        v = (h @ wv.double().T).view(n, NKV, HD).transpose(0, 1).contiguous()
        ks.append(k)
        vs.append(v)
        att = torch.empty(n, NQ, HD, dtype=torch.float64, device="cuda")
        for head in range(NQ):
            kk = torch.cat([s["kc"][layer, head // 2, :start].double(), k[head // 2]])
            vv = torch.cat([s["vc"][layer, head // 2, :start].double(), v[head // 2]])
            p = (q[:, head] @ kk.T * SCALE).masked_fill_(mask, -math.inf)
            att[:, head] = torch.softmax(p, -1) @ vv
        x = x + att.view(n, QSZ) @ wo.double().T
        h = _rms(x, g2)
        x = x + (torch.nn.functional.silu(h @ wg.double().T) * (h @ wu.double().T)) @ wd.double().T
    return x, torch.stack(ks), torch.stack(vs)


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    s = prepare(case, seed)
    if kind == "mlp":
        x = s["x"].double()
        h = _rms(x, s["norm"])
        act = torch.nn.functional.silu(s["gate"].double() @ h) * (s["up"].double() @ h)
        return x + s["down"].double() @ act
    if kind == "lm_head":
        y = s["w"].double() @ s["h"].double()
        return dict(token=y.argmax().view(1).int(), logits=y)
    m = s["m"]
    if kind == "prefill":
        x, k, v = _forward64(s, s["ids"], case["start"])
        return dict(k=k, v=v, hidden=x[-1])
    start, steps = (case["pos"], 1) if kind == "step" else (case["start"], case["steps"])
    ids = [s["first"]]
    for _ in range(steps - 1):  # the model is sure of perm of its last token
        ids.append(int(m["perm"][ids[-1]]))
    x, k, v = _forward64(s, torch.tensor(ids, device="cuda"), start)
    h = _rms(x, m["final_norm"])
    out = dict(k=k, v=v, hidden=x[-1], norm_out=h[-1])
    if kind == "sampled":
        out.update(tokens=m["perm"][torch.tensor(ids, device="cuda")].int(),
                   count=torch.tensor([steps], dtype=torch.int32, device="cuda"))
        return out
    w = m["lm_head"].double()
    logits = h @ w.T
    best = logits.argmax(-1).int()
    out["token" if kind == "step" else "tokens"] = best
    if kind == "generate":
        out["logits"] = logits
    return out
