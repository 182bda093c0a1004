"""What this framework is used for, as cases that can be timed and checked.

Two kinds of pass, both through the engine that a service holds (``LLMEngine``), with the weights
loaded once and kept:

* ``prompt``: one step over new prompts, ``LLMEngine.replay_step``, up to the logits of each prompt's
  last token (what a first token is sampled from); the requests end with the step.
* ``decode``: one token for each of a set of running sequences, ``ModelRunner.decode_launch`` and
  ``decode_collect`` (a captured graph with the sampler in it), with the logits beside it.  The
  sequences' histories are in the caches before the pass.  A sequence's last page has room for the token.

Models are the registry's: ``llama-4k-4l`` (layers of the service's default 8B model, four of them as
engine comparisons take them: through 32 layers with a bf16 residual two correct implementations drift
further apart than any tolerance could tell from a fault) and the 2048-wide preset of each other
architecture.  bf16 is the type that all of them are served in; fp32 activations are a mode for
checking, and fp8 caches and 4-bit weights of Llama have measurements of their own.

Weights are random, as a registry name gives them, with one change for mixtures of experts: a router
of random numbers decides by differences smaller than bf16's rounding now and then, and then two correct
implementations choose different experts.  A trained router is decisive; here every token's embedding
names its experts in columns that the routers read, so tokens spread evenly over the experts and no
choice hangs on rounding.
"""
import math

import numpy as np
import torch

FAMILIES = ("nulazen", "bagasun", "kerarax", "fufipel", "logirax", "pitelorn")
LLAMA = "llama-4k-4l"
PAGE = 16
# tokens of a running engine's pool: three states and one more of the largest case
POOL_TOKENS = {LLAMA: 700_000, "": 200_000}
# a prompt step of the service carries at most this many tokens
STEP_TOKENS = 8192


def listed():
    def case(name, model, kind, seqs, tokens):
        return {"name": name, "model": model, "kind": kind, "seqs": seqs, "tokens": tokens}

    return [
        # the service's headline load: 50 sessions in long conversations, one token each
        case("llama_decode_50", LLAMA, "decode", 50, 3300),
        # the longest prompt that engine comparisons use
        case("llama_prompt_4096", LLAMA, "prompt", 1, 4096),
        # a long document, alone
        case("nulazen_prompt_4096", "nulazen-2k", "prompt", 1, 4096),
        # a few sessions in conversation
        case("nulazen_decode_8", "nulazen-2k", "decode", 8, 540),
        # a prompt of the middle size of engine comparisons
        case("bagasun_prompt_2048", "bagasun-2k", "prompt", 1, 2048),
        # one session alone: latency of a token
        case("bagasun_decode_1", "bagasun-2k", "decode", 1, 540),
        # several sessions' turns that arrived together, of unlike lengths
        case("kerarax_prompt_5x400", "kerarax-2k", "prompt", 5, 400),
        # a busy service
        case("kerarax_decode_32", "kerarax-2k", "decode", 32, 540),
        # a system prompt and a first message, of odd length
        case("fufipel_prompt_777", "fufipel-2k", "prompt", 1, 777),
        # long conversations of a few sessions
        case("logirax_decode_3", "logirax-2k", "decode", 3, 1500),
        # a turn of an ordinary size: time to first token
        case("pitelorn_prompt_300", "pitelorn-2k", "prompt", 1, 300),
        # short conversations
        case("pitelorn_decode_16", "pitelorn-2k", "decode", 16, 300),
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))

    model = rng.choice((LLAMA,) + tuple(f + "-2k" for f in FAMILIES))
    llama = model == LLAMA
    if rng.random() < 0.5:
        total = log_int(16, 4096)
        seqs = min(log_int(1, 8), max(1, total // 16))
        return {"model": model, "kind": "prompt", "seqs": seqs, "tokens": max(1, total // seqs)}
    seqs = log_int(1, 50 if llama else 64)
    return {"model": model, "kind": "decode", "seqs": seqs,
            "tokens": log_int(24, min(3300, (165_000 if llama else 32_000) // seqs))}


def lengths(case):
    """The sequences' lengths: spread between half and one and a half times ``tokens``, none of
    them a multiple of the page."""
    n, mean = case["seqs"], case["tokens"]
    if n == 1:
        return [mean + (case["kind"] == "decode" and mean % PAGE == 0)]
    out = [max(1, round(mean * (0.5 + (i * 0.6180339887) % 1.0))) for i in range(n)]
    return [v + (v % PAGE == 0) for v in out]


def tokens_of(case, seed, vocab):
    """Per sequence its token ids; a decode case's last id is the token that the step carries."""
    rng = np.random.default_rng([seed, 7])
    extra = 1 if case["kind"] == "decode" else 0
    return [rng.integers(1, vocab, size=n + extra).tolist() for n in lengths(case)]


# --------------------------------------------------------------------------------- the engine
_engines = {}


def _config(model):
    from fasttalk_llm_microservice_amd.models.config import resolve_model

    return resolve_model(model)


def _family(model):
    return model.split("-")[0]


def _design(model):
    """(config.json's dict, tensors' shapes) of a preset of the families."""
    import importlib

    mod = importlib.import_module("fasttalk_llm_microservice_amd.models." + _family(model))
    cfg = _config(model)
    return mod.config_to_dict(cfg), mod.tensor_shapes(cfg)


def _weights(model, device):
    """The preset's random tensors with decisive routers (see the module's docstring)."""
    import importlib

    mod = importlib.import_module("fasttalk_llm_microservice_amd.models." + _family(model))
    ten = mod.random_tensors(_config(model), 0, device=device)
    moe = [(i, l["mlp"]) for i, l in enumerate(_design(model)[0]["layers"]) if l["mlp"] and l["mlp"]["kind"] == "moe"]
    if not moe:
        return ten
    r = moe[0][1]["router"]
    e, top, grp = r["experts"], r["top"], r.get("groups") or {"count": 1, "keep": 1}
    g = torch.Generator().manual_seed(1)
    size, vocab = e // grp["count"], ten["embed"].shape[0]
    kept = torch.rand(vocab, grp["count"], generator=g).argsort(1)[:, :grp["keep"]]
    open_ = torch.zeros(vocab, grp["count"]).scatter_(1, kept, 1.0).repeat_interleave(size, 1)
    pick = (torch.rand(vocab, e, generator=g) + open_).topk(top, 1).indices
    code = torch.zeros(vocab, e).scatter_(1, pick, 28.0)
    ten["embed"][:, :e] += code.to(device, ten["embed"].dtype)
    for i, _ in moe:
        # each layer reads the columns shifted by whole groups, so layers differ in their choice
        w = ten[f"l{i}.mlp.router"]
        w *= 0.05
        w[torch.arange(e), (torch.arange(e) + i * size) % e] += 0.5
        if f"l{i}.mlp.correction" in ten:       # balanced experts need little correction
            ten[f"l{i}.mlp.correction"] *= 0.01
    return ten


def _engine(model):
    if model not in _engines:
        from fasttalk_llm_microservice_amd.engine.config import EngineConfig
        from fasttalk_llm_microservice_amd.engine.engine import LLMEngine

        pool = POOL_TOKENS.get(model, POOL_TOKENS[""])
        eng = LLMEngine(EngineConfig(model=model, device="cuda", dtype="bfloat16", max_model_len=8192,
                                     num_kv_blocks=pool // PAGE, block_size=PAGE, max_num_seqs=256,
                                     max_num_batched_tokens=STEP_TOKENS, enable_prefix_caching=False,
                                     swap_space_gb=0.0))
        if model != LLAMA:
            ten = _weights(model, eng.runner.device)
            eng.runner.model.load_tensors(ten.__getitem__, ten.__contains__)
        _engines[model] = eng
    return _engines[model]


class State:
    """A case's inputs and, for a decode case, its running sequences (which end with it)."""

    def __init__(self, eng, case, ids):
        self.eng, self.case, self.ids, self.live = eng, case, ids, []
        self.seqs = []

    def __del__(self):
        if self.live:
            self.eng.replay_step([], self.live)


_next_id = [0]


def prepare(case, seed):
    eng = _engine(case["model"])
    ids = tokens_of(case, seed, eng.model_cfg.vocab_size)
    st = State(eng, case, ids)
    names = []
    for _ in ids:
        _next_id[0] += 1
        names.append("s%d" % _next_id[0])
    st.names = names
    if case["kind"] == "prompt":
        st.entries = [(n, t, [len(t) - 1]) for n, t in zip(names, ids)]
        return st
    from fasttalk_llm_microservice_amd.engine.sampling_params import SamplingParams

    step, rows = [], 0
    for n, t in zip(names, ids):
        if rows and rows + len(t) - 1 > STEP_TOKENS:
            eng.replay_step(step)
            step, rows = [], 0
        step.append((n, t[:-1], []))
        rows += len(t) - 1
        st.live.append(n)
    eng.replay_step(step)
    for n, t in zip(names, ids):
        seq = eng.scheduler.by_id[n]
        seq.params = SamplingParams(temperature=0.7, top_p=0.9, max_tokens=128, ignore_eos=True, seed=seed)
        seq.append(t[-1])
        st.seqs.append(seq)
    eng.runner.warmup([len(ids)])
    return st


def run(state):
    """Logits only: what a step writes into caches and states is the engine's own, and the next pass's
    logits of a decode case depend on it.  (Sampled tokens follow from the logits; a near tie may turn.)"""
    if state.case["kind"] == "prompt":
        return {"logits": state.eng.replay_step(state.entries, state.names)}
    runner = state.eng.runner
    runner.logits_tap = taps = []
    runner.decode_collect(runner.decode_launch(state.seqs))
    runner.logits_tap = None
    return {"logits": taps[0]}


# ------------------------------------------------------------------------- what a pass cannot do without
def _attended(case, window=0, blocks=False, keep=0):
    """(query, key) pairs and keys that are read, over all sequences."""
    pairs = keys = 0
    for n in lengths(case):
        first = 0 if case["kind"] == "prompt" else n
        last = n - 1 if case["kind"] == "prompt" else n
        i = np.arange(first, last + 1)
        seen = i + 1
        if window:
            seen = i % window + 1 if blocks else np.minimum(i + 1, np.minimum(i + 1, window) + keep)
        pairs += int(seen.sum())
        keys += int(last + 1 if case["kind"] == "prompt" else seen[-1])
    return pairs, keys


def _mixer_work(m, kind, case, rows, slots):
    """(bytes, flops) of one mixer beside its projections."""
    if "left" in m:
        a, b = (_mixer_work(m[k], kind + k, case, rows, slots) for k in ("left", "right"))
        return a[0] + b[0], a[1] + b[1]
    h, dk = m["heads"], m.get("dim", m.get("state"))
    dv = m.get("vdim", dk)
    if "kv_rank" in m:
        width = m["kv_rank"] + m["rot_dim"]
        pairs, keys = _attended(case)
        # in the plain form: keys and values of every head, scores and sums
        return 2.0 * width * keys, 2.0 * pairs * h * (dk + m["rot_dim"] + dv)
    if "scale" in m:
        mask = m.get("mask") or {}
        maps = 2 if "diff" in m else 1
        blocks = kind == "parallelleft" and "conv" not in m
        pairs, keys = _attended(case, mask.get("size", 0), blocks, mask.get("keep_first", 0))
        return 2.0 * keys * m.get("kv_heads", h) * (dk * maps + dv), 2.0 * pairs * h * maps * (dk + dv)
    # a recurrence: the state read and written once per sequence, two or three products a row
    read = 1 if case["kind"] == "prompt" else 2
    return 4.0 * read * slots * h * dk * dv, (6.0 if "conv" in m else 4.0) * rows * h * dk * dv


def work(case):
    rows = case["seqs"] if case["kind"] == "decode" else sum(lengths(case))
    wanted = case["seqs"]
    if case["model"] == LLAMA:
        c = _config(LLAMA)
        h, i, d, nq, nkv = c.hidden_size, c.intermediate_size, c.head_dim, c.num_heads, c.num_kv_heads
        layer = h * (nq + 2 * nkv) * d + nq * d * h + 3 * h * i
        pairs, keys = _attended(case)
        byts = 2.0 * (c.num_layers * (layer + 2 * keys * nkv * d) + c.vocab_size * h) + 2.0 * wanted * c.vocab_size
        flops = 2.0 * rows * c.num_layers * layer + 4.0 * pairs * nq * d * c.num_layers + 2.0 * wanted * c.vocab_size * h
        return {"bytes": byts, "flops": flops}
    cfg, shapes = _design(case["model"])
    byts = flops = 0.0
    for i, l in enumerate(cfg["layers"]):
        r = (l["mlp"] or {}).get("router")
        share = r["top"] / r["experts"] if r else 0.0          # rows that an expert gets
        hit = 1.0 - (1.0 - share) ** rows                      # whether it gets any
        for name, s in shapes.items():
            if name.startswith(f"l{i}.") and len(s) == 2 and not name.endswith(("conv", "rel")):
                size, routed = float(s[0] * s[1]), name.startswith(f"l{i}.mlp.e") and name[len(f"l{i}.mlp.e")].isdigit()
                byts += 2.0 * size * (hit if routed else 1.0)
                flops += 2.0 * size * rows * (share if routed else 1.0)
        b, f = _mixer_work(l["mixer"], l["type"], case, rows, case["seqs"])
        byts, flops = byts + b, flops + f
    head = cfg["vocab"] * cfg["width"]
    return {"bytes": byts + 2.0 * head + 2.0 * rows * cfg["width"] + 4.0 * wanted * cfg["vocab"],
            "flops": flops + 2.0 * wanted * head}


def tolerance(case):
    # bf16 operands, activations and caches through 4 layers: the logits are 0.004 to 0.008 (Llama, whose
    # residual is bf16 too: 0.02) from those of 64 bits, and 0.002 where the embedding is scaled up 16 times
    rel = 0.008 if _family(case["model"]) in ("bagasun", "fufipel", "logirax") else 0.03
    return {"rel": rel, "max": 10 * rel}


# ------------------------------------------------------------------------------ the same in 64 bits
D = torch.float64


def _lin(P, name, h):
    y = h @ P[name].to(D).T
    return y + P[name + ".b"].to(D) if name + ".b" in P else y


def _rms(x, eps, w=None):
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if w is None else x * w


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(D) + b.to(D)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


def _conv(x, w):
    w = w.to(D)
    taps = w.shape[1]
    pad = torch.cat([torch.zeros(taps - 1, x.shape[1], dtype=D, device=x.device), x])
    return sum(w[:, j] * pad[j:j + x.shape[0]] for j in range(taps))


def _frequencies(dims, base, scaling):
    """Angles per position and a factor on sine and cosine."""
    f = [float(base) ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not scaling:
        return f, 1.0
    s, orig = float(scaling["factor"]), float(scaling["original"])
    if "low" in scaling:                      # by wavelength
        out = []
        for v in f:
            turns = orig * v / (2 * math.pi)
            mix = min(max((turns - scaling["low"]) / (scaling["high"] - scaling["low"]), 0.0), 1.0)
            out.append((1 - mix) * v / s + mix * v)
        return out, 1.0

    def pair(turns):
        return dims * math.log(orig / (2 * math.pi * turns)) / (2 * math.log(base))

    lo, hi = max(math.floor(pair(scaling["fast"])), 0), min(math.ceil(pair(scaling["slow"])), dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [v / s * r + v * (1 - r) for v, r in zip(f, ramp)], 0.1 * math.log(s) + 1.0


def _rotate(x, rot, neighbours=False):
    """x [T, heads, n]; pairs (i, i + dims/2) of the first dims entries, or (2i, 2i + 1)."""
    if not rot or not rot.get("dims"):
        return x
    dims = rot["dims"]
    f, mult = _frequencies(dims, rot.get("base", 10000.0), rot.get("scaling"))
    ang = torch.arange(x.shape[0], dtype=D, device=x.device)[:, None] * torch.tensor(f, dtype=D, device=x.device)
    c, s = (ang.cos() * mult)[:, None], (ang.sin() * mult)[:, None]
    a, b = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
    out = x.clone()
    out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return out


def _hidden(T, device, size=0, blocks=False, keep=0):
    """[T, T]: the keys that a row does not see."""
    i, j = torch.arange(T, device=device)[:, None], torch.arange(T, device=device)[None]
    if not size:
        return j > i
    return (j > i) | ((i // size != j // size) if blocks else ((i - j >= size) & (j >= keep)))


def _softmax(s, hidden, sink=None):
    s = s.masked_fill(hidden, -math.inf)
    if sink is None:
        return torch.softmax(s, -1)
    top = torch.maximum(s.amax(-1, keepdim=True), sink)
    e = torch.exp(s - top)
    return e / (e.sum(-1, keepdim=True) + torch.exp(sink - top))


def _attend(q, k, v, weights):
    """q [T, H, dk], k [T, G, dk], v [T, G', dv]; ``weights(h, dot products)`` of head h."""
    H = q.shape[1]
    return torch.stack([weights(h, q[:, h] @ k[:, h * k.shape[1] // H].T) @ v[:, h * v.shape[1] // H]
                        for h in range(H)], 1)


def _recur(q, k, v, decay, beta=None):
    """S <- decay S + k u^T, o = S^T q; u = v, or beta (v - (decay S)^T k).  q, k [T, H, dk], v
    [T, H, dv], decay [T, H, dk or 1], beta [T, H]."""
    T, H, dk = q.shape
    S = torch.zeros(H, dk, v.shape[2], dtype=D, device=q.device)
    o = torch.empty(T, H, v.shape[2], dtype=D, device=q.device)
    for t in range(T):
        S *= decay[t][:, :, None]
        kt = k[t][:, :, None]
        u = v[t][:, None] if beta is None else beta[t][:, None, None] * (v[t][:, None] - (S * kt).sum(1, keepdim=True))
        S.addcmul_(kt.expand_as(S), u.expand_as(S))
        torch.sum(S * q[t][:, :, None], 1, out=o[t])
    return o


def _heads(x, n):
    return x.view(x.shape[0], n, -1)


def _delta(P, p, m, h, eps, per_head):
    H, G = m["heads"], m.get("kv_heads", m["heads"])
    q, k, v = (_heads(_silu(_conv(_lin(P, p + n, h), P[p + n + ".conv"])), g) for n, g in (("q", G), ("k", G), ("v", H)))
    q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    q, k = ((x * f).repeat_interleave(H // G, 1) for x, f in ((q, m["dim"] ** -0.5), (k, 1.0)))
    a = _lin(P, p + "a", h) if per_head else _lin(P, p + "a2", _lin(P, p + "a1", h))
    step = torch.nn.functional.softplus(a + P[p + "dt_bias"].to(D), threshold=1e9)
    decay = torch.exp(-torch.exp(P[p + "A_log"].to(D))[None, :, None] * _heads(step, H))
    o = _rms(_recur(q, k, v, decay, torch.sigmoid(_lin(P, p + "b", h))), eps, P[p + "norm"].to(D))
    gate = _silu(_lin(P, p + "g", h)) if per_head else torch.sigmoid(_lin(P, p + "g2", _lin(P, p + "g1", h)))
    return _lin(P, p + "o", o.flatten(1) * gate)


def _latent(P, p, m, h, eps, logirax):
    H, dn, R = m["heads"], m["dim"], m["kv_rank"]
    src = _rms(_lin(P, p + "dq", h), eps, P[p + "dq.norm"].to(D)) if logirax else h
    q = _heads(_lin(P, p + ("uq" if logirax else "q"), src), H)
    down = _lin(P, p + "dkv", h)
    c = _rms(down[:, :R], eps, P[p + "dkv.norm"].to(D))
    rot = dict({"dims": m["rot_dim"]}, **(m.get("rot") or {}))
    kr, qr = _rotate(down[:, None, R:], rot, logirax)[:, 0], _rotate(q[..., dn:], rot, logirax)
    k, v, hid = _heads(_lin(P, p + "uk", c), H), _heads(_lin(P, p + "uv", c), H), _hidden(h.shape[0], h.device)
    sink = P[p + "sink"].to(D) if logirax else [None] * H
    o = _attend(q[..., :dn], k, v, lambda a, s: _softmax((s + qr[:, a] @ kr.T) * m["scale"], hid, sink[a]))
    if logirax:
        o = o * torch.sigmoid(_lin(P, p + "g", h))[:, :, None]
    return _lin(P, p + "o", o.flatten(1))


def _glu(P, p, h, act, limit=0.0):
    if act == "relu_sq":
        return _lin(P, p + "down", torch.relu(_lin(P, p + "up", h)) ** 2)
    g, u = _lin(P, p + "gate", h), _lin(P, p + "up", h)
    if act == "clamp":
        g, u = g.clamp(max=limit), u.clamp(-limit, limit) + 1
        return _lin(P, p + "down", g * torch.sigmoid(1.702 * g) * u)
    return _lin(P, p + "down", {"silu": _silu, "gelu": _gelu, "relu": torch.relu}[act](g) * u)


def _grouped(score, r, group_score):
    """Scores with the experts outside the best groups taken out."""
    g = r.get("groups")
    if not g:
        return score
    s = score.view(score.shape[0], g["count"], -1)
    out = group_score(s).argsort(1, descending=True)[:, g["keep"]:]
    return s.scatter(1, out[:, :, None].expand(-1, -1, s.shape[2]), -math.inf).flatten(1)


def _experts(P, p, m, h, family):
    r = m["router"]
    z = _lin(P, p + "router", h)
    if family == "nulazen":
        s = torch.softmax(z, -1)
        idx = _grouped(s + P[p + "correction"].to(D), r, lambda x: x.amax(-1)).topk(r["top"], 1).indices
        w = s.gather(1, idx)
    elif family == "kerarax":
        top, idx = z.topk(r["top"], 1)
        w = torch.softmax(top, -1)
    else:
        s = torch.sigmoid(z)
        idx = _grouped(s, r, lambda x: x.topk(2, -1).values.sum(-1)).topk(r["top"], 1).indices
        w = s.gather(1, idx)
        w = w / (w.sum(1, keepdim=True) + 1e-20) * r.get("scale", 1.0)
    act = {"kerarax": "relu_sq", "logirax": "silu"}.get(family, "clamp")
    limit = m["expert"].get("limit", 0.0)
    y = torch.zeros_like(h)
    for e in range(r["experts"]):
        row, place = torch.nonzero(idx == e, as_tuple=True)
        if row.numel():
            y.index_add_(0, row, w[row, place][:, None] * _glu(P, f"{p}e{e}.", h[row], act, limit))
    if m.get("shared"):
        s = _glu(P, p + "shared.", h, act, m["shared"].get("limit", limit))
        y = y + (s if family == "logirax" else torch.sigmoid(_lin(P, p + "shared.sg", h)) * s)
    return y


def _last(P, name, x, eps, norm):
    return norm(x[-1:], "final.norm") @ P[name].to(D).T


def _nulazen(cfg, P, tok, x, eps):
    norm = lambda v, n: _rms(v, eps, P[n].to(D))   # noqa: E731
    for i, l in enumerate(cfg["layers"]):
        p, h = f"l{i}.", norm(x, f"l{i}.norm1")
        y = _latent(P, p + "mix.", l["mixer"], h, eps, False) if l["type"] == "latent_attention" else \
            _delta(P, p + "mix.", l["mixer"], h, eps, False)
        x = x + norm(y, p + "norm1b")
        h = norm(x, p + "norm2")
        y = _experts(P, p + "mlp.", l["mlp"], h, "nulazen") if l["mlp"]["kind"] == "moe" else _glu(P, p + "mlp.", h, "relu_sq")
        x = x + norm(y, p + "norm2b")
        n = cfg["token_side"]["dim"]
        e = P["side.embed"][tok][:, i * n:(i + 1) * n].to(D)
        x = x + norm(_lin(P, p + "side.proj", _gelu(_lin(P, p + "side.gate", x)) * e), p + "side.norm")
    return _last(P, "head", x, eps, norm)


def _bagasun(cfg, P, tok, x, eps):
    norm = lambda v, n: _rms(v, eps, P[n].to(D))   # noqa: E731
    for i, l in enumerate(cfg["layers"]):
        m, p = l["mixer"], f"l{l.get('weights_of', i)}."
        u, q = norm(x, p + "norm1"), p + "mix."
        if l["type"] == "mamba2":
            H, dv, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            n = H * dv
            z, xbc, dt = _lin(P, q + "in", u).split([n, n + 2 * G * N, H], 1)
            a, b, c = _silu(_conv(xbc, P[q + "conv"]) + P[q + "conv.b"].to(D)).split([n, G * N, G * N], 1)
            a, b, c = _heads(a, H), *(_heads(v, G).repeat_interleave(H // G, 1) for v in (b, c))
            dt = torch.nn.functional.softplus(dt + P[q + "dt_bias"].to(D), threshold=1e9)
            decay = torch.exp(-torch.exp(P[q + "A_log"].to(D)) * dt)
            y = _recur(c, b * dt[:, :, None], a, decay[:, :, None]) + P[q + "D"].to(D)[:, None] * a
            y = _rms(_heads(y.flatten(1) * _silu(z), m["norm_groups"]), eps).flatten(1)
            y = _lin(P, q + "o", y * P[q + "norm"].to(D))
        else:
            H, G = m["heads"], m["kv_heads"]
            hid = _hidden(len(tok), u.device, m["mask"]["size"])
            Q, K, V = (_lin(P, q + n, u) for n in "qkv")
            if l["type"] == "attention":
                Q, K = norm(Q, q + "q.norm"), norm(K, q + "k.norm")
                dist = torch.arange(len(tok), dtype=D, device=u.device)
                dist = (dist[:, None] - dist[None]).clamp_min(0.0)
                r1, r2, pb = (P[q + n].to(D) for n in ("r1", "r2", "pb"))
                y = _attend(_heads(Q, H), _heads(K, G), _heads(V, G), lambda a, s: torch.sigmoid(
                    s * m["scale"] - r1[a] * torch.log1p(r2[a] * dist) + pb[a]).masked_fill(hid, 0.0))
            else:
                # heads hold map 0's rows and then map 1's
                Q, K = (_rotate(_heads(v, 2 * n), m.get("rot")) for v, n in ((Q, H), (K, G)))
                maps = [_attend(Q[:, t::2], K[:, t::2], _heads(V, G), lambda a, s: _softmax(s * m["scale"], hid)) for t in (0, 1)]
                lam = [torch.exp((P[q + "lq" + n].to(D) * P[q + "lk" + n].to(D)).sum()) for n in "12"]
                y = _rms(maps[0] - (lam[0] - lam[1] + m["diff"]) * maps[1], eps) * (1 - m["diff"])
                y = y * torch.sigmoid(_lin(P, q + "g", u))[:, :, None]
            y = _lin(P, q + "o", y.flatten(1))
        x = x + norm(y, p + "norm1b")
        x = x + norm(_glu(P, p + "mlp.", norm(x, p + "norm2"), "gelu"), p + "norm2b")
    return _last(P, "head", x, eps, norm)


def _kerarax(cfg, P, tok, x, eps):
    norm = lambda v, n: _layer_norm(v, P[n], P[n + ".b"], eps)   # noqa: E731
    w = cfg["width"]
    ang = torch.arange(len(tok), dtype=D, device=x.device)[:, None] * \
        10000.0 ** (-2.0 * torch.arange(w // 2, dtype=D, device=x.device) / w)
    x = norm(x + torch.stack([ang.sin(), ang.cos()], -1).flatten(1), "embed.norm")
    cap = lambda s, c: c * torch.tanh(s / c) if c else s   # noqa: E731
    zero = torch.zeros((), dtype=D, device=x.device)
    for i, l in enumerate(cfg["layers"]):
        m, p, q = l["mixer"], f"l{i}.", f"l{i}.mix."
        H, G = m["heads"], m["kv_heads"]
        Q, K, V = (_heads(_conv(_lin(P, q + n, x), P[q + n + ".conv"]), g) for n, g in (("q", H), ("k", G), ("v", G)))
        Q, K = _rms(Q, eps, P[q + "q.norm"].to(D)), _rms(K, eps, P[q + "k.norm"].to(D))
        hid = _hidden(len(tok), x.device)
        y = _attend(Q, K, V, lambda a, s: _softmax(cap(s * m["scale"], m.get("softcap")), hid, zero))
        x = x + norm(_lin(P, q + "o", y.flatten(1)), p + "norm1")
        x = x + norm(_experts(P, p + "mlp.", l["mlp"], x, "kerarax"), p + "norm2")
    return cap(_last(P, "head", x, eps, norm), cfg.get("logit_softcap"))


def _pair_rows(cfg, P, tok):
    b = cfg["embedding"]["bigram"]
    row = (tok[:-1] * b["mul_prev"] + tok[1:] * b["mul_cur"]) % b["buckets"]
    return P["bigram"][torch.cat([row.new_full((1,), b["buckets"]), row])].to(D)


def _offset(P, eps):
    return lambda v, n: _rms(v, eps, 1 + P[n].to(D))


def _fufipel(cfg, P, tok, x, eps):
    norm, kvs = _offset(P, eps), {}
    x = x + _pair_rows(cfg, P, tok)
    T = len(tok)
    for i, l in enumerate(cfg["layers"]):
        p = f"l{i}."
        h, q, m = norm(x, p + "norm1"), p + "mix.", l["mixer"]
        if l["type"] == "parallel":
            a, r, q = m["left"], m["right"], p + "mix.left."
            H, G, mask = a["heads"], a["kv_heads"], a.get("mask") or {}
            Q, K = (_rotate(_heads(_lin(P, q + n, h), g), a.get("rot")) for n, g in (("q", H), ("k", G)))
            hid = _hidden(T, x.device, mask.get("size", 0), True)
            y = _attend(Q, K, _heads(_lin(P, q + "v", h), G), lambda _, s: _softmax(s * a["scale"], hid))
            left, q, H = _lin(P, q + "o", y.flatten(1)), p + "mix.right.", r["heads"]
            Q, K, V = (_heads(_lin(P, q + n, h), H) for n in "qkv")
            z = _lin(P, q + "a2", _lin(P, q + "a1", h))
            decay = torch.exp(_heads(torch.nn.functional.logsigmoid(z), H) / r["tau"])
            o = _rms(_recur(Q * r["dim"] ** -0.5, K, V, decay), eps, P[q + "norm"].to(D)).flatten(1)
            right = _lin(P, q + "o", o * _silu(_lin(P, q + "g", h)))
            y = 0.5 * (_rms(left, eps, P[p + "mix.left.out"].to(D)) + _rms(right, eps, P[p + "mix.right.out"].to(D)))
        else:
            H, G, mask, src = m["heads"], m["kv_heads"], m.get("mask") or {}, m.get("kv_from")
            if src is None:
                src = i
                kvs[i] = _heads(_rms(_lin(P, q + "k", h), eps, P[q + "k.norm"].to(D)), G), _heads(_lin(P, q + "v", h), G)
            Q = _heads(_rms(_lin(P, q + "q", h), eps, P[q + "q.norm"].to(D)), H)
            rel, half = P[q + "rel"].to(D), P[q + "rel"].shape[0] // 2
            d = torch.arange(T, dtype=D)
            far = half + torch.floor(torch.log(d.clamp_min(1) / half) / math.log(m["bias_max"] / half) * half)
            bucket = torch.where(d < half, d, far.clamp_max(2 * half - 1)).long().to(x.device)
            dist = (torch.arange(T, device=x.device)[:, None] - torch.arange(T, device=x.device)[None]).clamp_min(0)
            hid = _hidden(T, x.device, mask.get("size", 0), False, mask.get("keep_first", 0))
            y = _attend(Q, *kvs[src], lambda a, s: _softmax(s * m["scale"] + rel[:, a][bucket][dist], hid)).flatten(1)
            y = _lin(P, q + "o", y * torch.sigmoid(_lin(P, q + "g", h)))
        x = x + cfg["residual_mult"] * (y + _glu(P, p + "mlp.", h, "relu"))
    return _last(P, "embed", x, eps, norm) * cfg["logit_scale"]


def _logirax(cfg, P, tok, x, eps):
    norm = _offset(P, eps)
    T = len(tok)
    for i, l in enumerate(cfg["layers"]):
        m, p, q = l["mixer"], f"l{i}.", f"l{i}.mix."
        h = norm(x, p + "norm1")
        h = h + (torch.cat([torch.zeros_like(h[:1]), h[:-1]]) - h) * P[p + "shift"].to(D)
        if l["type"] == "latent_attention":
            y = _latent(P, q, m, h, eps, True)
        else:
            H, G, mask, c = m["heads"], m["kv_heads"], m.get("mask") or {}, m["softcap"]
            V = _heads(_lin(P, q + "k", h), G)
            Q, K = (_rms(_rotate(v, m.get("rot")), eps) for v in (_heads(_lin(P, q + "q", h), H), V))
            hid = _hidden(T, x.device, mask.get("size", 0), False, mask.get("keep_first", 0))
            temp, o = P[q + "temp"].to(D), []
            s = torch.stack([Q[:, a] @ K[:, a * G // H].T * (m["scale"] * temp[a]) for a in range(H)])
            s = c * torch.tanh(s / c)
            for a, mix in enumerate(P[q + "talk"].to(D)):
                o.append(_softmax(sum(f * t for f, t in zip(mix, s)), hid) @ V[:, a * G // H])
            y = _lin(P, q + "o", torch.cat(o, 1) * torch.sigmoid(_lin(P, q + "g", h)))
        x = x + norm(y, p + "norm1b")
        h, f = norm(x, p + "norm2"), l["mlp"]
        y = _experts(P, p + "mlp.", f, h, "logirax") if f["kind"] == "moe" else _glu(P, p + "mlp.", h, "clamp", f["limit"])
        x = x + norm(y, p + "norm2b")
    return _last(P, "embed", x, eps, norm) * cfg["logit_scale"]


def _pitelorn(cfg, P, tok, x, eps):
    norm = _offset(P, eps)
    x = x + _pair_rows(cfg, P, tok)
    T = len(tok)
    for i, l in enumerate(cfg["layers"]):
        m, p = l["mixer"], f"l{i}."
        h = norm(x, p + "norm1")
        if l["type"] == "delta":
            x = x + _delta(P, p + "mix.", m, h, eps, True)
        else:
            a, r, q = m["left"], m["right"], p + "mix.left."
            H, G = a["heads"], a["kv_heads"]
            Q, K, V = (_heads(_conv(_lin(P, q + n, h), P[q + n + ".conv"]), g) for n, g in (("q", H), ("k", G), ("v", G)))
            hid, sink = _hidden(T, x.device, (a.get("mask") or {}).get("size", 0)), P[q + "sink"].to(D)
            Q, K = _rotate(Q, a.get("rot"), True), _rotate(K, a.get("rot"), True)
            y = _lin(P, q + "o", _attend(Q, K, V, lambda b, s: _softmax(s * a["scale"], hid, sink[b])).flatten(1))
            q, H = p + "mix.right.", r["heads"]
            Q, K, V = (_heads(_lin(P, q + n, h), H) for n in "qkv")
            Q, K = _rotate(Q, r.get("rot")), _rotate(K, r.get("rot")) * r["dim"] ** -0.5
            decay = torch.tensor(r["decay"], dtype=D, device=x.device)[None, :, None].expand(T, -1, -1)
            o = _rms(_recur(Q, K, V, decay), eps).flatten(1) * _silu(_lin(P, q + "g", h))
            x = x + m["left_scale"] * y + m["right_scale"] * _lin(P, q + "o", o)
        h, f = norm(x, p + "norm2"), l["mlp"]
        x = x + (_experts(P, p + "mlp.", f, h, "pitelorn") if f["kind"] == "moe" else _glu(P, p + "mlp.", h, "silu"))
    return _last(P, "head", x, eps, norm)


def _llama(sequences, device):
    """Last-token logits of whole sequences, layer by layer over all of them: a layer's weights are
    drawn as the random-weight engine draws them (seed 0) and used once."""
    c = _config(LLAMA)
    h, n, d, H, G = c.hidden_size, c.intermediate_size, c.head_dim, c.num_heads, c.num_kv_heads
    eps, rot = c.rms_norm_eps, {"dims": d, "base": c.rope_theta}

    def normal(g, *shape):
        return torch.empty(*shape, dtype=torch.bfloat16, device=device).normal_(0.0, 0.02, generator=g).to(D)

    g = torch.Generator(device=device).manual_seed(3)
    embed = normal(g, c.vocab_size, h)
    xs = [embed[torch.tensor(t, device=device)] for t in sequences]
    del embed
    head = normal(g, c.vocab_size, h)
    for i in range(c.num_layers):
        g = torch.Generator(device=device).manual_seed(i * 9176 + 1)
        wqkv, wo, wgu, wd = (normal(g, *s) for s in (((H + 2 * G) * d, h), (h, H * d), (2 * n, h), (h, n)))
        for j, x in enumerate(xs):
            q, k, v = (_rms(x, eps) @ wqkv.T).split([H * d, G * d, G * d], 1)
            hid = _hidden(len(x), device)
            o = _attend(_rotate(_heads(q, H), rot), _rotate(_heads(k, G), rot), _heads(v, G),
                        lambda a, s: _softmax(s * d ** -0.5, hid))
            x = x + o.flatten(1) @ wo.T
            a, b = (_rms(x, eps) @ wgu.T).split([n, n], 1)
            xs[j] = x + (_silu(a) * b) @ wd.T
    return torch.cat([_rms(x[-1:], eps) @ head.T for x in xs])


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    ids = tokens_of(case, seed, _config(case["model"]).vocab_size)
    with torch.no_grad():
        if case["model"] == LLAMA:
            return {"logits": _llama(ids, dev)}
        cfg, P, out = _design(case["model"])[0], _weights(case["model"], dev), []
        scale = cfg.get("embedding", {}).get("scale", 1.0)
        for t in ids:
            tok = torch.tensor(t, device=dev)
            out.append(globals()["_" + _family(case["model"])](cfg, P, tok, P["embed"][tok].to(D) * scale, cfg["norm"]["eps"]))
        return {"logits": torch.cat(out)}
