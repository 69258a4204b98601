"""What a user of this framework has it do: steps of a model (a batch of prompts, or one more token for every running
sequence) through the runner that the engine drives, and the draw of tokens from logits.

Models: a Llama-3-8B-shaped and an fp8-weight Qwen2-7B-shaped decoder (the served families, full width, four layers
each) and three hybrid designs at the sizes of the hybrid comparison (width 2048, four layers).  Weights are random and
stay with the process, as a server's do; a case's own inputs (token ids, the context already in the cache and in the
recurrent states, pages in no particular order) come from the seed.  A step's outputs are the logits of the last
position of every sequence, and the pages and states that it wrote."""
from __future__ import annotations

import gc
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-backend-public_amd"))

PAGE = 16
PARTS = 4                       # sets of sequences that may hold pages and state slots of one engine side by side
LAYERS = 4
WIDTH = 2048                    # of the hybrid designs
HYBRID_ROWS, HYBRID_LEN = 32, 2320
# model -> (most sequences, longest sequence, tokens of context one set may hold)
LIMITS = {"llama": (64, 4352, 69632), "qwen-fp8": (64, 1088, 69632), "lozupel": (HYBRID_ROWS, HYBRID_LEN, HYBRID_ROWS * HYBRID_LEN),
          "bapavik": (HYBRID_ROWS, HYBRID_LEN, HYBRID_ROWS * HYBRID_LEN), "rigazen": (HYBRID_ROWS, HYBRID_LEN, HYBRID_ROWS * HYBRID_LEN)}
STEP_TOKENS = 8192              # prompt tokens of one step: the scheduler's default budget


def listed():
    return [
        # one user's chat: the latency of a token
        {"name": "llama decode 1", "model": "llama", "step": "decode", "rows": 1, "tokens": 200, "even": True},
        # the headline workload: 32 sequences, 128 tokens in, in the middle of 128 out
        {"name": "llama decode 32", "model": "llama", "step": "decode", "rows": 32, "tokens": 256, "even": False},
        # long documents: 16 sequences past 2048 tokens in
        {"name": "llama decode 16 long", "model": "llama", "step": "decode", "rows": 16, "tokens": 4100, "even": False},
        # fp8 weights, 512 tokens in, in the middle of 512 out
        {"name": "qwen fp8 decode 64", "model": "qwen-fp8", "step": "decode", "rows": 64, "tokens": 1024, "even": False},
        # time to first token of a burst of short prompts
        {"name": "llama prompts 32x128", "model": "llama", "step": "prompts", "rows": 32, "tokens": 128, "even": True},
        # a few long prompts of odd lengths in one step
        {"name": "llama prompts long", "model": "llama", "step": "prompts", "rows": 2, "tokens": 3977, "even": False},
        # random sampling of a batch's next tokens, each request with its own temperature, top-k and top-p
        {"name": "sample 32", "model": "sampler", "step": "draw", "rows": 32, "tokens": 128256, "even": True},
        # hybrid decoders: a step's worth of prompts, and a batch in generation
        {"name": "lozupel prompts 4x2048", "model": "lozupel", "step": "prompts", "rows": 4, "tokens": 2048, "even": True},
        {"name": "lozupel decode 32", "model": "lozupel", "step": "decode", "rows": 32, "tokens": 2100, "even": False},
        {"name": "bapavik prompts ragged", "model": "bapavik", "step": "prompts", "rows": 5, "tokens": 2011, "even": False},
        {"name": "bapavik decode 32", "model": "bapavik", "step": "decode", "rows": 32, "tokens": 2100, "even": False},
        {"name": "rigazen prompts 4x2048", "model": "rigazen", "step": "prompts", "rows": 4, "tokens": 2048, "even": True},
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    model = rng.choice(["llama", "llama", "llama", "qwen-fp8", "lozupel", "bapavik", "rigazen", "sampler"])
    if model == "sampler":
        return {"model": model, "step": "draw", "rows": _between(rng, 1, 64), "tokens": rng.choice([32000, 50272, 128256, 152064]),
                "even": True}
    most, longest, room = LIMITS[model]
    if rng.random() < 0.5:
        rows = _between(rng, 1, most)
        return {"model": model, "step": "decode", "rows": rows, "tokens": _between(rng, 33, min(longest - 8, room // rows - PAGE)),
                "even": rng.random() < 0.3}
    rows = _between(rng, 1, 32)
    return {"model": model, "step": "prompts", "rows": rows, "tokens": _between(rng, 16, min(longest - 8, STEP_TOKENS // rows)),
            "even": rng.random() < 0.3}


def _lengths(case):
    """Tokens of every sequence after the step; a case's own, whatever the seed."""
    rows, top = case["rows"], case["tokens"]
    if case["even"]:
        return [top] * rows
    r = random.Random("%d %d" % (rows, top))
    return [top if i == 0 else r.randint((top + 1) // 2, top) for i in range(rows)]


# ---- models: one engine at a time stays with the process
def _config(model):
    from mi355_decode import bench_hybrid
    from mi355_decode.config import KNOWN_MODELS
    if model in ("llama", "qwen-fp8"):
        return dict(KNOWN_MODELS["llama-3-8b" if model == "llama" else "qwen2-7b"], num_hidden_layers=LAYERS)
    return {"lozupel": bench_hybrid.lozupel_config, "bapavik": bench_hybrid.bapavik_config,
            "rigazen": bench_hybrid.rigazen_config}[model](WIDTH, LAYERS)


def _checkpoint(model):
    """The model's weights under their checkpoint names, bfloat16 (tables int32), on the GPU."""
    cfg = _config(model)
    if model not in ("llama", "qwen-fp8"):
        from mi355_decode import weights
        from mi355_decode.config import ModelConfig
        return weights.hybrid_synthetic_state(ModelConfig.from_dict(cfg), seed=1, device="cuda", dtype=torch.bfloat16)
    gen = torch.Generator(device="cuda").manual_seed(1)
    H, F, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
    nh, nkv = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    d = H // nh

    def mat(*shape, s=None, mean=0.0):
        return torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(mean, s or shape[-1] ** -0.5, generator=gen)

    st = {"model.embed_tokens.weight": mat(V, H, s=1.0), "model.norm.weight": mat(H, s=0.1, mean=1.0), "lm_head.weight": mat(V, H)}
    for i in range(LAYERS):
        p = "model.layers.%d." % i
        for n, rows in (("q", nh * d), ("k", nkv * d), ("v", nkv * d)):
            st[p + "self_attn.%s_proj.weight" % n] = mat(rows, H)
            if model == "qwen-fp8":
                st[p + "self_attn.%s_proj.bias" % n] = mat(rows, s=0.2)
        st[p + "self_attn.o_proj.weight"] = mat(H, nh * d)
        st[p + "mlp.gate_proj.weight"], st[p + "mlp.up_proj.weight"], st[p + "mlp.down_proj.weight"] = mat(F, H), mat(F, H), mat(H, F)
        st[p + "input_layernorm.weight"], st[p + "post_attention_layernorm.weight"] = mat(H, s=0.1, mean=1.0), mat(H, s=0.1, mean=1.0)
    return st


class _Engine:
    def __init__(self, model):
        from mi355_decode.config import EngineArgs, ModelConfig
        from mi355_decode.llm import build_engine
        most, longest, room = LIMITS[model]
        self.model, self.hybrid = model, model not in ("llama", "qwen-fp8")
        self.part_pages = (room + PAGE - 1) // PAGE + most
        self.part_slots, self.next_part = most, 0
        args = EngineArgs(model=model, dtype="bfloat16", max_num_seqs=most * PARTS if self.hybrid else most, max_model_len=longest,
                          max_num_batched_tokens=STEP_TOKENS, quantization="fp8" if model == "qwen-fp8" else None,
                          num_gpu_blocks_override=self.part_pages * PARTS)
        self.runner = build_engine(args, state_dict=_checkpoint(model), model_config=ModelConfig.from_dict(_config(model))).runner

    def pages(self):
        r = self.runner
        return list(r.k_cache) + list(r.v_cache) + [t for pair in getattr(r, "latent_cache", []) for t in pair if t is not None]


_engine = {}


def _get_engine(model):
    if model not in _engine:
        _engine.clear()
        gc.collect()
        torch.cuda.empty_cache()
        _engine[model] = _Engine(model)
    return _engine[model]


def _tokens(case, seed):
    """Token ids of every sequence."""
    vocab = _config(case["model"]).get("vocab_size") or _config(case["model"])["vocab"]
    rng = np.random.default_rng([seed, 7])
    return [rng.integers(0, vocab, n) for n in _lengths(case)]


def _prompt_step(e, chunks, tables, slots):
    """The arguments of the runner's step over chunks [(sequence, first position, ids)]."""
    ids, pos, where, cu = [], [], [], [0]
    for s, first, t in chunks:
        p = np.arange(first, first + len(t), dtype=np.int64)
        ids.append(np.asarray(t, dtype=np.int64))
        pos.append(p)
        where.append(tables[s, p // PAGE].astype(np.int64) * PAGE + p % PAGE)
        cu.append(cu[-1] + len(t))
    seqs = [c[0] for c in chunks]
    args = [np.concatenate(ids), np.concatenate(pos), np.concatenate(where), np.ascontiguousarray(tables[seqs]),
            np.asarray(cu, dtype=np.int32), np.asarray([c[1] + len(c[2]) for c in chunks], dtype=np.int32)]
    return args, max(len(c[2]) for c in chunks), np.asarray([slots[s] for s in seqs], dtype=np.int32)


def prepare(case, seed):
    if case["model"] == "sampler":
        return _prepare_sampler(case, seed)
    e = _get_engine(case["model"])
    r, lens, toks = e.runner, _lengths(case), _tokens(case, seed)
    rng = np.random.default_rng([seed, 11])
    part, e.next_part = e.next_part, (e.next_part + 1) % PARTS
    need = [(n + PAGE - 1) // PAGE for n in lens]
    at, used = part * e.part_pages, sum(need)
    order = (at + rng.permutation(used)).astype(np.int32)          # pages as a pool in use hands them out
    tables, k = np.zeros((len(lens), r.max_blocks), dtype=np.int32), 0
    for s, n in enumerate(need):
        tables[s, :n] = order[k:k + n]
        k += n
    slots = [part * e.part_slots + s for s in range(len(lens))]
    pages = [t[at:at + used] for t in e.pages()]
    for t in pages:
        t.zero_()
    states = [t[slots[0]:slots[0] + len(slots)] for t in getattr(r, "rec_state", [])]
    st = {"e": e, "step": case["step"], "rows": len(lens), "pages": pages, "states": states}
    if case["step"] == "prompts":
        args, longest, sl = _prompt_step(e, [(s, 0, t) for s, t in enumerate(toks)], tables, slots)
        if e.hybrid:
            last = args[4][1:] - 1
            st.update(args=args + [longest], kw={"state_slots": sl, "logit_rows": last.astype(np.int64)})
        else:
            st.update(args=[torch.from_numpy(a).cuda() for a in args] + [longest])
        return st
    todo = []                                                     # the context: prompts of all but the last token
    for s in range(len(lens) + 1):
        if todo and (s == len(lens) or sum(len(c[2]) for c in todo) + lens[s] > 2 * STEP_TOKENS):
            args, longest, sl = _prompt_step(e, todo, tables, slots)
            r.run_prefill(*args, longest, **({"state_slots": sl} if e.hybrid else {}))
            todo = []
        if s < len(lens):
            todo.append((s, 0, toks[s][:-1]))
    # the decode step's inputs: ids, positions, cache slots | context lengths, page tables (, state slots)
    B, MB, n = r.max_num_seqs, r.max_blocks, len(lens)
    n64, n32 = np.full(3 * B, -1, dtype=np.int64), np.zeros(r.inall.numel() - 6 * B, dtype=np.int32)
    n64[:2 * B] = 0
    for s in range(n):
        p = lens[s] - 1
        n64[s], n64[B + s], n64[2 * B + s] = toks[s][-1], p, int(tables[s, p // PAGE]) * PAGE + p % PAGE
    n32[:n] = lens
    n32[B:B + n * MB] = tables.reshape(-1)
    if e.hybrid:
        n32[B + B * MB:] = r.num_state_slots
        n32[B + B * MB:B + B * MB + n] = slots
    st["inputs"] = torch.from_numpy(np.concatenate([n64.view(np.int32), n32])).cuda()
    return st


def run(state):
    if state["step"] == "draw":
        from mi355_decode import ops
        return ops.sample(*state["args"])
    r = state["e"].runner
    if state["step"] == "decode":
        r.inall.copy_(state["inputs"])
        r.decode(state["rows"])
        logits = r.logits[:state["rows"]]
    elif state["e"].hybrid:
        logits = r.run_prefill(*state["args"], **state["kw"])
    else:
        _, logits = r.prefill(*state["args"])
    return {"logits": logits, "pages": state["pages"], "states": state["states"]}


def _prepare_sampler(case, seed):
    B, V = case["rows"], case["tokens"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rank = torch.rand(B, V, device="cuda", generator=gen).argsort(dim=1).float() + 1.0      # a language model's long tail
    logits = (12.0 - 1.5 * rank.log() + 0.5 * torch.randn(B, V, device="cuda", generator=gen)).to(torch.bfloat16)
    r = random.Random("%d" % seed)
    forms = [(1.0, 0, 1.0), (0.8, 0, 0.95), (0.7, 50, 1.0), (1.0, 40, 0.9), (0.0, 0, 1.0)]
    mine = [forms[i % len(forms)] for i in range(B)]
    return {"step": "draw", "args": (logits, torch.tensor([m[0] for m in mine], device="cuda"),
                                     torch.tensor([m[1] for m in mine], dtype=torch.int32, device="cuda"),
                                     torch.tensor([m[2] for m in mine], device="cuda"),
                                     torch.tensor([r.getrandbits(62) for _ in mine], device="cuda"),
                                     torch.tensor([r.randrange(500) for _ in mine], device="cuda"))}


# ---- what a pass cannot do without
_shapes = {}


def _sizes(model):
    if model not in _shapes:
        _shapes[model] = {k: tuple(t.shape) for k, t in _checkpoint(model).items()}
    return _shapes[model]


def _layer_runs(cfg):
    n, lp = len(cfg["layers"]), cfg.get("loop")
    if not lp:
        return list(range(n))
    return list(range(lp["start"])) + list(range(lp["start"], lp["stop"])) * lp["times"] + list(range(lp["stop"], n))


def work(case):
    if case["model"] == "sampler":
        return {"bytes": 2 * case["rows"] * case["tokens"], "flops": 4 * case["rows"] * case["tokens"]}
    cfg, lens, rows = _config(case["model"]), _lengths(case), case["rows"]
    hybrid, decode = "layers" in cfg, case["step"] == "decode"
    tokens = rows if decode else sum(lens)
    runs = _layer_runs(cfg) if hybrid else range(LAYERS)
    wide = 1 if case["model"] == "qwen-fp8" else 2
    byts, flops = 0.0, 0.0
    for name, shape in _sizes(case["model"]).items():
        if len(shape) != 2 or "embed" in name or name.endswith(("table", ".conv")) or name == "loop.step":
            continue
        size = shape[0] * shape[1]
        if name in ("lm_head.weight", "head"):
            byts, flops = byts + 2 * size, flops + 2.0 * size * rows
            continue
        i = int(name.split(".")[2] if not hybrid else name[1:name.index(".")])
        times, share, seen = runs.count(i) if hybrid else 1, 1.0, 1.0
        if hybrid and cfg["layers"][i].get("mlp", {}).get("kind") == "moe" and ".mlp.e" in name:
            m = cfg["layers"][i]["mlp"]["router"]
            share = m["top"] / m["experts"]
            seen = 1.0 - (1.0 - share) ** tokens
        byts += times * seen * wide * size
        flops += times * share * 2.0 * size * tokens
    if case["model"] == "rigazen":                                # the head is the embedding
        size = cfg["vocab"] * cfg["width"]
        byts, flops = byts + 2 * size, flops + 2.0 * size * rows
    width, vocab = (cfg["width"], cfg["vocab"]) if hybrid else (cfg["hidden_size"], cfg["vocab_size"])
    byts += tokens * width * 2 + rows * vocab * (2 if decode or not hybrid else 4)

    def seen_keys(window=0):
        """(query, key) pairs, keys read by a decode step."""
        cut = [min(n, window or n) for n in lens]
        pairs = sum(cut) if decode else sum(n * (n + 1) / 2 - (n - c) * (n - c + 1) / 2 for n, c in zip(lens, cut))
        return pairs, (sum(cut) if decode else sum(lens))

    def attention(heads, kv, d, dv, window=0):
        pairs, keys = seen_keys(window)
        return 2.0 * kv * (d + dv) * keys, 2.0 * heads * (d + dv) * pairs

    def memory(heads, d, dv, ops_):
        return 8.0 * rows * heads * d * dv, ops_ * heads * d * dv * tokens

    for i in runs:
        parts = []
        if not hybrid:
            d = cfg["hidden_size"] // cfg["num_attention_heads"]
            parts.append(attention(cfg["num_attention_heads"], cfg["num_key_value_heads"], d, d))
        else:
            L = cfg["layers"][i]
            m = L["mixer"]
            a = m.get("left", m)
            if L["type"] in ("attention", "parallel"):
                parts.append(attention(a["heads"], a["kv_heads"], a["dim"], a["vdim"], (a.get("mask") or {}).get("size") or 0))
            if L["type"] == "latent_attention":
                pairs, keys = seen_keys()
                parts.append((2.0 * (m["kv_rank"] + m["rot_dim"]) * keys, 2.0 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]) * pairs))
            if L["type"] in ("delta", "mlstm", "parallel"):
                b = m.get("right", m)
                parts.append(memory(b["heads"], b["dim"], b["vdim"], 6.0 if case["model"] == "lozupel" else 4.0))
        for x, y in parts:
            byts, flops = byts + x, flops + y
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    if case["model"] == "sampler":
        return "exact"
    # bfloat16 activations through four to six layers
    return {"rel": 0.03, "max": 0.5}


# ---- the same in 64 bits
def exact(case, seed):
    if case["model"] == "sampler":
        return None
    w = _checkpoint(case["model"])
    lens, toks = _lengths(case), _tokens(case, seed)
    L = max(lens)
    ids = torch.from_numpy(np.stack([np.pad(t, (0, L - len(t))) for t in toks])).cuda()
    n = torch.tensor(lens, device="cuda")
    f = {"llama": _llama64, "qwen-fp8": _llama64, "lozupel": _lozupel64, "bapavik": _bapavik64, "rigazen": _rigazen64}[case["model"]]
    logits, states = f(_config(case["model"]), w, ids, n, case["model"])
    return {"logits": logits, "pages": None, "states": states}


def _d(t):
    return t.double()


def _lin(x, t):
    return x @ _d(t).t()


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _last(x, n):
    return x[torch.arange(x.shape[0], device=x.device), n - 1]


def _turn(x, dims, base, neighbours=False):
    """x [R, T, heads, d]: the first `dims` coordinates of position t turned by t base^(-2i / dims); pairs
    (i, i + dims / 2), or (2i, 2i + 1)."""
    i = torch.arange(dims // 2, dtype=torch.float64, device=x.device)
    a = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * base ** (-2.0 * i / dims)
    c, s = a.cos()[None, :, None, :], a.sin()[None, :, None, :]
    y = x.clone()
    u, v = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
    y[..., u], y[..., v] = x[..., u] * c - x[..., v] * s, x[..., v] * c + x[..., u] * s
    return y


def _attend(q, k, v, scale, window=0, keep=0, cap=0.0, sink=None, sigmoid=None):
    """Causal attention, a head at a time.  sigmoid: (factor, bias) per head of weights that are not normalised."""
    R, T, H, _ = q.shape
    rep = H // k.shape[2]
    i, j = torch.arange(T, device=q.device)[:, None], torch.arange(T, device=q.device)[None, :]
    seen = j <= i
    if window:
        seen = seen & ((i - j < window) | (j < keep))
    out = []
    for h in range(H):
        s = (q[:, :, h] @ k[:, :, h // rep].transpose(1, 2).contiguous()) * scale
        if sigmoid is not None:
            p = torch.sigmoid(s * sigmoid[0][h] + sigmoid[1][h]) * seen
        else:
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(~seen, -math.inf)
            top = s.amax(-1, keepdim=True)
            top = top if sink is None else torch.maximum(top, sink[h])
            p = torch.exp(s - top)
            p = p / (p.sum(-1, keepdim=True) + (0.0 if sink is None else torch.exp(sink[h] - top)))
        out.append(p @ v[:, :, h // rep])
    return torch.stack(out, dim=2).flatten(2)


def _llama64(cfg, w, ids, n, model):
    H, nh, nkv, eps = cfg["hidden_size"], cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["rms_norm_eps"]
    d, base = H // nh, cfg.get("rope_theta", 10000.0)

    def weight(name):
        t = _d(w[name])
        if model == "qwen-fp8":                                   # one scale a row, 8-bit numbers
            s = w[name].float().abs().amax(dim=1, keepdim=True) / 448.0
            t = (w[name].float() / s).to(torch.float8_e4m3fn).double() * s.double()
        return t

    x = _d(w["model.embed_tokens.weight"][ids])
    R, T = ids.shape
    for i in range(LAYERS):
        p = "model.layers.%d." % i
        h = _rms(x, eps) * _d(w[p + "input_layernorm.weight"])
        q, k, v = (h @ weight(p + "self_attn.%s_proj.weight" % c).t() + (_d(w[p + "self_attn.%s_proj.bias" % c])
                   if p + "self_attn.%s_proj.bias" % c in w else 0.0) for c in "qkv")
        q, k = _turn(q.view(R, T, nh, d), d, base), _turn(k.view(R, T, nkv, d), d, base)
        x = x + _attend(q, k, v.view(R, T, nkv, d), d ** -0.5) @ weight(p + "self_attn.o_proj.weight").t()
        h = _rms(x, eps) * _d(w[p + "post_attention_layernorm.weight"])
        g = torch.nn.functional.silu(h @ weight(p + "mlp.gate_proj.weight").t()) * (h @ weight(p + "mlp.up_proj.weight").t())
        x = x + g @ weight(p + "mlp.down_proj.weight").t()
    return _lin(_rms(_last(x, n), eps) * _d(w["model.norm.weight"]), w["lm_head.weight"]), []


def _delta64(w, p, m, h, eps, n):
    """The gated delta rule over whole sequences: (result, state after the last token of each)."""
    R, T, _ = h.shape
    H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]

    def conv(c):
        t = _d(w[p + c + ".conv"])
        x = torch.nn.functional.pad(_lin(h, w[p + c]), (0, 0, t.shape[1] - 1, 0))
        return torch.nn.functional.silu(sum(x[:, j:j + T] * t[:, j] for j in range(t.shape[1])))

    def unit(x):
        return (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, dim=2)

    q, k, v = unit(conv("q").view(R, T, G, d)) * d ** -0.5, unit(conv("k").view(R, T, G, d)), conv("v").view(R, T, H, dv)
    alive = (torch.arange(T, device=h.device)[None, :] < n[:, None]).double()[..., None]
    beta = torch.sigmoid(_lin(h, w[p + "b"])) * alive
    rate = torch.exp(_d(w[p + "A_log"]))
    if p + "a1" in w:
        z = _lin(_lin(h, w[p + "a1"]), w[p + "a2"]) + _d(w[p + "dt_bias"])
        decay = torch.exp(-rate[:, None] * torch.nn.functional.softplus(z).view(R, T, H, d) * alive[..., None])
        gate = torch.sigmoid(_lin(_lin(h, w[p + "g1"]), w[p + "g2"]))
    else:
        decay = torch.exp(-rate * torch.nn.functional.softplus(_lin(h, w[p + "a"]) + _d(w[p + "dt_bias"])) * alive)[..., None]
        gate = torch.nn.functional.silu(_lin(h, w[p + "g"]))
    S, o = h.new_zeros(R, H, d, dv), h.new_zeros(R, T, H, dv)
    for t in range(T):
        S = S * decay[:, t, :, :, None]
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None, :] @ S).squeeze(2))
        S = S + k[:, t, :, :, None] * u[:, :, None, :]
        o[:, t] = (q[:, t, :, None, :] @ S).squeeze(2)
    o = (_rms(o, eps) * _d(w[p + "norm"])).flatten(2) * gate
    return _lin(o, w[p + "o"]), S


def _lozupel64(cfg, w, ids, n, _):
    eps = cfg["norm"]["eps"]
    R, T = ids.shape
    x = x0 = _d(w["embed"][ids]) * cfg["embedding"]["scale"]
    lp, states, done = cfg.get("loop"), [], 0
    for i in _layer_runs(cfg):
        L, p = cfg["layers"][i], "l%d." % i
        if lp and i == lp["start"]:
            x = x + (x0 if done else 0.0) + _d(w["loop.step"][done])
            done += 1
        h = _rms(x, eps) * _d(w[p + "norm1"])
        if L["type"] == "delta":
            y, S = _delta64(w, p + "mix.", L["mixer"], h, eps, n)
            x = x + y
        else:
            a, m = p + "mix.left.", L["mixer"]["left"]
            rot = m["rot"]
            q = _turn(_lin(h, w[a + "q"]).view(R, T, m["heads"], -1), rot["dims"], rot["base"])
            k = _turn(_lin(h, w[a + "k"]).view(R, T, m["kv_heads"], -1), rot["dims"], rot["base"])
            v = _lin(h, w[a + "v"]).view(R, T, m["kv_heads"], -1)
            o = _attend(q, k, v, m["scale"], m["mask"]["size"], sigmoid=(_d(w[a + "temp"]), _d(w[a + "pb"])))
            o = (o.view(R, T, m["heads"], -1) * torch.sigmoid(_lin(h, w[a + "g"]))[..., None]).flatten(2)
            y, S = _delta64(w, p + "mix.right.", L["mixer"]["right"], h, eps, n)
            x = x + 0.5 * (_rms(_lin(o, w[a + "o"]), eps) * _d(w[a + "out"]) + _rms(y, eps) * _d(w[p + "mix.right.out"]))
        states.append(S)
        h = _rms(x, eps) * _d(w[p + "norm2"])
        g = torch.nn.functional.gelu(_lin(h, w[p + "mlp.gate"]), approximate="tanh") * _lin(h, w[p + "mlp.up"])
        x = x + _lin(g, w[p + "mlp.down"])
    z, cap = _lin(_rms(_last(x, n), eps) * _d(w["final.norm"]), w["head"]), cfg["logit_softcap"]
    return cap * torch.tanh(z / cap), states


def _bapavik64(cfg, w, ids, n, _):
    eps = cfg["norm"]["eps"]
    R, T = ids.shape
    x = _d(w["embed"][ids]) * cfg["embedding"]["scale"]

    def ln(x, g):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], _d(g), None, eps)

    for i in _layer_runs(cfg):
        L, p = cfg["layers"][i], "l%d." % i
        m, a, f = L["mixer"], p + "mix.", p + "mlp."
        h = ln(x, w[p + "norm1"])
        if L["type"] == "attention":
            qt = m["q_temp"]
            pos = torch.arange(T, dtype=torch.float64, device=x.device)
            temp = 1.0 + qt["coef"] * torch.log(torch.floor((pos + 1) / qt["every"]) + 1)
            q = _rms(_lin(h, w[a + "q"]), eps) * _d(w[a + "q.norm"]) * temp[:, None]
            k = _rms(_lin(h, w[a + "k"]), eps) * _d(w[a + "k.norm"])
            v = _lin(h, w[a + "v"]).view(R, T, m["kv_heads"], -1)
            o = _attend(q.view(R, T, m["heads"], -1), k.view(R, T, m["kv_heads"], -1), v, m["scale"], cap=m["softcap"], sink=_d(w[a + "sink"]))
        else:
            H, d, r, rot = m["heads"], m["dim"], m["kv_rank"], m["rot"]
            q, z = _lin(h, w[a + "q"]).view(R, T, H, -1), _lin(h, w[a + "dkv"])
            c = _rms(z[..., :r], eps) * _d(w[a + "dkv.norm"])
            kr = _turn(z[..., r:].reshape(R, T, 1, -1), rot["dims"], rot["base"], neighbours=True)
            q = torch.cat([q[..., :d], _turn(q[..., d:].contiguous(), rot["dims"], rot["base"], neighbours=True)], dim=-1)
            k = torch.cat([_lin(c, w[a + "uk"]).view(R, T, H, d), kr.expand(R, T, H, -1)], dim=-1)
            o = _attend(q, k, _lin(c, w[a + "uv"]).view(R, T, H, -1), m["scale"])
        x = x + _lin(o, w[a + "o"])
        h, mlp = ln(x, w[p + "norm2"]), L["mlp"]
        if mlp["kind"] == "dense":
            g, u = _lin(h, w[f + "gate"]).clamp(max=mlp["limit"]), _lin(h, w[f + "up"]).clamp(-mlp["limit"], mlp["limit"])
            x = x + _lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), w[f + "down"])
            continue
        flat, names, y = h.flatten(0, 1), w[f + "table"][ids.flatten()].long(), torch.zeros_like(h).flatten(0, 1)
        for e in range(mlp["router"]["experts"]):
            rows = (names == e).any(dim=1).nonzero()[:, 0]
            y[rows] += _lin(torch.relu(_lin(flat[rows], w["%se%d.up" % (f, e)])) ** 2, w["%se%d.down" % (f, e)]) / mlp["router"]["top"]
        x = x + y.view_as(x)
    return _lin(ln(_last(x, n), w["final.norm"]), w["head"]), []


def _rigazen64(cfg, w, ids, n, _):
    eps, side = cfg["norm"]["eps"], cfg["token_side"]["dim"]
    R, T = ids.shape
    silu = torch.nn.functional.silu
    x = _d(w["embed"][ids]) * cfg["embedding"]["scale"]
    for i, L in enumerate(cfg["layers"]):
        p, a, m = "l%d." % i, "l%d.mix." % i, L["mixer"]
        if L["type"] == "mlstm":
            H, d, cap = m["heads"], m["dim"], m["gate_cap"]
            q, k, v = (_lin(x, w[a + c]).view(R, T, H, -1) for c in "qkv")
            q = q * d ** -0.5
            gi = cap * torch.tanh((_lin(x, w[a + "i"]) + _d(w[a + "i.b"])) / cap)
            gf = torch.nn.functional.logsigmoid(cap * torch.tanh((_lin(x, w[a + "f"]) + _d(w[a + "f.b"])) / cap))
            C, N, M, o = x.new_zeros(R, H, d, v.shape[-1]), x.new_zeros(R, H, d), x.new_zeros(R, H), torch.empty_like(v)
            for t in range(T):
                top = torch.maximum(gf[:, t] + M, gi[:, t])
                keep, add = torch.exp(gf[:, t] + M - top), torch.exp(gi[:, t] - top)
                C = keep[..., None, None] * C + (add[..., None] * k[:, t])[..., :, None] * v[:, t, :, None, :]
                N, M = keep[..., None] * N + add[..., None] * k[:, t], top
                den = torch.maximum((N * q[:, t]).sum(-1).abs(), torch.exp(-M)) + 1e-6
                o[:, t] = (q[:, t, :, None, :] @ C).squeeze(2) / den[..., None]
            y = _lin(_rms(o, eps).flatten(2) * _d(w[a + "norm"]) * torch.sigmoid(_lin(x, w[a + "g"])), w[a + "o"])
        else:
            b, l, c = a + "left.", m["left"], a + "right."
            q, k, v = (_lin(x, w[b + s]) + _d(w[b + s + ".b"]) for s in "qkv")
            q, k = (_rms(z, eps) * _d(w[b + s + ".norm"]) for s, z in (("q", q), ("k", k)))
            q, k = (_turn(z.view(R, T, g, -1), l["rot"]["dims"], l["rot"]["base"]) for z, g in ((q, l["heads"]), (k, l["kv_heads"])))
            o = _attend(q, k, v.view(R, T, l["kv_heads"], -1), l["scale"], l["mask"]["size"], l["mask"]["keep_first"])
            y = m["left_scale"] * _lin(o, w[b + "o"])
            q, k, v = (silu(_lin(x, w[c + s])).view(R, T, m["right"]["heads"], -1) for s in "qkv")
            dec = torch.tensor(m["right"]["decay"], dtype=torch.float64, device=x.device)[:, None, None]
            S, o = x.new_zeros(R, q.shape[2], q.shape[3], v.shape[3]), torch.empty_like(v)
            for t in range(T):
                S = dec * S + k[:, t, :, :, None] * v[:, t, :, None, :]
                o[:, t] = (q[:, t, :, None, :] @ S).squeeze(2)
            y = y + m["right_scale"] * _lin(_rms(o.flatten(2), eps) * _d(w[c + "norm"]) * torch.sigmoid(_lin(x, w[c + "g"])), w[c + "o"])
        x = x + _rms(y, eps) * (1.0 + _d(w[p + "norm1"]))
        x = x + _rms(_lin(torch.relu(_lin(x, w[p + "mlp.up"])) ** 2, w[p + "mlp.down"]), eps) * (1.0 + _d(w[p + "norm2"]))
        e = _d(w["side.embed"][ids][..., i * side:(i + 1) * side])
        g = torch.nn.functional.gelu(_lin(x, w[p + "side.gate"]), approximate="tanh") * e
        x = x + _rms(_lin(g, w[p + "side.proj"]), eps) * _d(w[p + "side.norm"])
    return _lin(_rms(_last(x, n), eps) * (1.0 + _d(w["final.norm"])), w["embed"]), [None] * LAYERS
