"""The work that a user of this engine has it do, as cases that can be timed and compared.

A case is a batch of requests taken from their prompts to their last tokens through the engine's step function: the prompts are fed
under a budget of tokens a step, as the scheduler does it (every decoding request's token first, then portions of prompts in the order
of arrival), and every request then takes ``new`` given tokens one a step, so that the outputs are logits that another
implementation can be compared with, and not a sampled text that parts at the first rounding.  Its fields:

    model      an entry of ``MODELS``: Qwen2 in the three sizes of the benchmark's configurations (all layers), and three of the further
               designs in the benchmark's "small" and "medium" sizes: experts (livovik), state spaces, differential and latent attention
               with experts over several streams (befirax), the delta rule and linear attention (salolorn)
    dtype      bf16, f16 or f32
    requests   how many requests
    prompt     tokens of the longest prompt; with ``ragged`` the others are shorter, down to a third, at odd lengths
    new        tokens that every request takes one at a time after its prompt
    scored     places at a prompt's end whose logits are wanted (1: the next token; more: the likelihood of a continuation)
    budget     most tokens of a step
    page       tokens a cache page
"""
from __future__ import annotations

import math

import torch

from machserve_amd.config import config_from_dict
from machserve_amd.engine import StepEntry, load_model
from machserve_amd.weights import random_tensor_dict

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
DEVICE = "cuda:0"
WARM_PASSES = 4  # a step's shape is captured when it has come three times: a server that runs has its steps captured

# ------------------------------------------------------------------------------------ models


def _qwen(hidden, layers, heads, kv, ff, vocab, tied):
    return {"architectures": ["Qwen2ForCausalLM"], "model_type": "qwen2", "hidden_size": hidden, "num_hidden_layers": layers,
            "num_attention_heads": heads, "num_key_value_heads": kv, "intermediate_size": ff, "vocab_size": vocab,
            "max_position_embeddings": 32768, "rms_norm_eps": 1e-6, "rope_theta": 1000000.0, "tie_word_embeddings": tied,
            "hidden_act": "silu", "use_sliding_window": False}


def _livovik(w, ff, H, kv, hd, window):
    att = {"heads": H, "kv_heads": kv, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "mask": {"size": window},
           "rot": {"base": 500000.0, "dims": hd // 2, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 1024}}}
    moe = {"kind": "moe", "expert": {"ff": ff // 2}, "router": {"experts": 8, "top": 2}, "shared": {"ff": ff // 2}}
    layers = [{"type": "attention", "mixer": att, "mlp": {"kind": "dense", "ff": ff}}, {"type": "attention", "mixer": att, "mlp": moe}]
    return {"architecture": "Livovik", "vocab": 32000, "width": w, "norm": {"eps": 1e-6}, "postln_alpha": 2.0, "layers": layers * 2}


def _befirax(w, ff, H, kv, hd, window):
    moe = {"kind": "moe", "expert": {"ff": ff // 2}, "router": {"experts": 8, "top": 2, "identity": 1}}
    att = {"heads": H // 2, "kv_heads": max(kv // 2, 1), "dim": hd, "vdim": hd, "scale": hd ** -0.5, "diff": 0.3, "conv": 4,
           "rot": {"base": 10000.0, "dims": hd // 2}}
    lat = {"heads": H, "dim": hd, "rot_dim": 64, "vdim": hd, "kv_rank": 192, "scale": (hd + 64) ** -0.5, "mask": {"size": window},
           "rot": {"base": 10000.0, "dims": 64}}
    ssd = {"heads": 2 * w // 64, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
    layers = [{"type": "mamba2", "mixer": ssd, "mlp": moe}, {"type": "attention", "mixer": att, "mlp": moe},
              {"type": "latent_attention", "mixer": lat, "mlp": moe}, {"type": "attention", "mixer": dict(att, kv_from=1), "mlp": moe}]
    return {"architecture": "Befirax", "vocab": 32000, "width": w, "norm": {"eps": 1e-6}, "streams": 2, "layers": layers}


def _salolorn(w, ff, H, kv, hd, window):
    mlp = {"kind": "dense", "ff": ff}
    delta = {"type": "delta", "mixer": {"heads": H, "kv_heads": H // 2, "dim": hd, "vdim": hd, "conv": 4}, "mlp": mlp}
    lat = {"type": "latent_attention", "mlp": mlp,
           "mixer": {"heads": H, "dim": hd, "rot_dim": 64, "vdim": hd, "kv_rank": 192, "scale": (hd + 64) ** -0.5, "rot": {"base": 10000.0, "dims": 64}}}
    left = {"heads": H, "kv_heads": kv, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "mask": {"size": window}, "rot": {"base": 250000.0, "dims": hd}}
    par = {"type": "parallel", "mlp": mlp, "mixer": {"left": left, "right": {"heads": H, "dim": hd // 2, "vdim": hd, "tau": 16.0},
                                                     "left_scale": 1.2, "right_scale": 1.1}}
    return {"architecture": "Salolorn", "vocab": 32000, "width": w, "norm": {"eps": 1e-6}, "logit_scale": 0.5, "layers": [delta, lat, par, delta]}


_SMALL, _MEDIUM = (1024, 2816, 8, 2, 128, 512), (2048, 5632, 16, 4, 128, 1024)  # the benchmark's sizes of the further designs

MODELS = {
    "qwen2-0.5b": _qwen(896, 24, 14, 2, 4864, 151936, True),
    "qwen2-1.5b": _qwen(1536, 28, 12, 2, 8960, 151936, True),
    "qwen2-7b": _qwen(3584, 28, 28, 4, 18944, 152064, False),
    "livovik-small": _livovik(*_SMALL), "livovik-medium": _livovik(*_MEDIUM),
    "befirax-small": _befirax(*_SMALL), "befirax-medium": _befirax(*_MEDIUM),
    "salolorn-small": _salolorn(*_SMALL), "salolorn-medium": _salolorn(*_MEDIUM),
}

# ------------------------------------------------------------------------------------ cases


def _case(name, model, dtype, requests, prompt, new, ragged=False, scored=1, budget=2048, page=64):
    return {"name": name, "model": model, "dtype": dtype, "requests": requests, "prompt": prompt, "new": new, "ragged": ragged,
            "scored": scored, "budget": budget, "page": page}


def listed():
    return [
        # one person at a prompt: a short question and the first tokens of its answer, bound by launches and latency
        _case("chat of one", "qwen2-0.5b", "bf16", 1, 17, 16),
        # eight long conversations: the benchmark's batch and context, from the prompts on
        _case("eight long contexts", "qwen2-0.5b", "bf16", 8, 2048, 32),
        # a busy server in half precision: 64 requests of unequal lengths, decoding beside prompts that still come in
        _case("64 requests", "qwen2-0.5b", "f16", 64, 512, 24, ragged=True),
        # one long prompt in one step: the benchmark's prefill
        _case("prompt of 2048", "qwen2-0.5b", "bf16", 1, 2048, 0),
        # the 32-bit path: a few unequal requests under the engine's default budget, small pages
        _case("32-bit", "qwen2-0.5b", "f32", 3, 501, 8, ragged=True, budget=512, page=16),
        # the largest configuration, in half precision: its prefill, and a batch that decodes
        _case("7b prompt of 2048", "qwen2-7b", "f16", 1, 2048, 0),
        _case("7b batch of 16", "qwen2-7b", "f16", 16, 96, 16, ragged=True),
        # layers with experts: a prompt whose continuation is scored, and a small batch that decodes
        _case("experts prompt", "livovik-medium", "bf16", 1, 2048, 0, scored=64),
        _case("experts batch of 4", "livovik-medium", "bf16", 4, 120, 32, ragged=True, scored=16),
        # state spaces, differential and latent attention with experts over two streams: three unequal prompts in one step
        _case("streams and experts prompts", "befirax-medium", "bf16", 3, 877, 0, ragged=True, scored=32),
        # the delta rule, latent attention, and chunked attention beside linear attention: a long odd prompt, a batch that decodes
        _case("delta rule prompt", "salolorn-medium", "bf16", 1, 3001, 0, scored=64),
        _case("delta rule batch of 16", "salolorn-medium", "bf16", 16, 200, 24, ragged=True),
    ]


_PROMPT_TOKENS = {"qwen2-0.5b": 16384, "qwen2-1.5b": 6144, "qwen2-7b": 1536}  # most prompt tokens of a drawn case; the designs: 4096


def draw(rng):
    family = rng.choice(["qwen2-0.5b", "qwen2-0.5b", "qwen2-1.5b", "qwen2-7b", "livovik", "livovik", "befirax", "befirax", "salolorn", "salolorn"])
    design = not family.startswith("qwen2")
    model = family + "-" + rng.choice(["small", "medium"]) if design else family
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    if model == "qwen2-7b" or (model == "qwen2-1.5b" and dtype == "f32"):
        dtype = "f16"  # (28 layers of the 7B's width in bfloat16 are 3.5 % off the exact logits: little to compare by)
    most = _PROMPT_TOKENS.get(model, 4096) // (16 if dtype == "f32" else 1)
    prefill = rng.random() < 0.4
    log = lambda a, b: max(a, min(b, int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))))  # noqa: E731
    requests = log(1, 4) if prefill else log(1, 16 if design or model == "qwen2-7b" else 64)
    prompt = log(64 if prefill else 8, max(64, min(4096, most // requests)))
    new = 0 if prefill else rng.randint(4, 24)
    # logits at a prompt's end are those of a continuation where experts are chosen: a single row says little about them
    scored = min(prompt // 3, rng.randint(24, 64)) if design and prefill else 1
    return {"model": model, "dtype": dtype, "requests": requests, "prompt": prompt, "new": new, "ragged": requests > 1, "scored": max(1, scored),
            "budget": rng.choice([512, 1024, 2048]), "page": rng.choice([16, 64])}


def _lengths(case):
    """Tokens of every request's prompt: the longest, and with ``ragged`` the others down to a third of it."""
    n, p = case["requests"], case["prompt"]
    if not case["ragged"]:
        return [p] * n
    return [max(1, case["scored"], p - (p * 2 // 3) * ((7 * i) % n) // n) for i in range(n)]


def _schedule(case):
    """The steps of a pass: lists of (request, first token, tokens, wanted places among them)."""
    lengths, new, scored = _lengths(case), case["new"], case["scored"]
    total = [n + new for n in lengths]
    done, steps = [0] * len(lengths), []
    while any(d < t for d, t in zip(done, total)):
        step, room = [], case["budget"]
        for i, d in enumerate(done):  # decoded tokens first
            if lengths[i] <= d < total[i] and room:
                step.append((i, d, 1, (0,)))
                room -= 1
        for i, d in enumerate(done):
            if d < lengths[i] and room:
                n = min(room, lengths[i] - d)
                step.append((i, d, n, tuple(range(max(0, lengths[i] - scored - d), n))))
                room -= n
        for i, _, n, _ in step:
            done[i] += n
        steps.append(step)
    return steps


def _config(case):
    return config_from_dict(MODELS[case["model"]])


def _weights(case, seed):
    """Random weights by the laws of the engine's random-weights mode, in the run's element type.  Routers are as decided as trained
    ones: a token's embedding leans towards two experts, and a router's rows are the directions of that leaning.  (Where the router is
    random as well, one token in seventy changes an expert with the rounding of its activations.)"""
    raw, dtype = MODELS[case["model"]], DTYPES[case["dtype"]]
    t = random_tensor_dict(_config(case), seed, dtype, device=DEVICE)
    routers = [name for name in t if name.endswith(".router")]
    if routers:
        gen = torch.Generator().manual_seed(seed)
        n, w = t[routers[0]].shape
        to = torch.linalg.qr(torch.randn(w, n, generator=gen, dtype=torch.float64))[0].T.float()
        first = torch.randint(0, n, (raw["vocab"],), generator=gen)
        second = (first + torch.randint(1, n, (raw["vocab"],), generator=gen)) % n
        leaning = (to[first] + 0.75 * to[second]) * (0.35 * math.sqrt(w))
        t["embed"] = (t["embed"].float() / 0.02 + leaning.to(DEVICE)).to(dtype)
        for name in routers:
            t[name] = to.to(DEVICE, dtype)
    return t


def _tokens(case, seed):
    vocab = MODELS[case["model"]].get("vocab") or MODELS[case["model"]]["vocab_size"]
    gen = torch.Generator().manual_seed(seed)
    return [torch.randint(0, vocab, (n + case["new"],), generator=gen).tolist() for n in _lengths(case)]


def prepare(case, seed):
    page, tokens = case["page"], _tokens(case, seed)
    room = sum(-(-len(t) // page) * page for t in tokens)
    lm = load_model(config=_config(case), tensors=_weights(case, seed), dtype=DTYPES[case["dtype"]], device=DEVICE, page_size=page,
                    max_tokens=room, max_requests=len(tokens))
    state = {"lm": lm, "tokens": tokens, "steps": _schedule(case)}
    for _ in range(WARM_PASSES):
        run(state)
    return state


def run(state):
    """One pass: requests admitted, prompts fed, tokens taken, requests released; the logits of every step that wants some."""
    lm, tokens = state["lm"], state["tokens"]
    slots = [lm.cache.admit() for _ in tokens]
    logits = []
    for step in state["steps"]:
        got = lm.step([StepEntry(slots[i], tokens[i][d:d + n], want) for i, d, n, want in step])
        if got is not None:
            logits.append(got)
    for slot in slots:
        lm.cache.release(slot)
    return logits


# ------------------------------------------------------------------------------------ what a pass cannot do without


def _sizes(raw):
    """(weights of a token's own layers, weights of one expert, experts, experts a token, layers with experts, vocabulary x width,
    key and value numbers a token keeps, operations a visible key costs a token, its window) of a model; a window of 0: every key."""
    if "hidden_size" in raw:
        d, L, H, kv, ff = (raw[k] for k in ("hidden_size", "num_hidden_layers", "num_attention_heads", "num_key_value_heads", "intermediate_size"))
        hd = d // H
        return L * (2 * d * H * hd + 2 * d * kv * hd + 3 * d * ff), 0, 1, 1, 0, d * raw["vocab_size"], L * 2 * kv * hd, [(L * 4 * H * hd, 0)]
    w, own, per, E, top, moe, kept, keys = raw["width"], 0, 0, 1, 1, 0, 0, []
    for layer in raw["layers"]:
        m, f, kind = layer["mixer"], layer["mlp"], layer["type"]
        for a in (m["left"], m["right"]) if kind == "parallel" else (m,):
            H, dim, dv = a["heads"], a.get("dim", 0), a["vdim"]
            window = a.get("mask", {}).get("size", 0)
            if kind == "mamba2":
                own += w * (2 * H * dv + 2 * a["groups"] * a["state"] + H) + w * H * dv
            elif kind == "latent_attention":
                own += w * (H * (dim + 64) + a["kv_rank"] + 64 + H * dv) + a["kv_rank"] * H * (dim + dv)
                kept += a["kv_rank"] + 64
                keys.append((4 * H * dim + 2 * H * 64, window))
            elif kind == "delta":
                own += w * (2 * a["kv_heads"] * dim + 3 * H * dv)
            elif "tau" in a:
                own += w * (2 * H * dim + 3 * H * dv)
            else:
                maps = 2 if "diff" in a else 1
                own += w * (maps * H * dim + (2 if "diff" in a else 1) * H * dv)
                if "kv_from" not in a:
                    own += w * a["kv_heads"] * (maps * dim + dv)
                    kept += a["kv_heads"] * (maps * dim + dv)
                keys.append((2 * maps * H * (dim + dv), window))
        if f["kind"] == "dense":
            own += (2 if raw["architecture"] == "Livovik" else 3) * w * f["ff"]
        else:
            per, E, top, moe = 3 * w * f["expert"]["ff"], f["router"]["experts"], f["router"]["top"], moe + 1
            own += 3 * w * f.get("shared", {"ff": 0})["ff"]
    return own, per, E, top, moe, w * raw["vocab"], kept, keys


def work(case):
    """Every step's weights once (of the experts those that its tokens can be expected to choose), the keys and values that it sees and
    writes, its logits; the operations of its tokens."""
    own, per, E, top, moe, head, kept, keys = _sizes(MODELS[case["model"]])
    vocab = MODELS[case["model"]].get("vocab") or MODELS[case["model"]]["vocab_size"]
    elem = 4 if case["dtype"] == "f32" else 2
    nbytes = flops = 0.0
    for step in _schedule(case):
        rows = sum(n for _, _, n, _ in step)
        want = sum(len(w) for _, _, _, w in step)
        touched = E * (1.0 - (1.0 - top / E) ** rows)
        nbytes += elem * (own + moe * per * touched + (head if want else 0)) + 4 * want * vocab + elem * kept * rows
        nbytes += elem * kept * sum(d for _, d, _, _ in step)
        flops += 2.0 * rows * (own + moe * per * top) + 2.0 * want * head
        for _, d, n, _ in step:
            for cost, window in keys:
                full = n * d + n * (n + 1) / 2
                flops += cost * (min(full, n * window / 2 if d == 0 and n > window else n * window) if window else full)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Logits of one precision under another order of the sums: roundings of the stored activations part from the first layer on."""
    return {"rel": {"bf16": 0.025, "f16": 0.01, "f32": 2e-5}[case["dtype"]], "max": {"bf16": 0.6, "f16": 0.2, "f32": 2e-3}[case["dtype"]]}


# ------------------------------------------------------------------------------------ the same in 64 bits, in plain torch


class _Plain:
    """Whole sequences in 64 bits.  The rows of all requests stand one below the other in ``x``; ``parts`` are their ranges."""

    def __init__(self, raw, tensors, lengths):
        self.raw, self.t = raw, tensors
        ends = [sum(lengths[:i + 1]) for i in range(len(lengths))]
        self.parts = [slice(e - n, e) for n, e in zip(lengths, ends)]
        self.pos = torch.cat([torch.arange(n, device=DEVICE) for n in lengths]).double()

    def w(self, name):
        return self.t[name].double()

    def lin(self, x, name):
        y = x @ self.w(name).T
        return y

    def norm(self, x, name, eps):
        x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
        return x if name is None else x * self.w(name)

    def rotate(self, x, freqs, neighbours):
        """``x [n, heads, d]``: the first ``2 len(freqs)`` numbers of a head in pairs."""
        f = torch.tensor(freqs, dtype=torch.float64, device=DEVICE)
        a = (self.pos[:, None] * f)[:, None, :]
        c, s, half, out = torch.cos(a), torch.sin(a), len(freqs), x.clone()
        i, j = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if neighbours else (slice(0, half), slice(half, 2 * half))
        u, v = x[..., i], x[..., j]
        out[..., i], out[..., j] = u * c - v * s, v * c + u * s
        return out

    def attend(self, q, k, v, scale, window=0, chunk=0, sink=None):
        """Softmax attention of every request's rows over its own; ``q [n, H, d]``, ``k [n, G, d]``, ``v [n, G, dv]``."""
        H, G = q.shape[1], k.shape[1]
        out = q.new_empty(q.shape[0], H, v.shape[-1])
        for part in self.parts:
            n = part.stop - part.start
            i, j = torch.arange(n, device=DEVICE)[:, None], torch.arange(n, device=DEVICE)[None, :]
            see = j <= i
            if window:
                see = see & (i - j < window)
            if chunk:
                see = see & (i // chunk == j // chunk)
            for h in range(H):
                g = h // (H // G)
                s = (q[part, h] @ k[part, g].T * scale).masked_fill(~see, -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[h].expand(n, 1)], 1)
                p = torch.softmax(s, -1)
                out[part, h] = p[:, :n] @ v[part, g]
        return out

    def conv(self, x, name):
        w = self.w(name)
        taps = w.shape[1]
        out = torch.zeros_like(x)
        for part in self.parts:
            y = x[part]
            past = torch.cat([y.new_zeros(taps - 1, y.shape[1]), y])
            for j in range(taps):
                out[part] += past[j:j + y.shape[0]] * w[:, j]
        return out

    def recur(self, step, n, state):
        """Every request's rows in turn through ``step(state, row) -> (state, out)``."""
        out = [None] * n
        for part in self.parts:
            s = torch.zeros(state, dtype=torch.float64, device=DEVICE)
            for i in range(part.start, part.stop):
                s, out[i] = step(s, i)
        return torch.stack(out)

    # ---- mixers of the further designs
    def chunked(self, h, p, m, eps):
        n, H, G, d, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q = self.norm(self.lin(h, p + "q").view(n, H, d), p + "q.norm", eps)
        k = self.norm(self.lin(h, p + "k").view(n, G, d), p + "k.norm", eps)
        f = _frequencies(m["rot"])
        o = self.attend(self.rotate(q, f, False), self.rotate(k, f, False), self.lin(h, p + "v").view(n, G, dv), m["scale"],
                        chunk=m["mask"]["size"], sink=self.w(p + "sink"))
        o = o * torch.sigmoid(self.lin(h, p + "g"))[..., None]
        return self.lin(o.reshape(n, H * dv), p + "o")

    def latent(self, h, p, m, eps, neighbours, gate):
        n, H, d, r, dv, rank = h.shape[0], m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        f = _frequencies(m["rot"])
        q, down = self.lin(h, p + "q").view(n, H, d + r), self.lin(h, p + "dkv")
        q = torch.cat([q[..., :d], self.rotate(q[..., d:], f, neighbours)], -1)
        c = self.norm(down[:, :rank], p + "dkv.norm", eps)
        k = torch.cat([self.lin(c, p + "uk").view(n, H, d), self.rotate(down[:, None, rank:], f, neighbours).expand(n, H, r)], -1)
        o = self.attend(q, k, self.lin(c, p + "uv").view(n, H, dv), m["scale"], window=m.get("mask", {}).get("size", 0))
        if gate:
            o = o * torch.sigmoid(self.lin(h, p + "g"))[..., None]
        return self.lin(o.reshape(n, H * dv), p + "o")

    def linear(self, h, p, m, eps):
        n, H, d, dv = h.shape[0], m["heads"], m["dim"], m["vdim"]
        q, k, v = self.lin(h, p + "q").view(n, H, d) * d ** -0.5, self.lin(h, p + "k").view(n, H, d), self.lin(h, p + "v").view(n, H, dv)
        a = torch.sigmoid(self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "a2.b")).pow(1.0 / m["tau"]).view(n, H, d)

        def step(S, i):
            S = a[i][:, :, None] * S + k[i][:, :, None] * v[i][:, None, :]
            return S, torch.einsum("hdv,hd->hv", S, q[i])
        o = self.norm(self.recur(step, n, (H, d, dv)), p + "norm", eps).reshape(n, H * dv)
        return self.lin(o * torch.nn.functional.silu(self.lin(h, p + "g")), p + "o")

    def delta(self, h, p, m, eps):
        n, H, G, d, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (torch.nn.functional.silu(self.conv(self.lin(h, p + s), p + s + ".conv")) for s in "qkv")
        unit = lambda x: x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q = (unit(q.view(n, G, d)) * d ** -0.5).repeat_interleave(H // G, 1)
        k, v = unit(k.view(n, G, d)).repeat_interleave(H // G, 1), v.view(n, H, dv)
        beta = torch.sigmoid(self.lin(h, p + "b"))
        g = torch.exp(-torch.exp(self.w(p + "A_log")) * torch.nn.functional.softplus(self.lin(h, p + "a") + self.w(p + "dt_bias")))

        def step(S, i):
            S = g[i][:, None, None] * S
            u = beta[i][:, None] * (v[i] - torch.einsum("hdv,hd->hv", S, k[i]))
            S = S + k[i][:, :, None] * u[:, None, :]
            return S, torch.einsum("hdv,hd->hv", S, q[i])
        o = self.norm(self.recur(step, n, (H, d, dv)), p + "norm", eps).reshape(n, H * dv)
        return self.lin(o * torch.nn.functional.silu(self.lin(h, p + "g")), p + "o")

    def mamba(self, h, p, m, eps):
        n, H, P, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * P
        z, xbc, dt = self.lin(h, p + "in").split([inner, inner + 2 * G * N, H], -1)
        xbc = torch.nn.functional.silu(self.conv(xbc, p + "conv") + self.w(p + "conv.b"))
        x = xbc[:, :inner].view(n, H, P)
        B, C = (y.reshape(n, G, N).repeat_interleave(H // G, 1) for y in xbc[:, inner:].split(G * N, -1))
        dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias"))
        keep = torch.exp(-torch.exp(self.w(p + "A_log")) * dt)

        def step(S, i):
            S = keep[i][:, None, None] * S + (dt[i][:, None] * B[i])[:, :, None] * x[i][:, None, :]
            return S, torch.einsum("hnp,hn->hp", S, C[i])
        y = self.recur(step, n, (H, N, P)) + self.w(p + "D")[:, None] * x
        y = y.reshape(n, inner) * torch.nn.functional.silu(z)
        y = self.norm(y.view(n, m["norm_groups"], -1), None, eps).reshape(n, inner) * self.w(p + "norm")
        return self.lin(y, p + "o")

    def diff(self, h, p, m, eps, caches, i):
        n, H, G, d, dv, f = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"], _frequencies(m["rot"])
        part = lambda s: self.conv(self.lin(h, p + s) + self.w(p + s + ".b"), p + s + ".conv")  # noqa: E731
        q = self.rotate(part("q").view(n, H * 2, d), f, True).view(n, H, 2, d)
        if "kv_from" in m:
            k, v = caches[m["kv_from"]]
        else:
            k, v = caches[i] = self.rotate(part("k").view(n, G * 2, d), f, True).view(n, G, 2, d), part("v").view(n, G, dv)
        lam = torch.exp((self.w(p + "lq1") * self.w(p + "lk1")).sum()) - torch.exp((self.w(p + "lq2") * self.w(p + "lk2")).sum()) + m["diff"]
        o = self.attend(q[:, :, 0], k[:, :, 0], v, m["scale"]) - lam * self.attend(q[:, :, 1], k[:, :, 1], v, m["scale"])
        o = (self.norm(o, None, eps) * (1.0 - m["diff"])).reshape(n, H * dv)
        return self.lin(o * torch.sigmoid(self.lin(h, p + "g")), p + "o") + self.w(p + "o.b")

    # ---- feed-forwards
    def gated(self, h, p):
        return self.lin(torch.nn.functional.silu(self.lin(h, p + "gate")) * self.lin(h, p + "up"), p + "down")

    def experts(self, h, p, mlp):
        r = mlp["router"]
        z, real = self.lin(h, p + "router"), r["experts"]
        if "identity" in r:  # softmax over all outputs, a correction of the choice, chosen scores over their sum, outputs weighed
            s = torch.softmax(z, -1)
            idx = torch.topk(s + self.w(p + "correction"), r["top"], -1).indices
            g = s.gather(1, idx)
            g = g / (g.sum(-1, keepdim=True) + 1e-20)
        else:  # sigmoid scores as they are, inputs weighed
            g, idx = torch.topk(torch.sigmoid(z), r["top"], -1)
        weight = torch.zeros_like(z).scatter(1, idx, g)
        out = torch.zeros_like(h)
        for e in range(real):
            rows = torch.nonzero((idx == e).any(-1))[:, 0]
            if rows.numel():
                we = weight[rows, e][:, None]
                out[rows] += self.gated(h[rows], f"{p}e{e}.") * we if "identity" in r else self.gated(h[rows] * we, f"{p}e{e}.")
        if "identity" in r:
            out += weight[:, real:].sum(-1, keepdim=True) * h
        if "shared" in mlp:
            out += self.gated(h, p + "shared.") * torch.sigmoid(self.lin(h, p + "shared.sg"))
        return out

    # ---- models
    def qwen(self, x):
        r, n = self.raw, x.shape[0]
        H, G, eps = r["num_attention_heads"], r["num_key_value_heads"], r["rms_norm_eps"]
        hd = r["hidden_size"] // H
        f = _frequencies({"base": r["rope_theta"], "dims": hd})
        for i in range(r["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.norm(x, p + "input_layernorm.weight", eps)
            q, k, v = (self.lin(h, f"{p}self_attn.{s}_proj.weight") + self.w(f"{p}self_attn.{s}_proj.bias") for s in "qkv")
            o = self.attend(self.rotate(q.view(n, H, hd), f, False), self.rotate(k.view(n, G, hd), f, False), v.view(n, G, hd), hd ** -0.5)
            x = x + self.lin(o.reshape(n, H * hd), p + "self_attn.o_proj.weight")
            h = self.norm(x, p + "post_attention_layernorm.weight", eps)
            a = torch.nn.functional.silu(self.lin(h, p + "mlp.gate_proj.weight")) * self.lin(h, p + "mlp.up_proj.weight")
            x = x + self.lin(a, p + "mlp.down_proj.weight")
        return self.norm(x, "model.norm.weight", eps)

    def livovik(self, x):
        r = self.raw
        eps, alpha = r["norm"]["eps"], r["postln_alpha"]
        for i, layer in enumerate(r["layers"]):
            p, f = f"l{i}.", layer["mlp"]
            x = self.norm(alpha * x + self.chunked(x, p + "mix.", layer["mixer"], eps), p + "norm1", eps)
            y = self.experts(x, p + "mlp.", f) if f["kind"] == "moe" else self.lin(torch.relu(self.lin(x, p + "mlp.up")) ** 2, p + "mlp.down")
            x = self.norm(alpha * x + y, p + "norm2", eps)
        return self.norm(x, "final.norm", eps)

    def befirax(self, x):
        r, caches = self.raw, {}
        eps = r["norm"]["eps"]
        xs = x[None].repeat(r["streams"], 1, 1)

        def branch(xs, p, norm, fn):
            y = fn(self.norm(torch.einsum("s,snw->nw", self.w(p + "in"), xs), norm, eps))
            return torch.einsum("st,snw->tnw", self.w(p + "mix"), xs) + self.w(p + "out")[:, None, None] * y
        for i, layer in enumerate(r["layers"]):
            p, m, kind = f"l{i}.", layer["mixer"], layer["type"]
            mixers = {"mamba2": lambda h: self.mamba(h, p + "mix.", m, eps), "attention": lambda h: self.diff(h, p + "mix.", m, eps, caches, i),
                      "latent_attention": lambda h: self.latent(h, p + "mix.", m, eps, False, True)}
            xs = branch(xs, p + "hc1.", p + "norm1", mixers[kind])
            xs = branch(xs, p + "hc2.", p + "norm2", lambda h: self.experts(h, p + "mlp.", layer["mlp"]))
        return self.norm(xs.sum(0), "final.norm", eps)

    def salolorn(self, x):
        r = self.raw
        eps = r["norm"]["eps"]
        for i, layer in enumerate(r["layers"]):
            p, m = f"l{i}.", layer["mixer"]
            h = self.norm(x, p + "norm1", eps)
            if layer["type"] == "delta":
                y = self.delta(h, p + "mix.", m, eps)
            elif layer["type"] == "latent_attention":
                y = self.latent(h, p + "mix.", m, eps, True, False)
            else:
                y = (m["left_scale"] * self.chunked(h, p + "mix.left.", m["left"], eps)
                     + m["right_scale"] * self.linear(h, p + "mix.right.", m["right"], eps))
            x = x + self.norm(y, p + "norm1b", eps)
            x = x + self.norm(self.gated(self.norm(x, p + "norm2", eps), p + "mlp."), p + "norm2b", eps)
        return self.norm(x, "final.norm", eps)


def _frequencies(rot):
    """``base^(-2i / dims)``, under ``scaling`` by wavelength: short periods stay, long ones are divided, mixed in between."""
    out = []
    for i in range(rot["dims"] // 2):
        f = float(rot["base"]) ** (-2.0 * i / rot["dims"])
        sc = rot.get("scaling")
        if sc:
            period, long, short = 2.0 * math.pi / f, sc["original"] / sc["low"], sc["original"] / sc["high"]
            if period > long:
                f /= sc["factor"]
            elif period >= short:
                s = (sc["original"] / period - sc["low"]) / (sc["high"] - sc["low"])
                f = (1.0 - s) * f / sc["factor"] + s * f
        out.append(f)
    return out


def exact(case, seed):
    raw, t, tokens = MODELS[case["model"]], _weights(case, seed), _tokens(case, seed)
    qwen = "hidden_size" in raw
    plain = _Plain(raw, t, [len(s) for s in tokens])
    table = t["model.embed_tokens.weight" if qwen else "embed"]
    x = table[torch.tensor([v for s in tokens for v in s], device=DEVICE)].double()
    x = plain.qwen(x) if qwen else getattr(plain, raw["architecture"].lower())(x)
    head = t.get("lm_head.weight", t.get("head", table)).double()
    scale = raw.get("logit_scale", 1.0)
    out = []
    for step in _schedule(case):
        rows = [plain.parts[i].start + d + w for i, d, _, want in step for w in want]
        if rows:
            out.append(x[torch.tensor(rows, device=DEVICE)] @ head.T * scale)
    return out
