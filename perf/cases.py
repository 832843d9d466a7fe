"""The workloads this framework is timed on: requests of given token ids taken through the persistent kernel.

Two ways of use.  "offline": the on-GPU scheduler takes R requests of P given tokens through P / portion iterations of one
launch (Qwen3Decoder of demo_qwen3.py, Generator of generate.py).  With one token per request and iteration that is the decode
loop itself, with ids that do not hang on which of two nearly equal logits is larger; with one request of 64 rows per iteration
it is the ingestion of a long prompt.  "serving": the host loop (mirage.mpk.ServingSession) ingests R prompts of unequal lengths,
decodes N further tokens of each step by step, reads the logits of every step and ends the requests.

Shapes are the named ones of demo_qwen3.py and generate.py with fewer layers (a layer costs the same at any depth) and the
vocabulary of `bench.py --compare`, which keeps the output matrix's share of a step what it is at full depth; "small" is the
size of the test models.  Matrices are N(0, 1/fan-in) and embeddings N(0, 1), so that activations are of order one as in a
trained model; vectors lie around their neutral values; routers are wide enough that most choices have a margin.
"""
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "fleet-chiplet-megakernel_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

VOCAB = 32768
DEVICE = "cuda"
QWEN = {"qwen3-8b": dict(width=4096, heads=32, kv_heads=8, ff=12288, experts=0, top=0), "qwen3-30b-a3b": dict(width=2048, heads=32, kv_heads=4, ff=768, experts=128, top=8)}
CYCLE = {"suborax": 1, "dodonex": 2, "bukatar": 4, "vizonex": 4}


def _case(name, model, engine, layers, requests, prompt, steps=0, portion=1, dtype="bf16"):
    return {"name": name, "model": model, "engine": engine, "layers": layers, "requests": requests, "prompt": prompt, "steps": steps, "portion": portion, "dtype": dtype}


def listed():
    return [
        # the smallest calls: a short exchange with a small model, where launches and the host loop are what a step costs
        _case("small_chat", "suborax-small", "serving", 2, 1, 7, 12),
        # the headline: single-stream decode of the dense shape
        _case("qwen_decode_1", "qwen3-8b", "offline", 8, 1, 64),
        # the headline's other batch size: 64 streams at contexts up to a few hundred
        _case("qwen_decode_64", "qwen3-8b", "offline", 6, 64, 320),
        # a long prompt, 64 rows an iteration; nothing divides its length
        _case("qwen_prompt", "qwen3-8b", "offline", 8, 1, 2501, portion=64),
        # mixture of experts, one stream and a batch in which most experts are visited
        _case("qwen_moe_decode_1", "qwen3-30b-a3b", "offline", 8, 1, 64),
        _case("qwen_moe_decode_16", "qwen3-30b-a3b", "offline", 6, 16, 48),
        # a few users with long prompts and answers of some lines
        _case("suborax_serving_4", "suborax-8b", "serving", 8, 4, 1501, 24),
        # the 32-bit build, requests of unequal lengths
        _case("suborax_f32_serving_3", "suborax-2k", "serving", 4, 3, 301, 16, dtype="f32"),
        # latent attention and delta rule, eight users
        _case("dodonex_serving_8", "dodonex-8b", "serving", 6, 8, 203, 32),
        # windowed and latent attention, scans and experts: single-stream decode, and a batch of short chats
        _case("bukatar_decode_1", "bukatar-8b", "offline", 4, 1, 96),
        _case("bukatar_serving_16", "bukatar-2k", "serving", 4, 16, 100, 24),
        # chunked attention, recurrences per head and grouped experts: 64 streams, the largest iterations there are
        _case("vizonex_decode_64", "vizonex-8b", "offline", 4, 64, 48),
    ]


def draw(rng):
    logu = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    largest = max(_cost(c) for c in listed())
    while True:
        model = rng.choice(["qwen3-8b", "qwen3-30b-a3b", "suborax-small"] + [f"{m}-{s}" for m in CYCLE for s in ("8b", "2k")])
        family = model.split("-")[0]
        c = {"model": model, "engine": "offline" if model in QWEN else rng.choice(["offline", "serving"]), "layers": rng.randint(2, 8)}
        if CYCLE.get(family) == 4:
            c["layers"] = rng.choice([4, 5, 6])
        c["requests"] = logu(1, 64) if rng.random() < 0.7 else 1
        c["dtype"] = "f32" if family in CYCLE and rng.random() < 0.15 else "bf16"
        c["portion"], c["steps"] = 1, 0
        if c["engine"] == "serving":
            c["prompt"], c["steps"] = logu(1, 2000), logu(1, 40)
        elif c["requests"] == 1 and rng.random() < 0.5:
            c["prompt"], c["portion"] = logu(65, 3000), 64
        else:
            c["prompt"] = logu(1, 320)
        if _cost(c) <= largest:
            return c


# ------------------------------------------------------------------------------------------------ models and inputs
def _config(case):
    """Parsed config.json of a layer-list shape."""
    import generate
    family, size = case["model"].split("-")
    if size == "small":
        return generate.suborax_shape(width=256, heads=8, kv_heads=2, dim=64, vdim=64, ff=768, layers=case["layers"], vocab=1000)
    make, sizes = generate.SHAPES[case["model"]]
    extra = {"positions": 4096} if family == "vizonex" else {}
    return make(**sizes, layers=case["layers"], vocab=VOCAB, **extra)


def _shapes(case):
    """Tensor name -> shape."""
    if case["model"] not in QWEN:
        from mirage.mpk.models import bukatar, dodonex, suborax, vizonex
        c = _config(case)
        kind = {"Suborax": suborax.SuboraxConfig, "Dodonex": dodonex.DodonexConfig, "Bukatar": bukatar.BukatarConfig, "Vizonex": vizonex.VizonexConfig}[c["architecture"]]
        return kind.from_dict(c).tensor_shapes()
    s = QWEN[case["model"]]
    W, D, E, F = s["width"], 128, s["experts"], s["ff"]
    out = {"embed": (VOCAB, W)}
    for i in range(case["layers"]):
        p = f"l{i}."
        out.update({p + "input_norm": (W,), p + "q_proj": (s["heads"] * D, W), p + "k_proj": (s["kv_heads"] * D, W), p + "v_proj": (s["kv_heads"] * D, W), p + "q_norm": (D,), p + "k_norm": (D,),
                    p + "o_proj": (W, s["heads"] * D), p + "post_norm": (W,)})
        if E:
            out.update({p + "router": (E, W), p + "gate_up_proj": (E, 2 * F, W), p + "down_proj": (E, W, F)})
        else:
            out.update({p + "gate_proj": (F, W), p + "up_proj": (F, W), p + "down_proj": (W, F)})
    out.update({"final_norm": (W,), "lm_head": (VOCAB, W)})
    return out


def _weights(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    offset = case["model"].startswith("suborax")  # norm weights are stored as their distance from one
    out, shapes = {}, _shapes(case)
    for name, shape in shapes.items():
        t = torch.empty(shape, dtype=dtype if len(shape) > 1 else torch.float32, device=DEVICE).normal_(0.0, 1.0, generator=g)
        if name.endswith(".A_log"):
            t *= 0.5
        elif name.endswith((".dt_bias", ".dt.b", ".w0")):
            t = 0.3 * t - 3.0
        elif name.endswith((".b", ".sink")):
            t *= 0.3
        elif name.endswith(".correction"):
            t *= 0.1
        elif name.endswith("router"):
            t *= (2.0 if case["model"].startswith("vizonex") else 4.0) / shape[-1] ** 0.5
        elif name == "pos":
            t *= 0.5
        elif name.endswith((".ls1", ".ls2")):  # (eight experts' outputs are summed, each with a share of up to 2.5)
            t = (0.02 if name.endswith("2") and f"{name[:-4]}.mlp.router" in shapes else 0.3) * (1.0 + 0.1 * t)
        elif len(shape) == 3 and name.endswith("down_proj"):  # (a choice that rounding turns changes its token for good)
            t *= 0.4 * shape[-1] ** -0.5
        elif len(shape) > 1:
            t *= 1.0 if name in ("embed", "side.embed") else shape[-1] ** -0.5
        else:
            t = 0.1 * t + (0.0 if offset else 1.0)
        out[name] = t.to(dtype)
    return out


def _lengths(case):
    """Prompt lengths: the longest is case["prompt"], in the serving loop the others are down to half of it."""
    P, R = case["prompt"], case["requests"]
    return [max(1, P - (r * P) // (2 * R)) if case["engine"] == "serving" else P for r in range(R)]


def _tokens(case, seed):
    """Every request's ids: prompt and, behind it, the tokens of its steps."""
    g = torch.Generator().manual_seed(seed + 1000003)
    vocab = _shapes(case)["embed"][0]
    return [torch.randint(0, vocab, (n + case["steps"],), generator=g) for n in _lengths(case)]


def _rope(n):
    f = 1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float32, device=DEVICE) / 128))
    a = torch.arange(n, dtype=torch.float32, device=DEVICE)[:, None] * f[None, :]
    a = torch.cat([a, a], dim=-1)
    return a.cos().to(torch.bfloat16).contiguous(), a.sin().to(torch.bfloat16).contiguous()


def _page(case):
    return 64 if case["portion"] > 1 else -(-(case["prompt"] + 8) // 64) * 64


def prepare(case, seed):
    w, tokens, R, P = _weights(case, seed), _tokens(case, seed), case["requests"], case["prompt"]
    rows = case["portion"] if R == 1 else R
    max_seq = P + 8
    if case["model"] in QWEN:
        import demo_qwen3 as demo
        s = QWEN[case["model"]]
        shape = demo.Qwen3Shape(hidden_size=s["width"], num_q_heads=s["heads"], num_kv_heads=s["kv_heads"], head_dim=128, intermediate_size=0 if s["experts"] else s["ff"],
                                num_layers=case["layers"], vocab_size=VOCAB, num_experts=s["experts"], num_experts_per_tok=s["top"], moe_intermediate_size=s["ff"] if s["experts"] else 0)
        layers = [{n.split(".", 1)[1]: t for n, t in w.items() if n.startswith(f"l{i}.")} for i in range(case["layers"])]
        weights = {"embed": w["embed"], "layers": layers, "final_norm": w["final_norm"], "lm_head": w["lm_head"]}
        runner = demo.Qwen3Decoder(shape, weights, max_num_batched_tokens=rows, max_num_batched_requests=R, max_seq_length=max_seq, page_size=_page(case), cos_sin=_rope(max_seq),
                                   max_tokens_per_request=case["portion"])
    else:
        import generate
        from mirage.mpk import MirageModelConfig, ServingSession
        model = MirageModelConfig(architecture=_config(case), state_dict=w)
        dtype = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
        if case["engine"] == "serving":
            longest = P + case["steps"]
            pages = -(-longest // 64)
            runner = ServingSession.open(model_config=model, dtype=dtype, max_tokens=R * pages * 64, max_requests=R, page_size=64, max_seq_length=pages * 64)
        else:
            runner = generate.Generator(max_seq, model_config=model, batch=R, max_num_batched_tokens=rows, max_tokens_per_request=case["portion"], page_size=_page(case), eos_token_id=-1,
                                        dtype=dtype)
    if case["engine"] == "serving":
        tokens = [t.tolist() for t in tokens]
    return {"case": case, "runner": runner, "tokens": tokens}


def run(state):
    case, runner, tokens = state["case"], state["runner"], state["tokens"]
    if case["engine"] == "serving":
        cut = _lengths(case)
        logits, _ = runner.step([(r, t[:n]) for r, (t, n) in enumerate(zip(tokens, cut))], [[n - 1] for n in cut])
        out = [logits]
        for i in range(case["steps"]):
            logits, _ = runner.step([(r, [t[n + i]]) for r, (t, n) in enumerate(zip(tokens, cut))], [[0]] * len(tokens))
            out.append(logits)
        for r in range(len(tokens)):
            runner.end(r)
        return out
    runner.load_prompts(tokens)
    iterations = -(-case["prompt"] // case["portion"])
    runner.mpk.run_steps(iterations)
    last = case["requests"] if case["portion"] == 1 else case["prompt"] - (iterations - 1) * case["portion"]
    out = {"logits": runner.logits()[:last].clone()}  # (a copy: the rows themselves belong to the library and go with the runner)
    if case["model"] in QWEN:  # (the caches are the caller's tensors: what every layer appended at every step)
        out.update(k=runner.k_cache, v=runner.v_cache)
    return out


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _parts(case):
    """Elements of one iteration's matrices (experts apart), of one expert layer's experts, and of the head; layers with experts
    and their (experts, top)."""
    dense, routed = 0, []
    shapes = _shapes(case)
    per_layer = {}
    for name, s in shapes.items():
        if len(s) < 2 or name in ("embed", "side.embed", "pos", "lm_head", "head") or name.endswith((".conv", ".canon1", ".A_log")):
            continue
        n = math.prod(s)
        layer = name.split(".")[0]
        if ".mlp.e" in name or name.endswith(("gate_up_proj",)) or (len(s) == 3 and name.endswith("down_proj")):
            per_layer[layer] = per_layer.get(layer, 0) + n
        else:
            dense += n
    head = math.prod(shapes["embed"])
    for layer, n in per_layer.items():
        if case["model"] in QWEN:
            E, k = QWEN[case["model"]]["experts"], QWEN[case["model"]]["top"]
        else:
            r = _config(case)["layers"][int(layer[1:])]["mlp"]["router"]
            E, k = r["experts"], r["top"]
        routed.append((n, E, k))
    return dense, routed, head


def _mixers(case):
    """(cached elements per position, visible positions at most, attention multiply-adds per token and position, state elements) summed
    or listed per layer."""
    if case["model"] in QWEN:
        s = QWEN[case["model"]]
        return [(2 * s["kv_heads"] * 128, None, 2 * s["heads"] * 128, 0)] * case["layers"]
    out = []
    for layer in _config(case)["layers"]:
        m, kind = layer["mixer"], layer["type"]
        if kind == "attention":
            mask = m.get("mask") or {}
            most = mask["size"] + mask.get("keep_first", 0) if mask.get("size") else None
            out.append((m["kv_heads"] * (m["dim"] + m["vdim"]), most, m["heads"] * (m["dim"] + m["vdim"]), 0))
        elif kind == "latent_attention":
            out.append((m["kv_rank"] + m["rot_dim"], None, m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), 0))
        elif kind == "general_delta":
            out.append((0, None, 0, m["heads"] * m["dim"] ** 2))
        elif kind == "mamba1":
            out.append((0, None, 0, m["inner"] * m["state"]))
        else:
            out.append((0, None, 0, m["heads"] * m["vdim"] * m["state"]))
    return out


def work(case):
    """A prompt's tokens together read every matrix once; a decoded token per request reads them again, and the cache and state of every
    request.  Experts count as far as the tokens that run together choose different ones."""
    elem = 4 if case["dtype"] == "f32" else 2
    dense, routed, head = _parts(case)
    mixers, R = _mixers(case), case["requests"]
    lengths = _lengths(case)
    if case["engine"] == "offline" and case["portion"] == 1:
        lengths, steps = [0] * R, case["prompt"]
    else:
        steps = case["steps"]

    def iteration(tokens):
        b = dense + head + sum(n * (1 - (1 - k / E) ** tokens) for n, E, k in routed)
        f = 2 * tokens * (dense + sum(n * k / E for n, E, k in routed))
        return elem * b, f

    total_b = total_f = 0
    seen = lambda at, most: at if most is None else min(at, most)
    if sum(lengths):
        total_b, total_f = iteration(sum(lengths))
        total_f += 2 * R * head
        for cached, most, macs, state in mixers:
            for n in lengths:
                total_b += 2 * elem * cached * n + 4 * state
                total_f += 2 * macs * sum(seen(i + 1, most) for i in range(n)) + 4 * state * n
    for i in range(steps):
        b, f = iteration(R)
        total_b, total_f = total_b + b, total_f + f + 2 * R * head
        for cached, most, macs, state in mixers:
            at = sum(seen(n + i + 1, most) for n in lengths)
            total_b += elem * cached * (at + R) + 8 * state * R
            total_f += 2 * macs * at + 4 * state * R
    return {"bytes": float(total_b), "flops": float(total_f)}


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def tolerance(case):
    # bf16 activations at every stage of 2 to 8 layers; the 32-bit build sums in another order only
    if case["dtype"] == "f32":
        return {"rel": 2e-5, "max": 1e-3}
    return {"rel": 0.03, "max": 0.9}


# ------------------------------------------------------------------------------------------------ the same in 64 bits, in plain torch
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _turn_halves(x, pos, freq):
    """Dimension i of the first half turns with dimension i of the second one.  x [T, heads, dims]"""
    a = pos.double()[:, None, None] * freq
    c, s = a.cos(), a.sin()
    u, v = x.chunk(2, dim=-1)
    return torch.cat([u * c - v * s, v * c + u * s], dim=-1)


def _turn_pairs(x, pos, dims, base):
    a = pos.double()[:, None, None] * _freq(base, dims)
    c, s, out = a.cos(), a.sin(), x.clone()
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    out[..., 0:dims:2], out[..., 1:dims:2] = u * c - v * s, v * c + u * s
    return out


def _freq(base, dims, scaling=None):
    out = []
    for i in range(dims // 2):
        f = float(base) ** (-2.0 * i / dims)
        if scaling:
            wave = 2 * math.pi / f
            if wave > scaling["original"] / scaling["low"]:
                f /= scaling["factor"]
            elif wave >= scaling["original"] / scaling["high"]:
                t = (scaling["original"] / wave - scaling["low"]) / (scaling["high"] - scaling["low"])
                f = (1 - t) * f / scaling["factor"] + t * f
        out.append(f)
    return torch.tensor(out, dtype=torch.float64, device=DEVICE)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _clamped(a, b, limit):
    g, u = a.clamp(max=limit), b.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


def _attend(q, k, v, scale, sees, sink=None, cap=None):
    """q [T, H, D], k [T, G, D], v [T, G, E]; `sink` [H]: a further term of the softmax's denominator."""
    T, H = q.shape[:2]
    per = H // k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    for h in range(H):
        s = (q[:, h] @ k[:, h // per].T) * (scale if not torch.is_tensor(scale) else scale[h])
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~sees, float("-inf"))
        m = s.amax(dim=-1, keepdim=True)
        if sink is not None:
            m = torch.maximum(m, sink[h])
        e = torch.exp(s - m)
        total = e.sum(dim=-1, keepdim=True)
        out[:, h] = (e / (total if sink is None else total + torch.exp(sink[h] - m))) @ v[:, h // per]
    return out


class _Truth:
    """A forward pass over whole sequences, laid end to end."""

    def __init__(self, case, seed):
        self.case, self.w = case, _weights(case, seed)
        ids = _tokens(case, seed)
        self.lengths = [len(t) for t in ids]
        self.ids = torch.cat(ids).to(DEVICE)
        self.pos = torch.cat([torch.arange(n, device=DEVICE) for n in self.lengths])
        self.cache = []

    def __getitem__(self, name):
        return self.w[name].double()

    def lin(self, x, name):
        return x @ self[name].T

    def per_sequence(self, f, *rows):
        return torch.cat([f(*parts) for parts in zip(*(r.split(self.lengths) for r in rows))])

    def padded(self, x):
        return torch.nn.utils.rnn.pad_sequence(list(x.split(self.lengths)), batch_first=True)

    def joined(self, y):
        return torch.cat([y[r, :n] for r, n in enumerate(self.lengths)])

    def causal(self, n, size=None, keep=0, chunk=None):
        i = torch.arange(n, device=DEVICE)[:, None]
        j = i.T
        sees = j <= i
        if size:
            sees = sees & ((i - j < size) | (j < keep))
        if chunk:
            sees = sees & (i // chunk == j // chunk)
        return sees

    def conv(self, x, w, b=None):
        """Causal, per channel; the last column of w is the current token's."""
        taps = w.shape[1]

        def one(rows):
            rows = torch.cat([torch.zeros(taps - 1, rows.shape[1], dtype=rows.dtype, device=DEVICE), rows])
            return sum(rows[j:j + len(rows) - taps + 1] * w[:, j] for j in range(taps))
        y = self.per_sequence(one, x)
        return y if b is None else y + b

    def experts(self, h, p, choice, share, act, packed=False):
        """choice, share [T, top]."""
        y = torch.zeros_like(h)
        for e in choice.unique().tolist():
            t, k = (choice == e).nonzero(as_tuple=True)
            x = h[t]
            if packed:
                g, u = (x @ self.w[p + "gate_up_proj"][e].double().T).chunk(2, dim=-1)
                o = act(g, u) @ self.w[p + "down_proj"][e].double().T
            else:
                o = self.lin(act(self.lin(x, f"{p}.e{e}.gate"), self.lin(x, f"{p}.e{e}.up")), f"{p}.e{e}.down")
            y.index_add_(0, t, o * share[t, k][:, None])
        return y

    # -------------------------------------------------------------------------------------------- models
    def qwen(self):
        s, n = QWEN[self.case["model"]], self.case["layers"]
        H, G, D, T = s["heads"], s["kv_heads"], 128, len(self.ids)
        cos, sin = (t.double()[self.pos][:, None, :] for t in _rope(max(self.lengths) + 8))
        norm = lambda x, name: _rms(x, 1e-6) * self[name]
        turn = lambda x: x * cos + torch.cat([-x[..., D // 2:], x[..., :D // 2]], dim=-1) * sin
        x = self["embed"][self.ids]
        for i in range(n):
            p = f"l{i}."
            h = norm(x, p + "input_norm")
            q, k, v = (self.lin(h, p + c + "_proj").view(T, -1, D) for c in "qkv")
            q, k = turn(norm(q, p + "q_norm")), turn(norm(k, p + "k_norm"))
            self.cache.append((k, v))
            o = self.per_sequence(lambda q, k, v: _attend(q, k, v, D ** -0.5, self.causal(len(q))), q, k, v)
            x = x + self.lin(o.reshape(T, H * D), p + "o_proj")
            h = norm(x, p + "post_norm")
            silu = lambda g, u: g * torch.sigmoid(g) * u
            if s["experts"]:
                share, choice = torch.softmax(self.lin(h, p + "router"), dim=-1).topk(s["top"], dim=-1)
                x = x + self.experts(h, p, choice, share / share.sum(dim=-1, keepdim=True), silu, packed=True)
            else:
                x = x + self.lin(silu(self.lin(h, p + "gate_proj"), self.lin(h, p + "up_proj")), p + "down_proj")
        return norm(x, "final_norm"), "lm_head"

    def suborax(self):
        c, T = _config(self.case), len(self.ids)
        eps, alpha = c["norm"]["eps"], c["postln_alpha"]
        norm = lambda x, name: _rms(x, eps) * (1.0 + self[name])
        x = self["embed"][self.ids] * c["embedding"]["scale"]
        for i, layer in enumerate(c["layers"]):
            m, p = layer["mixer"], f"l{i}."
            d = m["rot"]["dims"]
            freq = _freq(m["rot"]["base"], d, m["rot"].get("scaling"))
            unit = lambda t: _rms(torch.cat([_turn_halves(t[..., :d], self.pos, freq), t[..., d:]], dim=-1), eps)
            q, k, v = unit(self.lin(x, p + "mix.q").view(T, -1, m["dim"])), unit(self.lin(x, p + "mix.k").view(T, -1, m["dim"])), self.lin(x, p + "mix.v").view(T, -1, m["vdim"])
            o = self.per_sequence(lambda q, k, v: _attend(q, k, v, m["scale"], self.causal(len(q)), self[p + "mix.sink"], m["softcap"]), q, k, v)
            x = norm(alpha * x + self.lin(o.reshape(T, -1), p + "mix.o"), p + "norm1")
            g = self.lin(x, p + "mlp.gate")
            x = norm(alpha * x + self.lin(g * torch.sigmoid(g) * self.lin(x, p + "mlp.up"), p + "mlp.down"), p + "norm2")
        return norm(x, "final.norm"), "head"

    def latent(self, h, p, m, q, turn, eps):
        H, D, P, E, R, T = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], len(h)
        q = q.view(T, H, D + P)
        ckr = self.lin(h, p + "dkv")
        c, kr = _rms(ckr[:, :R], eps) * self[p + "dkv.norm"], turn(ckr[:, None, R:])
        k = torch.cat([(c @ self[p + "uk"].T).view(T, H, D), kr.expand(T, H, P)], dim=-1)
        q = torch.cat([q[..., :D], turn(q[..., D:])], dim=-1)
        v = (c @ self[p + "uv"].T).view(T, H, E)
        return self.per_sequence(lambda q, k, v: _attend(q, k, v, m["scale"], self.causal(len(q))), q, k, v).reshape(T, H * E)

    def dodonex(self):
        c, T = _config(self.case), len(self.ids)
        eps, groups, mult, side = c["norm"]["eps"], c["norm"]["groups"], c["residual_mult"], c["token_side"]["dim"]
        norm = lambda x, name: _rms(x.view(T, groups, -1), eps).reshape(x.shape) * self[name]
        x = self["embed"][self.ids] * c["embedding"]["scale"]
        for i, layer in enumerate(c["layers"]):
            m, p, q = layer["mixer"], f"l{i}.", f"l{i}.mix."
            h = norm(x, p + "norm1")
            if layer["type"] == "latent_attention":
                freq = _freq(m["rot"]["base"], m["rot_dim"])
                cq = _rms(self.lin(h, q + "dq"), eps) * self[q + "dq.norm"]
                o = self.latent(h, q, m, self.lin(cq, q + "uq"), lambda t: _turn_halves(t, self.pos, freq), eps)
            else:
                H, D = m["heads"], m["dim"]
                heads = lambda t: self.padded(t.view(T, H, D))
                r, k, v = (heads(self.lin(h, q + n)) for n in "rkv")
                dec = heads(torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(self.lin(h, q + "w1")) @ self[q + "w2"].T + self[q + "w0"])))
                a = heads(torch.sigmoid(self.lin(h, q + "a") + self[q + "a.b"]))
                u = k / torch.sqrt((k * k).sum(dim=-1, keepdim=True) + 1e-6)
                S = torch.zeros(len(self.lengths), H, D, D, dtype=torch.float64, device=DEVICE)
                o = torch.empty_like(v)
                for t in range(v.shape[1]):
                    seen = (u[:, t, :, :, None] * S).sum(dim=2)
                    S = dec[:, t, :, :, None] * S - (a[:, t] * u[:, t])[..., None] * seen[:, :, None, :] + k[:, t, :, :, None] * v[:, t, :, None, :]
                    o[:, t] = (S * r[:, t, :, :, None]).sum(dim=2)
                o = _rms(self.joined(o), eps).reshape(T, H * D) * self[q + "norm"] * torch.sigmoid(self.lin(h, q + "g"))
            y = self.lin(o, q + "o") + self.lin(_clamped(self.lin(h, p + "mlp.gate"), self.lin(h, p + "mlp.up"), layer["mlp"]["limit"]), p + "mlp.down")
            x = x + mult * y
            extra = self["side.embed"][self.ids][:, i * side:(i + 1) * side]
            x = x + mult * _rms(self.lin(_gelu(self.lin(x, p + "side.gate")) * extra, p + "side.proj"), eps) * self[p + "side.norm"]
        return norm(x, "final.norm") * c["logit_scale"], "embed"

    def bukatar(self):
        c, T = _config(self.case), len(self.ids)
        eps = c["norm"]["eps"]
        silu = lambda g: g * torch.sigmoid(g)
        norm = lambda x, name: _rms(x, eps) * self[name]
        x = self["embed"][self.ids]
        for i, layer in enumerate(c["layers"]):
            m, p, q, mlp = layer["mixer"], f"l{i}.", f"l{i}.mix.", layer["mlp"]
            h = norm(x, p + "norm1")
            if layer["type"] == "attention":
                mask, rot = m["mask"], m["rot"]
                turn = lambda t: _turn_pairs(t, self.pos, rot["dims"], rot["base"])
                k = (self.lin(h, q + "k") + self[q + "k.b"]).view(T, -1, m["dim"])
                qq = turn((self.lin(h, q + "q") + self[q + "q.b"]).view(T, -1, m["dim"]))
                one = torch.zeros(m["heads"], dtype=torch.float64, device=DEVICE)  # (exp(0) in the denominator)
                y = self.per_sequence(lambda a, b, d: _attend(a, b, d, m["scale"], self.causal(len(a), mask["size"], mask["keep_first"]), one), qq, turn(k), k)
                y = self.lin(y.reshape(T, -1), q + "o") + self[q + "o.b"]
            elif layer["type"] == "latent_attention":
                turn = lambda t: _turn_pairs(t, self.pos, m["rot_dim"], m["rot"]["base"])
                y = self.lin(self.latent(h, q, m, self.lin(h, q + "q"), turn, eps), q + "o")
            else:
                I, N, K = m["inner"], m["state"], m["dt_rank"]
                xz = self.lin(h, q + "in")
                u = silu(self.conv(xz[:, :I], self[q + "conv"], self[q + "conv.b"]))
                dbc = self.lin(u, q + "x")
                dt = torch.nn.functional.softplus(dbc[:, :K] @ self[q + "dt"].T + self[q + "dt.b"])
                A = -torch.exp(self[q + "A_log"])
                us, dts, B, C = (self.padded(t) for t in (u, dt, dbc[:, K:K + N], dbc[:, K + N:]))
                S, out = torch.zeros(len(self.lengths), I, N, dtype=torch.float64, device=DEVICE), torch.empty_like(us)
                for t in range(us.shape[1]):
                    S = torch.exp(dts[:, t, :, None] * A) * S + (dts[:, t] * us[:, t])[..., None] * B[:, t, None, :]
                    out[:, t] = (S * C[:, t, None, :]).sum(dim=-1)
                y = self.lin((self.joined(out) + self[q + "D"] * u) * silu(xz[:, I:]), q + "o")
            x = x + norm(y, p + "norm1b")
            h = norm(x, p + "norm2")
            if mlp["kind"] == "dense":
                y = self.lin(torch.relu(self.lin(h, p + "mlp.up")) ** 2, p + "mlp.down")
            else:
                gate = lambda a, b: silu(a) * b
                share, choice = torch.softmax(self.lin(h, p + "mlp.router"), dim=-1).topk(mlp["router"]["top"], dim=-1)
                y = self.experts(h, p + "mlp", choice, share / (share.sum(dim=-1, keepdim=True) + 1e-20), gate)
                y = y + torch.sigmoid(self.lin(h, p + "mlp.shared.sg")) * self.lin(gate(self.lin(h, p + "mlp.shared.gate"), self.lin(h, p + "mlp.shared.up")), p + "mlp.shared.down")
            x = x + norm(y, p + "norm2b")
        return norm(x, "final.norm"), "embed"

    def vizonex(self):
        c, T = _config(self.case), len(self.ids)
        eps = c["norm"]["eps"]
        silu = lambda g: g * torch.sigmoid(g)
        norm = lambda x, name: _rms(x, eps) * self[name]
        x = self["embed"][self.ids] + self["pos"][self.pos]
        for i, layer in enumerate(c["layers"]):
            m, p, q, mlp = layer["mixer"], f"l{i}.", f"l{i}.mix.", layer["mlp"]
            h = norm(x, p + "norm1")
            g = h + self.conv(h, self[p + "canon1"])
            if layer["type"] == "attention":
                qq, k = norm(self.lin(g, q + "q"), q + "q.norm").view(T, -1, m["dim"]), norm(self.lin(g, q + "k"), q + "k.norm").view(T, -1, m["dim"])
                v = self.lin(g, q + "v").view(T, -1, m["vdim"])
                y = self.per_sequence(lambda a, b, d: _attend(a, b, d, m["scale"] * self[q + "temp"], self.causal(len(a), chunk=m["mask"]["size"]), self[q + "sink"]), qq, k, v).reshape(T, -1)
            else:
                H, V, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
                I = H * V
                z, xbc, dt = self.lin(g, q + "in").split([I, I + 2 * G * N, H], dim=1)
                u, B, C = silu(self.conv(xbc, self[q + "conv"], self[q + "conv.b"])).split([I, G * N, G * N], dim=1)
                dt = torch.nn.functional.softplus(dt + self[q + "dt_bias"])
                wide = lambda t: self.padded(t.reshape(T, G, N).repeat_interleave(H // G, dim=1))
                us, dts, B, C = self.padded(u.view(T, H, V)), self.padded(dt), wide(B), wide(C)
                A = -torch.exp(self[q + "A_log"])
                S, out = torch.zeros(len(self.lengths), H, V, N, dtype=torch.float64, device=DEVICE), torch.empty_like(us)
                for t in range(us.shape[1]):
                    S = torch.exp(dts[:, t] * A)[..., None, None] * S + (dts[:, t, :, None] * us[:, t])[..., None] * B[:, t, :, None, :]
                    out[:, t] = (S * C[:, t, :, None, :]).sum(dim=-1)
                y = (self.joined(out) + self[q + "D"][:, None] * u.view(T, H, V)).reshape(T, I) * silu(z)
                y = _rms(y.view(T, m["norm_groups"], -1), eps).reshape(T, I) * self[q + "norm"]
            out = self[p + "ls1"] * self.lin(y, q + "o")
            if mlp["kind"] == "dense":
                f = self.lin(_gelu(self.lin(h, p + "mlp.gate")) * self.lin(h, p + "mlp.up"), p + "mlp.down")
            else:
                r = mlp["router"]
                scores = torch.sigmoid(self.lin(h, p + "mlp.router"))
                choice = (scores + self[p + "mlp.correction"]).view(T, r["groups"]["count"], -1)
                kept = choice.topk(2, dim=-1).values.sum(dim=-1).topk(r["groups"]["keep"], dim=-1).indices
                closed = torch.ones(choice.shape[:2], dtype=torch.bool, device=DEVICE).scatter_(1, kept, False)
                idx = choice.masked_fill(closed[..., None], float("-inf")).reshape(T, -1).topk(r["top"], dim=-1).indices
                f = self.experts(h, p + "mlp", idx, scores.gather(1, idx) * r["scale"], lambda a, b: _clamped(a, b, mlp["expert"]["limit"]))
                s = p + "mlp.shared"
                f = f + self.lin(_clamped(self.lin(h, s + ".gate"), self.lin(h, s + ".up"), mlp["shared"]["limit"]), s + ".down")
            x = x + out + self[p + "ls2"] * f
        return norm(x, "final.norm"), "head"


def exact(case, seed):
    t = _Truth(case, seed)
    h, head = getattr(t, "qwen" if case["model"] in QWEN else case["model"].split("-")[0])()
    rows = list(h.split(t.lengths))
    logits = lambda x: x @ t[head].T
    if case["engine"] == "serving":
        return [logits(torch.stack([x[n - 1 + i] for x, n in zip(rows, _lengths(case))])) for i in range(case["steps"] + 1)]
    if case["portion"] > 1:
        out = {"logits": logits(rows[0][(case["prompt"] - 1) // case["portion"] * case["portion"]:])}
    else:
        out = {"logits": logits(torch.stack([x[-1] for x in rows]))}
    if case["model"] in QWEN:
        page, R = _page(case), case["requests"]
        pages = R * -(-(case["prompt"] + 8) // page)

        def laid(part):
            full = torch.zeros(case["layers"], pages * page, *t.cache[0][part].shape[1:], dtype=torch.float64, device=DEVICE)
            for i, kv in enumerate(t.cache):
                for r, x in enumerate(kv[part].split(t.lengths)):
                    full[i, r * (pages // R) * page:][:len(x)] = x
            return full.view(case["layers"], pages, page, *full.shape[2:])
        out.update(k=laid(0), v=laid(1))
    return out
