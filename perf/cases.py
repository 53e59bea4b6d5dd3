"""Cases to time: what a server or a replaying program has this engine do, from one decoded token to a long prompt.

Most cases are one call of the step function (``ModelRunner.step``: the one the serving engine, ``Model.logits`` and the
replay program run) on a model with random weights, over caches that earlier steps have filled; the result is the logits at
each request's last token.  One case is the serving engine itself in the 32-bit mode, where tokens and fingerprints are
defined to the last bit.  Layer sizes are the benchmark's: the SmolLM2-1.7B shape, the Llama-3-8B shape, and the eight
Kuponex layers of width 2048.
"""

import math

import torch

import bitwise_amd as bw
from bitwise_amd.engine.batch import Segment
from bitwise_amd.engine.runner import ModelRunner
from bitwise_amd.engine.storage import CacheStorage

PAGE = 16
MAX_POSITIONS = 16384
STEP_TOKENS = 2048                   # token budget of a step, as the benchmark's engines have it
WEIGHT_SEED = 77                      # the random model's weights: WEIGHT_SEED + seed


def _llama(hidden, layers, heads, kv_heads, head_dim, ff, vocab, theta, tied):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_act": "silu", "vocab_size": vocab,
            "hidden_size": hidden, "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": kv_heads,
            "head_dim": head_dim, "intermediate_size": ff, "rope_theta": theta, "rms_norm_eps": 1e-5,
            "tie_word_embeddings": tied, "max_position_embeddings": MAX_POSITIONS, "bos_token_id": 1, "eos_token_id": 2}


def _kuponex(width, ff, groups, vocab):
    heads, layers = width // 128, []
    mlp = {"kind": "dense", "ff": ff}
    for _ in range(groups):
        layers.append({"type": "latent_attention", "mlp": mlp,
                       "mixer": {"heads": heads, "dim": 96, "rot_dim": 32, "vdim": 128, "kv_rank": 256, "scale": 128 ** -0.5,
                                 "rot": {"base": 500000.0, "dims": 32}}})
        layers.append({"type": "mlstm", "mlp": mlp, "mixer": {"heads": heads // 2, "dim": 128, "vdim": 256, "gate_cap": 15.0}})
        for _ in range(2):
            layers.append({"type": "gla", "mlp": mlp, "mixer": {"heads": heads, "dim": 64, "vdim": 128, "tau": 16.0, "rank": 64}})
    return {"architecture": "Kuponex", "vocab": vocab, "width": width, "norm": {"eps": 1e-6}, "layers": layers,
            "max_positions": MAX_POSITIONS, "eos_token_id": 2}


SHAPES = {
    "smollm2_1_7b": _llama(2048, 24, 32, 32, 64, 8192, 49152, 130000.0, True),
    "llama3_8b": _llama(4096, 32, 32, 8, 128, 14336, 128256, 500000.0, False),
    "kuponex_2048": _kuponex(2048, 8192, 2, 32000),
}


def _case(name, shape, dtype, batch, context, portion=0, past=0, ragged=False, new=0):
    """``batch`` requests decode a token each behind ``context`` cached ones (``ragged``: behind up to that many, all
    different); beside them one request runs ``portion`` prompt tokens behind ``past`` cached ones.  ``new``: the serving
    engine instead, ``batch`` prompts of up to ``context`` tokens and ``new`` generated tokens each."""
    return {"name": name, "shape": shape, "dtype": dtype, "batch": batch, "context": context, "portion": portion, "past": past,
            "ragged": ragged, "new": new}


def listed():
    return [
        # the smallest call of a chat: one user's next token; its launches and first loads count as much as its bytes
        _case("decode_b1", "smollm2_1_7b", "bfloat16", 1, 331),
        # the benchmark's headline: eight requests with 2,048-token contexts
        _case("decode_b8", "smollm2_1_7b", "bfloat16", 8, 2048),
        # a busy server: many requests of very different lengths, one more than a graph bucket's half
        _case("decode_b43_ragged", "smollm2_1_7b", "bfloat16", 43, 4001, ragged=True),
        # a few long conversations on the larger model with grouped heads
        _case("decode_8b_b5", "llama3_8b", "bfloat16", 5, 4500),
        # a short question arrives
        _case("prefill_117", "smollm2_1_7b", "bfloat16", 0, 0, portion=117),
        # the benchmark's prompt: a whole token budget
        _case("prefill_2048", "smollm2_1_7b", "bfloat16", 0, 0, portion=2048),
        # an ordinary prompt on the larger model
        _case("prefill_8b_777", "llama3_8b", "bfloat16", 0, 0, portion=777),
        # the last portion of a long document: 2,048 tokens behind 6,144 cached ones
        _case("portion_8b_2048", "llama3_8b", "bfloat16", 0, 0, portion=2048, past=6144),
        # continuous batching: decoding requests beside a portion of somebody's prompt
        _case("mixed_7_1341", "smollm2_1_7b", "bfloat16", 7, 600, portion=1341, past=640),
        # true 32-bit mode: the benchmark's second decode line
        _case("fp32_decode_b8", "smollm2_1_7b", "float32", 8, 1024),
        # true 32-bit mode through the serving engine: prompts, then decoded tokens; the bits are defined
        _case("fp32_serve_b5", "smollm2_1_7b", "float32", 5, 150, ragged=True, new=6),
        # recurrent memories and attention over a compressed cache: a whole budget, cuts exact (the default)
        _case("kuponex_prefill_2048", "kuponex_2048", "bfloat16", 0, 0, portion=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "prefill", "mixed", "fp32", "serve", "kuponex"))
        shape = rng.choice(("smollm2_1_7b", "smollm2_1_7b", "llama3_8b"))
        if kind == "decode":
            c = _case("", shape, "bfloat16", _log(rng, 1, 64), _log(rng, 16, 8192), ragged=rng.random() < 0.5)
        elif kind == "prefill":
            c = _case("", shape, "bfloat16", 0, 0, portion=_log(rng, 16, STEP_TOKENS), past=rng.choice((0, 0, _log(rng, 64, 6144) // 16 * 16)))
        elif kind == "mixed":
            c = _case("", shape, "bfloat16", _log(rng, 1, 24), _log(rng, 16, 4096), portion=_log(rng, 64, STEP_TOKENS - 64),
                      past=rng.choice((0, 64 * rng.randint(1, 32))), ragged=True)
        elif kind == "fp32":
            c = _case("", "smollm2_1_7b", "float32", _log(rng, 1, 32), _log(rng, 16, 2048), ragged=rng.random() < 0.5)
        elif kind == "serve":
            c = _case("", "smollm2_1_7b", "float32", _log(rng, 1, 8), _log(rng, 16, 200), ragged=True, new=rng.randint(2, 8))
        else:
            c = _case("", "kuponex_2048", "bfloat16", 0, 0, portion=_log(rng, 64, STEP_TOKENS))
        del c["name"]
        cached = sum(p for p, _ in _requests(c))
        largest = work(listed()[7])
        w = work(c)
        # no more than the largest listed case, and caches that are filled in about half a second
        if max(w["bytes"], w["flops"] / 50) <= max(largest["bytes"], largest["flops"] / 50) and cached <= (25000 if shape == "llama3_8b" else 80000):
            return c


def _requests(case):
    """(cached tokens, tokens of this step) per request: the portion last."""
    out = []
    for i in range(case["batch"]):
        n = case["context"]
        if case["ragged"]:
            n = max(1, int(n * ((i * 0.6180339887498949 + 0.37) % 1.0)))
        out.append((n, 1))
    if case["portion"]:
        out.append((case["past"], case["portion"]))
    return out


def _tokens(case, seed):
    """Every request's token ids, cached ones and this step's together."""
    cfg = SHAPES[case["shape"]]
    vocab = cfg["vocab_size"] if "vocab_size" in cfg else cfg["vocab"]
    g = torch.Generator().manual_seed(seed)
    return [torch.randint(0, vocab, (p + n,), generator=g).tolist() for p, n in _requests(case)]


def prepare(case, seed):
    tokens, reqs = _tokens(case, seed), _requests(case)
    model = bw.Model.random(SHAPES[case["shape"]], WEIGHT_SEED + seed, case["dtype"], on_device=True)
    if case["new"]:
        prompts = [t[:-1] for t in tokens]
        pages = sum((len(p) + case["new"]) // PAGE + 2 for p in prompts)
        engine = bw.Engine(model, None, bw.EngineConfig(num_blocks=pages, max_batched_tokens=STEP_TOKENS, max_num_seqs=case["batch"],
                                                        prefix_caching=False, block_size=PAGE, dtype=case["dtype"], max_model_len=4096))
        state = {"case": case, "model": model, "engine": engine, "prompts": prompts}
        warm = engine.add_request(prompts[0][:8], bw.SamplingParams(max_new_tokens=2, ignore_eos=True))     # a server that has run before
        while not engine.result(warm).finished:
            engine.step()
        return state
    asm = model.assembled
    pages = [(p + n + PAGE - 1) // PAGE for p, n in reqs]
    storage = CacheStorage(asm, sum(pages), len(reqs), PAGE)
    runner = ModelRunner(asm, storage, max_model_len=MAX_POSITIONS // 2, max_rows=STEP_TOKENS, max_logit_rows=max(64, len(reqs)))
    tables, first = [], 0
    for n in pages:
        tables.append([list(range(first, first + n)) for _ in asm.group_specs])
        first += n
    # the caches: what earlier steps of the same requests leave (the last cached token of a decoding request has been
    # decoded, so the step's graph is captured as a running server's is)
    alone = not case["portion"]
    fill, room = [], STEP_TOKENS
    for i, (p, n) in enumerate(reqs):
        start, end = 0, p - 1 if alone else p
        while start < end:
            take = min(end - start, room)
            fill.append(Segment(tokens[i][start:start + take], start, tables[i], i))
            start, room = start + take, room - take
            if not room:
                runner.step(fill)
                fill, room = [], STEP_TOKENS
    if fill:
        runner.step(fill)
    if alone:
        runner.step([Segment(tokens[i][p - 1:p], p - 1, tables[i], i, (0,)) for i, (p, n) in enumerate(reqs)])
    step = [Segment(tokens[i][p:p + n], p, tables[i], i, (n - 1,)) for i, (p, n) in enumerate(reqs)]
    return {"case": case, "model": model, "storage": storage, "runner": runner, "segments": step}


def run(state):
    if "engine" in state:
        engine, n = state["engine"], state["case"]["new"]
        ids = [engine.add_request(p, bw.SamplingParams(max_new_tokens=n, ignore_eos=True)) for p in state["prompts"]]
        while not engine.idle():
            engine.step()
        results = [engine.result(i) for i in ids]
        # (a fingerprint is a 64-bit word: as two halves it fits a whole number of any kind)
        return {"tokens": torch.tensor([r.tokens for r in results]),
                "fingerprints": torch.tensor([[r.logits_fingerprint >> 32, r.logits_fingerprint & 0xFFFFFFFF] for r in results])}
    if state["model"].assembled.has_state:
        state["storage"].reset_slot(0)            # a request takes the slot
    return {"logits": state["runner"].step(state["segments"])}


def _sizes(cfg):
    """(parameters of the matrices a token goes through, parameters read a step, cache elements a token, the pairs' cost:
    multiply-adds a query and key, all layers)."""
    if "hidden_size" in cfg:
        h, ff, v, L = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"], cfg["num_hidden_layers"]
        q, kv = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
        body = L * (h * (q + 2 * kv) + q * h + 3 * h * ff)
        return body, v * h, L * 2 * kv, L * 2 * q
    w, v, body, cache, pair = cfg["width"], cfg["vocab"], 0, 0, 0
    for layer in cfg["layers"]:
        m = layer["mixer"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        if layer["type"] == "latent_attention":
            R, C = m["rot_dim"], m["kv_rank"]
            body += w * (H * (D + R) + C + R) + H * D * C + H * C * V + H * V * w
            cache, pair = cache + C + R, pair + H * (2 * C + R)
        else:
            body += w * H * (2 * D + 2 * V) + H * V * w + (w * 2 * H if layer["type"] == "mlstm" else m["rank"] * (w + H * D))
        body += 3 * w * layer["mlp"]["ff"]
    return body, v * w, cache, pair


def work(case):
    cfg, reqs = SHAPES[case["shape"]], _requests(case)
    body, head, cache, pair = _sizes(cfg)
    size = 4 if case["dtype"] == "float32" else 2
    vocab = cfg["vocab_size"] if "vocab_size" in cfg else cfg["vocab"]
    if case["new"]:
        # one step for the prompts, then a step a token: weights once a step, the caches behind them
        rows, steps = sum(p for p, _ in reqs) + case["batch"] * (case["new"] - 1), case["new"]
        kv = sum(p * steps for p, _ in reqs)
        pairs = sum(p * (p + 1) / 2 + p * (steps - 1) for p, _ in reqs)
        wanted = case["batch"] * steps
    else:
        rows, steps = sum(n for _, n in reqs), 1
        kv = sum(p + n for p, n in reqs)
        pairs = sum(p * n + n * (n + 1) / 2 for p, n in reqs)
        wanted = len(reqs)
    state = 0.0
    for layer in cfg.get("layers", ()):
        if layer["type"] != "latent_attention":     # a memory's update and read-out of every token
            m = layer["mixer"]
            state += 2 * m["heads"] * m["dim"] * m["vdim"]
    return {"bytes": float(steps * (body + head) * 2 + kv * cache * size + rows * cache * size + 4 * wanted * vocab),
            "flops": float(2 * (rows * (body + state) + wanted * head + pairs * pair))}


def tolerance(case):
    if case["new"]:
        return "exact"               # the 32-bit mode's tokens and fingerprints are defined to the last bit
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.2}


# ------------------------------------------------------------------------------------------------ in 64 bits

F = torch.float64


class _Weights:
    """The random model's tensors as it draws them: standard normals in the model's order from one generator, shaped by
    kind, stored in bfloat16; kept in bfloat16 and widened where they are used."""

    def __init__(self, case, seed):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(WEIGHT_SEED + seed)
        self.t = {}
        for name, spec in bw.describe(SHAPES[case["shape"]]).items():      # (names, shapes and kinds; nothing is computed)
            z = torch.randn(spec.shape, generator=gen, dtype=torch.float32, device="cuda")
            shaped = {"norm": lambda: 1.0 + 0.1 * z, "around_zero": lambda: 0.1 * z, "unit_interval": lambda: torch.sigmoid(z),
                      "bias": lambda: z, "linear": lambda: 0.02 * z, "embedding": lambda: 0.02 * z}[spec.kind]()
            self.t[name] = shaped.to(torch.bfloat16)

    def __getitem__(self, name):
        return self.t[name].to(F)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate(x, positions, inv):
    """x [T, heads, 2 * len(inv)]: pairs (i, i + half)."""
    a = positions[:, None, None] * inv
    c, s, half = torch.cos(a), torch.sin(a), inv.numel()
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _attend(q, k, v, scale, sink=None):
    """Causal attention of the last q.shape[0] of k.shape[0] positions; q [T, H, D], k [S, G, D], v [S, G, V]."""
    T, H, S, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    out = torch.empty(T, H, v.shape[2], dtype=F, device=q.device)
    keys = torch.arange(S, device=q.device)
    for g in range(G):
        heads = slice(g * H // G, (g + 1) * H // G)
        for t0 in range(0, T, 2048):
            qq = q[t0:t0 + 2048, heads]
            s = torch.einsum("thd,sd->hts", qq, k[:, g]) * scale
            seen = keys[None, :] <= (S - T + t0 + torch.arange(qq.shape[0], device=q.device))[:, None]
            s = s.masked_fill(~seen, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[heads][:, None, None].expand(-1, s.shape[1], 1)], -1)
            p = torch.softmax(s, -1)[..., :S]
            out[t0:t0 + 2048, heads] = torch.einsum("hts,sv->thv", p, v[:, g])
    return out


def _exact_llama(cfg, w, requests):
    """Last-row logits of every request.  ``requests``: token lists, run whole, all rows side by side."""
    H, G, D, eps = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["rms_norm_eps"]
    dev = "cuda"
    # (angles are 32-bit products of a 32-bit frequency, which is part of the rotary definition)
    inv = 1.0 / torch.pow(torch.tensor(cfg["rope_theta"], dtype=torch.float32), torch.arange(0, D, 2, dtype=torch.float32) / D)
    inv = inv.to(dev).to(F)
    lens = [len(r) for r in requests]
    ids = torch.tensor(sum(requests, []), device=dev)
    pos = torch.cat([torch.arange(n, dtype=F, device=dev) for n in lens])
    x = w["model.embed_tokens.weight"][ids]
    last = torch.cumsum(torch.tensor(lens), 0).to(dev) - 1
    step = 16384

    def linear(a, name):
        m = w[name]
        return torch.cat([a[i:i + step] @ m.T for i in range(0, a.shape[0], step)])

    for i in range(cfg["num_hidden_layers"]):
        pre, final = f"model.layers.{i}.", i == cfg["num_hidden_layers"] - 1
        h = _rms(x, eps) * w[pre + "input_layernorm.weight"]
        q = linear(h, pre + "self_attn.q_proj.weight").view(-1, H, D)
        k = linear(h, pre + "self_attn.k_proj.weight").view(-1, G, D)
        v = linear(h, pre + "self_attn.v_proj.weight").view(-1, G, D)
        q, k = _rotate(q, pos, inv), _rotate(k, pos, inv)
        o, at = [], 0
        for n in lens:
            o.append(_attend(q[at:at + n], k[at:at + n], v[at:at + n], D ** -0.5))
            at += n
        o = torch.cat(o).view(-1, H * D)
        if final:                       # only the last rows go on
            x, o = x[last], o[last]
        x = x + linear(o, pre + "self_attn.o_proj.weight")
        h = _rms(x, eps) * w[pre + "post_attention_layernorm.weight"]
        m_gate, m_up, m_down = w[pre + "mlp.gate_proj.weight"], w[pre + "mlp.up_proj.weight"], w[pre + "mlp.down_proj.weight"]
        for j in range(0, x.shape[0], step):
            part = h[j:j + step]
            x[j:j + step] += (torch.nn.functional.silu(part @ m_gate.T) * (part @ m_up.T)) @ m_down.T
    x = _rms(x, eps) * w["model.norm.weight"]
    return x @ w["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"].T


def _exact_kuponex(cfg, w, tokens):
    dev, eps, T = "cuda", cfg["norm"]["eps"], len(tokens)
    pos = torch.arange(T, dtype=F, device=dev)
    x = w["embed"][torch.tensor(tokens, device=dev)]
    around_zero = lambda a, name: _rms(a, eps) * (1.0 + w[name])
    for i, layer in enumerate(cfg["layers"]):
        pre, m = f"l{i}.", layer["mixer"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        n1 = around_zero(x, pre + "norm1")
        before = torch.cat([torch.zeros_like(n1[:1]), n1[:-1]])
        h = n1 + (before - n1) * w[pre + "shift"]
        lin = lambda name: h @ w[pre + "mix." + name].T
        if layer["type"] == "latent_attention":
            R, C, dims = m["rot_dim"], m["kv_rank"], m["rot"]["dims"]
            inv = m["rot"]["base"] ** (-2.0 * torch.arange(dims // 2, dtype=F, device=dev) / dims)
            q = lin("q").view(T, H, D + R)
            kv = lin("dkv")
            c = _rms(kv[:, :C], eps) * w[pre + "mix.dkv.norm"]
            q = torch.cat([q[..., :D], _rotate(q[..., D:D + dims], pos, inv), q[..., D + dims:]], -1)
            kr = torch.cat([_rotate(kv[:, None, C:C + dims], pos, inv), kv[:, None, C + dims:]], -1)
            k = torch.cat([(c @ w[pre + "mix.uk"].T).view(T, H, D), kr.expand(T, H, R)], -1)
            val = (c @ w[pre + "mix.uv"].T).view(T, H, V)
            o = _attend(q, k, val, m["scale"], w[pre + "mix.sink"]).reshape(T, H * V)
        else:
            q, k, v = lin("q").view(T, H, D) * D ** -0.5, lin("k").view(T, H, D), lin("v").view(T, H, V)
            S = torch.zeros(H, D, V, dtype=F, device=dev)
            o = torch.empty(T, H, V, dtype=F, device=dev)
            if layer["type"] == "mlstm":
                cap = m["gate_cap"]
                gi = cap * torch.tanh((lin("i") + w[pre + "mix.i.b"]) / cap)
                gf = torch.nn.functional.logsigmoid(cap * torch.tanh((lin("f") + w[pre + "mix.f.b"]) / cap))
                n, mx, ex = torch.zeros(H, D, dtype=F, device=dev), torch.zeros(H, dtype=F, device=dev), []
                for t in range(T):
                    new = torch.maximum(gf[t] + mx, gi[t])
                    a, b = torch.exp(gf[t] + mx - new)[:, None], torch.exp(gi[t] - new)[:, None]
                    kt = b * k[t]
                    S.mul_(a[:, :, None]).addcmul_(kt[:, :, None], v[t][:, None, :])
                    n = a * n + kt
                    mx = new
                    den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-mx)) + 1e-6
                    o[t] = (q[t][:, None, :] @ S)[:, 0] / den[:, None]
                o = _rms(o, eps).reshape(T, H * V) * w[pre + "mix.norm"] * torch.sigmoid(lin("g"))
            else:
                alpha = torch.sigmoid(lin("a1") @ w[pre + "mix.a2"].T + w[pre + "mix.a2.b"]).pow(1.0 / m["tau"]).view(T, H, D)
                for t in range(T):
                    S.mul_(alpha[t][:, :, None]).addcmul_(k[t][:, :, None], v[t][:, None, :])
                    o[t] = (q[t][:, None, :] @ S)[:, 0]
                o = (_rms(o, eps) * w[pre + "mix.norm"]).reshape(T, H * V) * torch.nn.functional.silu(lin("g"))
        y = o @ w[pre + "mix.o"].T
        h2 = around_zero(x, pre + "norm2")
        gelu = torch.nn.functional.gelu(h2 @ w[pre + "mlp.gate"].T, approximate="tanh")
        x = x + y + (gelu * (h2 @ w[pre + "mlp.up"].T)) @ w[pre + "mlp.down"].T
    return around_zero(x[-1:], "final.norm") @ w["head"].T


def exact(case, seed):
    if case["new"]:
        return None                                         # whole numbers, compared as they are
    cfg, tokens = SHAPES[case["shape"]], _tokens(case, seed)
    body = _sizes(cfg)[0]
    if 2.0 * body * sum(len(t) for t in tokens) > 4.5e14:   # about fifteen seconds at the card's 64-bit rate
        return None
    w = _Weights(case, seed)
    if case["shape"].startswith("kuponex"):
        return {"logits": _exact_kuponex(cfg, w, tokens[0])}
    return {"logits": _exact_llama(cfg, w, tokens)}
