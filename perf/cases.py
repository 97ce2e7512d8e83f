"""What is timed when this engine is made faster: steps of a loaded model through ``Engine.step``, as a serving program makes them.

A case is a model at a real model's layer sizes (random weights), its type, the requests that decode (``requests`` of about
``context`` tokens each; ``spread``: from half of that to one and a half times) and a prompt (``prompt`` tokens, cut into portions
of at most ``portion`` tokens, one a step) that enters beside them.  One pass is the steps it takes to bring the prompt in, or one
decode step where there is none; every decoding request gets one token a step.  Tokens are given, not sampled, so that any correct
implementation returns the same logits.  The prompt's request ends with the pass; the decoding requests go on from pass to pass, one
token longer each, as they do in a server.
"""
import math
import random
import zlib

import torch

from zedinfer_amd import InferenceEngine, SchedulerConfig, StepEntry
from zedinfer_amd.config import find_architecture
from zedinfer_amd.engine import Engine

ROOM = 2048        # tokens that a decoding request can still grow by when it is handed over
WARM = 8           # passes the engine has made when it is handed over: a kind of step is recorded once it has come a few times
PAGE = 16

SIZES = {
    # the benchmark's model and the next larger one of the same architecture
    "1.5B": dict(width=1536, heads=12, kv_heads=2, ff=8960, layers=28, vocab=151936, tied=True, experts=32, top=4, expert_ff=1536),
    "7B": dict(width=3584, heads=28, kv_heads=4, ff=18944, layers=28, vocab=152064, tied=False, experts=32, top=4, expert_ff=2560),
}
DESIGN_LAYERS, DESIGN_VOCAB = 8, 32000      # the Dedelorn design: three layers of the delta rule, one of latent attention, twice


def _case(name, model="qwen2", sizes="1.5B", dtype="bfloat16", requests=0, context=0, spread=False, prompt=0, portion=2048):
    c = dict(model=model, sizes=sizes, dtype=dtype, requests=requests, context=context, spread=spread, prompt=prompt, portion=portion)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one user waiting for a token: the smallest call there is, launches and latency
        _case("decode 1", requests=1, context=2048),
        # the benchmark's own headline: eight requests decoding
        _case("decode 8", requests=8, context=2048),
        # a busy server of the small model
        _case("decode 64", requests=64, context=2048),
        # a few requests with long documents: the cache is most of what a step reads
        _case("decode 8 long", requests=8, context=12300),
        # a server of the larger model with many short chats of different lengths
        _case("decode 150 ragged 7B", sizes="7B", requests=150, context=360, spread=True),
        # a chat message enters an idle server (the reference's own bench -p 128)
        _case("prompt 128", prompt=128),
        # the benchmark's prompt, in one step
        _case("prompt 2048", prompt=2048),
        # continuous batching: a long prompt enters in portions beside requests that decode
        _case("mixed 7B", sizes="7B", requests=23, context=1500, spread=True, prompt=3211),
        # the float32 path (a checkpoint stored in 32 bits, results to compare others with): a prompt and decoding
        _case("float32 prompt 450", dtype="float32", prompt=450),
        _case("float32 decode 8", dtype="float32", requests=8, context=400),
        # a design with recurrent layers, latent attention and routed experts: a prompt and a busy server
        _case("dedelorn prompt 2000", model="dedelorn", prompt=2000),
        _case("dedelorn decode 32", model="dedelorn", requests=32, context=1500, spread=True),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model, sizes, dtype = rng.choice([("qwen2", "1.5B", "bfloat16")] * 3 + [("qwen2", "7B", "bfloat16")] * 2 +
                                     [("qwen2", "1.5B", "float32"), ("dedelorn", "1.5B", "bfloat16")])
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed"])
    tokens = 6000 if dtype == "float32" else 50000 if sizes == "7B" else 100000      # cached, over all requests
    longest = 450 if dtype == "float32" else 2048
    requests = context = prompt = 0
    if kind != "prompt":
        requests = _log_uniform(rng, 1, 16 if dtype == "float32" else 150)
        context = min(_log_uniform(rng, 64, 12300), max(64, tokens // requests))
        if dtype == "float32":
            context = min(context, 900)
    if kind != "decode":
        prompt = _log_uniform(rng, 16, longest)
    return _case("", model, sizes, dtype, requests, context, rng.random() < 0.5, prompt, rng.choice([512, 2048]))


# ---- the models -----------------------------------------------------------------------------------------------------------
def _config(case):
    z = SIZES[case["sizes"]]
    if case["model"] == "qwen2":
        return dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", hidden_size=z["width"], intermediate_size=z["ff"],
                    vocab_size=z["vocab"], max_position_embeddings=32768, num_hidden_layers=z["layers"],
                    num_attention_heads=z["heads"], num_key_value_heads=z["kv_heads"], head_dim=128, rope_theta=1000000.0,
                    rms_norm_eps=1e-6, tie_word_embeddings=z["tied"], use_sliding_window=False, torch_dtype="bfloat16")
    layers, last_latent = [], None
    for i in range(DESIGN_LAYERS):
        if i % 4 == 3:
            mixer = dict(heads=z["heads"], dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5, mask=dict(size=1024),
                         rot=dict(base=10000.0, dims=64))
            if last_latent is not None:
                mixer["kv_from"], last_latent = last_latent, None
            else:
                last_latent = i
            kind = "latent_attention"
        else:
            mixer, kind = dict(heads=z["heads"], kv_heads=z["heads"] // 2, dim=128, vdim=128, conv=4), "delta"
        mlp = dict(kind="dense", ff=z["ff"]) if i % 2 == 0 else \
            dict(kind="moe", expert=dict(ff=z["expert_ff"]), router=dict(experts=z["experts"], top=z["top"], scale=1.0))
        layers.append(dict(type=kind, mixer=mixer, mlp=mlp))
    return dict(architecture="Dedelorn", width=z["width"], vocab=DESIGN_VOCAB, norm=dict(eps=1e-6), layers=layers)


def _shapes(case):
    """Every tensor's name and shape, as the checkpoint has them."""
    cfg, out = _config(case), {}
    if case["model"] == "qwen2":
        H, F, V = cfg["hidden_size"], cfg["intermediate_size"], cfg["vocab_size"]
        Q, KV = cfg["num_attention_heads"] * 128, cfg["num_key_value_heads"] * 128
        out["model.embed_tokens.weight"] = (V, H)
        for i in range(cfg["num_hidden_layers"]):
            p = "model.layers.%d." % i
            out[p + "input_layernorm.weight"] = out[p + "post_attention_layernorm.weight"] = (H,)
            for n, r in (("q", Q), ("k", KV), ("v", KV)):
                out[p + "self_attn.%s_proj.weight" % n], out[p + "self_attn.%s_proj.bias" % n] = (r, H), (r,)
            out[p + "self_attn.o_proj.weight"] = (H, Q)
            out[p + "mlp.gate_proj.weight"] = out[p + "mlp.up_proj.weight"] = (F, H)
            out[p + "mlp.down_proj.weight"] = (H, F)
        out["model.norm.weight"] = (H,)
        if not cfg["tie_word_embeddings"]:
            out["lm_head.weight"] = (V, H)
        return out
    W = cfg["width"]
    out["embed"], out["embed.norm"], out["final.norm"], out["head"] = (cfg["vocab"], W), (W,), (W,), (cfg["vocab"], W)
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        out[p + "norm1"] = (W,)
        h = m["heads"]
        if layer["type"] == "delta":
            qk, v = m["kv_heads"] * m["dim"], h * m["vdim"]
            out.update({p + "mix.q": (qk, W), p + "mix.q.conv": (qk, m["conv"]), p + "mix.k": (qk, W), p + "mix.k.conv": (qk, m["conv"]),
                        p + "mix.v": (v, W), p + "mix.v.conv": (v, m["conv"]), p + "mix.b": (h, W), p + "mix.a": (h, W),
                        p + "mix.A_log": (h,), p + "mix.dt_bias": (h,), p + "mix.norm": (m["vdim"],), p + "mix.g": (v, W),
                        p + "mix.o": (W, v)})
        else:
            out.update({p + "mix.q": (h * (m["dim"] + m["rot_dim"]), W), p + "mix.uk": (h * m["dim"], m["kv_rank"]),
                        p + "mix.uv": (h * m["vdim"], m["kv_rank"]), p + "mix.o": (W, h * m["vdim"])})
            if "kv_from" not in m:
                out.update({p + "mix.dkv": (m["kv_rank"] + m["rot_dim"], W), p + "mix.dkv.norm": (m["kv_rank"],)})
        if mlp["kind"] == "dense":
            out.update({p + "mlp.gate": (mlp["ff"], W), p + "mlp.up": (mlp["ff"], W), p + "mlp.down": (W, mlp["ff"])})
        else:
            E, ff = mlp["router"]["experts"], mlp["expert"]["ff"]
            out.update({p + "mlp.router": (E, W), p + "mlp.correction": (E,)})
            for e in range(E):
                out.update({p + "mlp.e%d.up" % e: (ff, W), p + "mlp.e%d.down" % e: (W, ff)})
    return out


def _weights(case, seed):
    """Random weights on the GPU, from the seed and the tensors' names alone."""
    dt = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    out, g = {}, torch.Generator(device="cuda")
    for name, shape in _shapes(case).items():
        g.manual_seed((seed * 1000003 + zlib.crc32(name.encode())) % (1 << 62))
        last = name.split(".")[-1]
        if "norm" in name:
            t = 1.0 + 0.05 * torch.randn(shape, generator=g, device="cuda")
        elif last == "A_log":            # decays from a few tokens to a few thousand, as such layers are trained with
            t = torch.log(1.0 + 15.0 * torch.rand(shape, generator=g, device="cuda"))
        elif last == "dt_bias":
            step = torch.exp(math.log(0.001) + math.log(100.0) * torch.rand(shape, generator=g, device="cuda"))
            t = torch.log(torch.expm1(step))
        elif last == "conv":
            t = 0.3 * torch.randn(shape, generator=g, device="cuda")
        elif name in ("model.embed_tokens.weight", "embed"):      # as large as what the layers add to it, all together
            t = torch.randn(shape, generator=g, device="cuda", dtype=dt)
        elif last == "bias":
            t = 0.1 * torch.randn(shape, generator=g, device="cuda")
        else:
            # what writes into the residual stream is smaller the more layers do, as models are initialised and trained
            writes = last in ("o", "down") or ".o_proj." in name or ".down_proj." in name
            layers = DESIGN_LAYERS if case["model"] == "dedelorn" else SIZES[case["sizes"]]["layers"]
            t = torch.randn(shape, generator=g, device="cuda", dtype=dt).mul_(0.02 / math.sqrt(2 * layers) if writes else 0.02)
        out[name] = t.to(dt)
    if case["model"] == "qwen2" and SIZES[case["sizes"]]["tied"]:
        out["lm_head.weight"] = out["model.embed_tokens.weight"]
    return out


# ---- inputs ---------------------------------------------------------------------------------------------------------------
def _contexts(case):
    B, C = case["requests"], case["context"]
    return [max(1, C // 2 + C * i // max(B - 1, 1)) if case["spread"] else C for i in range(B)]


def _portions(case):
    n, most = case["prompt"], case["portion"]
    return [min(most, n - at) for at in range(0, n, most)]


def _vocab(case):
    return DESIGN_VOCAB if case["model"] == "dedelorn" else SIZES[case["sizes"]]["vocab"]


def _tokens(case, seed):
    """(the cached tokens of every decoding request, the tokens each of them is given next, in turn, the prompt)."""
    rng, V = random.Random("%s %s" % (seed, sorted((k, v) for k, v in case.items() if k != "name"))), _vocab(case)
    ids = lambda n: [rng.randrange(100, V - 100) for _ in range(n)]  # noqa: E731
    return [ids(n) for n in _contexts(case)], [ids(64) for _ in range(case["requests"])], ids(case["prompt"])


def prepare(case, seed):
    """A loaded engine whose decoding requests hold their tokens, and that has made a few steps of the kind."""
    cached, coming, prompt = _tokens(case, seed)
    d = _config(case)
    arch = find_architecture(d)
    fc = arch.forward_config(arch.config_cls.from_dict(d))
    B, longest = case["requests"], max([len(c) for c in cached] + [0])
    blocks = sum(-(-(len(c) + ROOM) // PAGE) + 1 for c in cached) + -(-len(prompt) // PAGE) + 16
    sched = SchedulerConfig(num_kv_blocks=blocks, kv_block_size=PAGE, max_batch_requests=B + 1, max_batch_tokens=8192 + B,
                            max_prefill_tokens=8192, max_seq_len=max(16384, longest + ROOM))
    engine = Engine(fc, _weights(case, seed), case["dtype"], sched)
    seqs = [engine.open(("request", i)) for i in range(B)]
    # the requests' prompts, several a step
    room, entries = 8192, []
    for seq, ids in zip(seqs, cached):
        at = 0
        while at < len(ids):
            n = min(room, len(ids) - at)
            entries.append(StepEntry(seq, ids[at:at + n]))
            at, room = at + n, room - n
            if room == 0 or at < len(ids):
                engine.step(entries)
                room, entries = 8192, []
    if entries:
        engine.step(entries)
    serving = InferenceEngine(engine)       # from here on as a server runs it: a size's choices are measured at its first step
    state = dict(serving=serving, engine=engine, seqs=seqs, coming=coming, portions=_portions(case), prompt=prompt, steps=0, passes=0)
    for _ in range(WARM):
        run(state)
    torch.cuda.synchronize()
    return state


def run(state):
    engine, out = state["engine"], []
    portions, prompt, at = state["portions"], None, 0
    if portions:
        state["passes"] += 1
        prompt = engine.open(("prompt", state["passes"]), len(state["prompt"]))
    for n in portions or [0]:
        entries = [StepEntry(seq, [ids[state["steps"] % len(ids)]], [0]) for seq, ids in zip(state["seqs"], state["coming"])]
        if n:
            at += n
            entries.append(StepEntry(prompt, state["prompt"][at - n:at], [n - 1] if at == len(state["prompt"]) else []))
        logits = engine.step(entries)
        state["steps"] += 1
        if logits is not None:
            out.append(logits)
    if prompt is not None:
        engine.close(prompt)
    return out


# ---- the work that cannot be done without ---------------------------------------------------------------------------------
def _counts(case):
    """(the parameters of the layers that every token meets, those of one expert over all layers, tokens a layer of attention
    sees at most or 0 for all, heads x (score and value dims) and cached values a token, both over all layers, state values)."""
    cfg = _config(case)
    if case["model"] == "qwen2":
        H, F, L = cfg["hidden_size"], cfg["intermediate_size"], cfg["num_hidden_layers"]
        Q, KV = cfg["num_attention_heads"] * 128, cfg["num_key_value_heads"] * 128
        return L * (H * (Q + 2 * KV) + Q * H + 3 * H * F), 0, 0, 2 * Q * L, 2 * KV * L, 0
    always = expert = dims = cache = state = 0
    for name, shape in _shapes(case).items():
        if name.startswith("l") and len(shape) == 2:
            if ".e" in name:
                expert += shape[0] * shape[1]
            else:
                always += shape[0] * shape[1]
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "delta":
            state += m["heads"] * m["dim"] * m["vdim"]
        else:
            dims += m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
            cache += m["kv_rank"] + m["rot_dim"]
    return always, expert // SIZES[case["sizes"]]["experts"], 1024, dims, cache, state


def work(case):
    z, el = SIZES[case["sizes"]], 4 if case["dtype"] == "float32" else 2
    H, V, B = z["width"], _vocab(case), case["requests"]
    always, expert, window, dims, cache, state = _counts(case)
    total_bytes = total_flops = 0.0
    lens, past = _contexts(case), 0
    for k, n in enumerate(_portions(case) or [0]):
        rows = B + n
        wanted = B + (1 if n and past + n == case["prompt"] else 0)
        experts = min(z["experts"], z["top"] * rows) if expert else 0
        seen = [min(c + k + 1, window or c + k + 1) for c in lens]
        read = sum(seen) + (min(past, window or past) if n else 0)
        pairs = sum(seen) + sum(min(past + j + 1, window or past + j + 1) for j in range(n))
        total_bytes += el * (always + expert * experts + (V * H if wanted else 0) + cache * (read + rows) + H * rows)
        total_bytes += 4 * (V * wanted + 2 * state * (B + (1 if n else 0)))
        total_flops += 2.0 * rows * (always + expert * (z["top"] if expert else 0)) + 2.0 * wanted * V * H
        total_flops += 2.0 * dims * pairs + 6.0 * state * rows
        past += n
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    # About four times what was seen: float32 1.2e-6 against exact(); bfloat16 0.0023 to 0.0026 and, at the 7B sizes (wider sums,
    # whose gains are larger with these weights), 0.0074, each twice in a difference of two; in the design with experts a
    # router's near-tie may fall the other way.
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4}
    rel = 0.03 if case["sizes"] == "7B" else 0.02 if case["model"] == "dedelorn" else 0.012
    return {"rel": rel, "max": 10 * rel}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------
D = torch.float64


def _rms(x, eps, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _attend(q, k, v, scale, window):
    """One sequence: q, k [T, heads, d], v [T, heads, dv] -> [T, heads, dv]; causal, under a window if there is one."""
    T = q.shape[0]
    out = torch.empty(T, q.shape[1], v.shape[2], dtype=D, device=q.device)
    j = torch.arange(T, device=q.device)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    rows = max(16, 100_000_000 // (T * q.shape[1]))
    for a in range(0, T, rows):
        b = min(T, a + rows)
        lo = max(0, a - window + 1) if window else 0
        s = torch.matmul(q[a:b].transpose(0, 1).contiguous(), kt[:, :, lo:b].contiguous()) * scale
        i = torch.arange(a, b, device=q.device)[:, None]
        hidden = j[None, lo:b] > i
        if window:
            hidden = hidden | (i - j[None, lo:b] >= window)
        s.masked_fill_(hidden, -math.inf)
        out[a:b] = torch.matmul(torch.softmax(s, -1), vt[:, lo:b].contiguous()).transpose(0, 1)
    return out


def _by_rows(f, x, rows=16384):
    return torch.cat([f(x[a:a + rows]) for a in range(0, x.shape[0], rows)])


def _qwen2_64(case, w, ids, lens, want):
    cfg = _config(case)
    eps, nh, nkv = cfg["rms_norm_eps"], cfg["num_attention_heads"], cfg["num_key_value_heads"]
    x = w["model.embed_tokens.weight"][ids].to(D)
    pos = torch.cat([torch.arange(n, device=x.device) for n in lens]).to(D)
    a = pos[:, None] * cfg["rope_theta"] ** (-torch.arange(64, device=x.device, dtype=D) / 64)
    cos, sin = torch.cos(a)[:, None], torch.sin(a)[:, None]

    def turn(t):
        u, v = t[..., :64], t[..., 64:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)

    for i in range(cfg["num_hidden_layers"]):
        p = "model.layers.%d." % i
        t = lambda n: w[p + n].to(D)  # noqa: E731
        n1 = _rms(x, eps, t("input_layernorm.weight"))
        q, k, v = ((n1 @ t("self_attn.%s_proj.weight" % n).t() + t("self_attn.%s_proj.bias" % n)).view(len(ids), -1, 128) for n in "qkv")
        q, k = turn(q), turn(k)
        k, v = k.repeat_interleave(nh // nkv, 1), v.repeat_interleave(nh // nkv, 1)
        o = torch.cat([_attend(*s, 128 ** -0.5, 0) for s in zip(q.split(lens), k.split(lens), v.split(lens))])
        x = x + o.reshape(len(ids), -1) @ t("self_attn.o_proj.weight").t()
        g, u, d, n2 = t("mlp.gate_proj.weight"), t("mlp.up_proj.weight"), t("mlp.down_proj.weight"), t("post_attention_layernorm.weight")

        def ff(r):
            r = _rms(r, eps, n2)
            return (torch.nn.functional.silu(r @ g.t()) * (r @ u.t())) @ d.t()

        x = x + _by_rows(ff, x)
    return _rms(x[want], eps, w["model.norm.weight"].to(D)) @ w["lm_head.weight"].to(D).t()


def _dedelorn_64(case, w, ids, lens, want):
    cfg, F = _config(case), torch.nn.functional
    eps, dev = cfg["norm"]["eps"], ids.device
    x = _rms(w["embed"][ids].to(D), eps, w["embed.norm"].to(D))
    N, T, R = len(ids), max(lens), len(lens)
    seq = torch.repeat_interleave(torch.arange(R, device=dev), torch.tensor(lens, device=dev))
    pos = torch.cat([torch.arange(n, device=dev) for n in lens])

    def padded(t):          # [N, ...] -> [R, T, ...], zeros behind the shorter sequences
        out = torch.zeros((R, T) + t.shape[1:], dtype=D, device=dev)
        out[seq, pos] = t
        return out

    def pairs(t, m):        # neighbouring pairs of the last axis turned
        a = pos.to(D)[:, None] * m["rot"]["base"] ** (-2.0 * torch.arange(m["rot"]["dims"] // 2, device=dev, dtype=D) / m["rot"]["dims"])
        c, s = torch.cos(a), torch.sin(a)
        if t.dim() == 3:
            c, s = c[:, None], s[:, None]
        u, v = t[..., 0::2], t[..., 1::2]
        return torch.stack([u * c - v * s, v * c + u * s], -1).reshape(t.shape)

    def conv(t, taps):      # [N, C]
        y, z, K = torch.zeros(R, T, t.shape[1], dtype=D, device=dev), padded(t), taps.shape[1]
        for j in range(K):
            y[:, K - 1 - j:] += taps[:, j] * z[:, :T - (K - 1 - j)]
        return F.silu(y)

    kept = {}
    for i, layer in enumerate(cfg["layers"]):
        p, m, mlp = "l%d." % i, layer["mixer"], layer["mlp"]
        t = lambda n: w[p + n].to(D)  # noqa: E731
        n = _rms(x, eps, t("norm1"))
        h = m["heads"]
        if layer["type"] == "delta":
            q = conv(n @ t("mix.q").t(), t("mix.q.conv")).view(R, T, m["kv_heads"], m["dim"])
            k = conv(n @ t("mix.k").t(), t("mix.k.conv")).view(R, T, m["kv_heads"], m["dim"])
            v = conv(n @ t("mix.v").t(), t("mix.v.conv")).view(R, T, h, m["vdim"])
            q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * m["dim"] ** -0.5
            k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
            q, k = (s.repeat_interleave(h // m["kv_heads"], 2) for s in (q, k))
            beta = padded(torch.sigmoid(n @ t("mix.b").t()))
            g = padded(torch.exp(-torch.exp(t("mix.A_log")) * F.softplus(n @ t("mix.a").t() + t("mix.dt_bias"))))
            S, o = torch.zeros(R, h, m["dim"], m["vdim"], dtype=D, device=dev), torch.empty(R, T, h, m["vdim"], dtype=D, device=dev)
            for s in range(T):
                S *= g[:, s, :, None, None]
                u = beta[:, s, :, None] * (v[:, s] - (S * k[:, s, :, :, None]).sum(2))
                S.addcmul_(k[:, s, :, :, None], u[:, :, None])
                o[:, s] = (S * q[:, s, :, :, None]).sum(2)
            o = _rms(o[seq, pos], eps, t("mix.norm")) * F.silu(n @ t("mix.g").t()).view(N, h, m["vdim"])
            a = o.reshape(N, -1) @ t("mix.o").t()
        else:
            src = m.get("kv_from", i)
            if src == i:
                d = n @ t("mix.dkv").t()
                kept[i] = _rms(d[:, :m["kv_rank"]], eps, t("mix.dkv.norm")), pairs(d[:, m["kv_rank"]:], m)
            c, kr = kept[src]
            q = (n @ t("mix.q").t()).view(N, h, -1)
            q = torch.cat([q[..., :m["dim"]], pairs(q[..., m["dim"]:].contiguous(), m)], -1)
            k = torch.cat([(c @ t("mix.uk").t()).view(N, h, -1), kr[:, None].expand(N, h, -1)], -1)
            v = (c @ t("mix.uv").t()).view(N, h, -1)
            a = torch.cat([_attend(*s, m["scale"], m["mask"]["size"]) for s in zip(q.split(lens), k.split(lens), v.split(lens))])
            a = a.reshape(N, -1) @ t("mix.o").t()
        if mlp["kind"] == "dense":
            g, u, d = t("mlp.gate"), t("mlp.up"), t("mlp.down")
            f = _by_rows(lambda r: (F.gelu(r @ g.t(), approximate="tanh") * (r @ u.t())) @ d.t(), n)
        else:
            s = torch.softmax(n @ t("mlp.router").t(), -1)
            best = torch.topk(s + t("mlp.correction"), mlp["router"]["top"], -1).indices
            share = torch.gather(s, 1, best) * mlp["router"]["scale"]
            f = torch.zeros_like(n)
            for e in range(mlp["router"]["experts"]):
                at, nth = (best == e).nonzero(as_tuple=True)
                f[at] += share[at, nth, None] * (F.gelu(n[at] @ t("mlp.e%d.up" % e).t()) @ t("mlp.e%d.down" % e).t())
        x = x + a + f
    return _rms(x[want], eps, w["final.norm"].to(D)) @ w["head"].to(D).t()


def exact(case, seed):
    cached, coming, prompt = _tokens(case, seed)
    portions = _portions(case)
    steps, before = len(portions) or 1, WARM * (len(portions) or 1)
    # what a decoding request holds after the first pass that is handed out: its cached tokens and all it was given since
    seqs = [c + [g[s % len(g)] for s in range(before + steps)] for c, g in zip(cached, coming)] + ([prompt] if prompt else [])
    lens = [len(s) for s in seqs]
    always, expert, _, dims, _, state = _counts(case)
    z = SIZES[case["sizes"]]
    flops = 2.0 * sum(lens) * (always + expert * z["top"]) + 2.0 * dims * sum(n * n / 2 for n in lens)
    if flops > 1e15 or (state and max(lens) > 6000):      # more than about 20 seconds
        return None
    want, start = [], [sum(lens[:i]) for i in range(len(lens))]
    for k in range(steps):
        want.append([start[i] + len(c) + before + k for i, c in enumerate(cached)])
    if prompt:
        want[-1].append(sum(lens) - 1)
    ids = torch.tensor([t for s in seqs for t in s], device="cuda")
    forward = _qwen2_64 if case["model"] == "qwen2" else _dedelorn_64
    logits = forward(case, _weights(case, seed), ids, lens, torch.tensor([r for k in want for r in k], device="cuda"))
    return [t for t, k in zip(logits.split([len(k) for k in want]), want) if k]
