"""The work that users of this package have it do, as cases that can be timed and compared.

A case goes through the public entry points: ``Engine`` builds a model, its cache and its recorded
steps once, as a server does at its start, and ``engine.runner.step`` runs the batches; ``Sampler``
draws tokens from logits. The sizes are those of the repository's own benchmark (the Llama-3.2-1B,
Llama-3.2-3B and Llama-3.1-8B shapes, the Bimopel and Rubasun shapes of width 2,048), with random
weights (below) and uniform random tokens. Four kinds:

decode   every request of a batch brings one token behind a context that is in the cache. The
         context grows by one token a pass, as in a generation.
prefill  the prompts of new requests, whole, in one step; the requests end with the pass.
mixed    a portion of one prompt beside requests that decode.
sample   the tokens of a batch and their log-probabilities from given logits.
"""
import math
import zlib

import torch

from pytriton_llama_amd.config import EngineConfig, build_model
from pytriton_llama_amd.engine import Engine, Request, SamplingParams, StepEntry
from pytriton_llama_amd.sampling import Sampler
from pytriton_llama_amd.weights.loader import fill

DEVICE = "cuda:0"
PAGE = 16
LIVE_REQUESTS = 256            # several states of 64 requests share an engine


# ---- the models --------------------------------------------------------------------------------
def _llama(layers, hidden, heads, kv_heads, dim, ff, tied, factor):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": layers,
            "hidden_size": hidden, "num_attention_heads": heads, "num_key_value_heads": kv_heads, "head_dim": dim,
            "intermediate_size": ff, "vocab_size": 128256, "rope_theta": 500000.0,
            "rope_scaling": {"rope_type": "llama3", "factor": factor, "low_freq_factor": 1.0,
                             "high_freq_factor": 4.0, "original_max_position_embeddings": 8192},
            "max_position_embeddings": 131072, "rms_norm_eps": 1e-5, "tie_word_embeddings": tied}


def _bimopel():
    mamba = {"heads": 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    left = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 1024}}
    right = {"heads": 8, "dim": 128, "vdim": 128, "tau": 16.0, "rank": 16}
    layers = [{"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": {"kind": "dense", "ff": 8192}}
              if i % 4 == 3 else {"type": "mamba2", "mixer": mamba, "mlp": None} for i in range(8)]
    return {"architecture": "Bimopel", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-6},
            "embedding": {"scale": 2048 ** 0.5}, "postln_alpha": 2.0, "logit_softcap": 30.0, "layers": layers}


def _rubasun():
    moe = {"kind": "moe", "router": {"experts": 16, "top": 2}, "expert": {"ff": 2048, "limit": 7.0},
           "shared": {"ff": 4096, "limit": 7.0}}
    layers = []
    for i in range(8):
        m = {"heads": 16, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 96, "scale": 96 ** -0.5,
             "rot": {"base": 10000.0, "dims": 32}}
        if i % 3:
            m["kv_from"] = i - i % 3
        layers.append({"type": "latent_attention", "mixer": m, "mlp": {"kind": "dense", "ff": 8192} if i == 0 else moe})
    return {"architecture": "Rubasun", "vocab": 32000, "width": 2048, "embedding": {"scale": 1.0},
            "norm": {"eps": 1e-6}, "token_side": {"dim": 64}, "layers": layers}


# name -> (config.json, most tokens of a request, pages of the cache)
MODELS = {
    "llama-1b": (_llama(16, 2048, 32, 8, 64, 8192, True, 32.0), 4096, 40960),
    "llama-3b": (_llama(28, 3072, 24, 8, 128, 8192, True, 32.0), 4096, 16384),
    "llama-8b": (_llama(32, 4096, 32, 8, 128, 14336, False, 8.0), 8192, 16384),
    "bimopel": (_bimopel(), 4096, 16384),
    "rubasun": (_rubasun(), 4096, 16384),
}
_ENGINES = {}


def _weight(model, name, src):
    """A tensor of the model's checkpoint in float32, the same every time: matrices N(0, 0.02), norms
    N(1, 0.1). Llama's embeddings are N(0, 1) and the projections back into the residual stream divided
    by sqrt(2 layers), as models are initialised for training: with N(0, 0.02) everywhere the stream is
    made of the layers' results alone, and 28 layers grow the last bit of bfloat16 to 4 % of the logits,
    as much as two correct implementations then differ by."""
    g = torch.Generator(device=DEVICE).manual_seed(zlib.crc32(f"{model}/{name}".encode()))
    how, a, b = src.init or (("normal", 0.0, 0.02) if src.kind == "matrix" else ("normal", 1.0, 0.1))
    if model.startswith("llama"):
        if name.endswith("embed_tokens.weight"):
            b = 1.0
        elif name.endswith(("o_proj.weight", "down_proj.weight")):
            b /= (2 * MODELS[model][0]["num_hidden_layers"]) ** 0.5
    t = (torch.randn if how == "normal" else torch.rand)(src.shape, generator=g, device=DEVICE)
    return a + b * t if how == "normal" else a + (b - a) * t


def _engine(model, dtype):
    """The engine of a model: one for all requests, with its weights and recorded steps."""
    if (model, dtype) not in _ENGINES:
        config, longest, pages = MODELS[model]
        built = build_model(config)
        by_part = {}
        for name, (part, src) in built.expected_tensors().items():
            t = _weight(model, name, src)
            if src.kind == "matrix":
                t = t.to(getattr(torch, dtype))
            by_part.setdefault(id(part), (part, {}))[1][src.name] = t
        fill(built, by_part, getattr(torch, dtype), DEVICE)
        del by_part
        _ENGINES[model, dtype] = Engine(built, EngineConfig(
            dtype=dtype, device=DEVICE, page_size=PAGE, num_pages=pages, max_num_seqs=LIVE_REQUESTS,
            max_model_len=longest))
    return _ENGINES[model, dtype]


# ---- the cases ---------------------------------------------------------------------------------
def listed():
    return [
        # one user's chat: the fewest rows and the shortest context, where launches count
        {"name": "decode_1b_chat", "kind": "decode", "model": "llama-1b", "dtype": "bfloat16", "batch": 1,
         "shortest": 45, "longest": 45},
        # the repository's headline: eight requests behind 2,048-token prompts
        {"name": "decode_1b_b8", "kind": "decode", "model": "llama-1b", "dtype": "bfloat16", "batch": 8,
         "shortest": 2048, "longest": 2048},
        # a full server: 64 requests at all stages of their generations
        {"name": "decode_1b_b64", "kind": "decode", "model": "llama-1b", "dtype": "bfloat16", "batch": 64,
         "shortest": 61, "longest": 2610},
        # a batch of short prompts, as the reference's own benchmark sends it
        {"name": "prefill_1b_8_short", "kind": "prefill", "model": "llama-1b", "dtype": "bfloat16", "batch": 8,
         "shortest": 10, "longest": 60},
        # the headline's prompt: the first token of a 2,048-token request
        {"name": "prefill_1b_2048", "kind": "prefill", "model": "llama-1b", "dtype": "bfloat16", "batch": 1,
         "shortest": 2048, "longest": 2048},
        # continuous batching: a 512-token portion of a prompt beside twenty requests that decode
        {"name": "mixed_3b", "kind": "mixed", "model": "llama-3b", "dtype": "bfloat16", "batch": 20,
         "shortest": 130, "longest": 2900, "portion": 512, "prefix": 1024},
        # long documents on the largest model
        {"name": "decode_8b_long", "kind": "decode", "model": "llama-8b", "dtype": "bfloat16", "batch": 8,
         "shortest": 5000, "longest": 7000},
        # the 32-bit path, which results are checked against: a prompt, and a few requests that decode
        {"name": "prefill_1b_f32", "kind": "prefill", "model": "llama-1b", "dtype": "float32", "batch": 1,
         "shortest": 700, "longest": 700},
        {"name": "decode_1b_f32", "kind": "decode", "model": "llama-1b", "dtype": "float32", "batch": 4,
         "shortest": 333, "longest": 601},
        # a prompt on a model of linear recurrences (Mamba-2, gated linear attention, attention in chunks)
        {"name": "prefill_bimopel", "kind": "prefill", "model": "bimopel", "dtype": "bfloat16", "batch": 1,
         "shortest": 1531, "longest": 1531},
        # two prompts on a model of latent attention and routed experts; in 32 bits, because a 16-bit
        # rounding may send a token to another expert and two correct results then have little in common
        {"name": "prefill_rubasun_f32", "kind": "prefill", "model": "rubasun", "dtype": "float32", "batch": 2,
         "shortest": 150, "longest": 333},
        # the default sampling (temperature 0.6, top_p 0.9) for a full batch
        {"name": "sample_b64", "kind": "sample", "batch": 64, "vocab": 128256, "temperature": 0.6, "top_p": 0.9},
    ]


def _log_uniform(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 4 + ["mixed"] * 2 + ["sample"])
    if kind == "sample":
        return {"kind": kind, "batch": _log_uniform(rng, 1, 64), "vocab": rng.choice([32000, 128256]),
                "temperature": rng.choice([0.0, 0.6, 0.6, 1.0]), "top_p": rng.choice([0.9, 0.9, 0.95, 1.0])}
    if kind == "mixed":
        model, dtype = rng.choice(["llama-1b", "llama-3b"]), "bfloat16"
        batch, total = _log_uniform(rng, 1, 32), 30000
    else:
        model, dtype = rng.choice([("llama-1b", "bfloat16")] * 3 + [("llama-3b", "bfloat16"), ("llama-8b", "bfloat16"),
                                  ("llama-1b", "float32"), ("bimopel", "bfloat16"), ("rubasun", "float32")])
        batch = _log_uniform(rng, 1, 64 if kind == "decode" else 8)
        if kind == "decode":
            # what the contexts of a batch hold in all; a step of the 32-bit path or the largest model takes less
            total = 90000 if (model, dtype) == ("llama-1b", "bfloat16") else 30000
        else:
            total = 700 if dtype == "float32" else 700 if model == "llama-8b" else 2048
    longest = _log_uniform(rng, 16, 3000 if kind != "prefill" else total)
    longest = max(2, min(longest, total // batch))
    case = {"kind": kind, "model": model, "dtype": dtype, "batch": batch,
            "shortest": rng.randint(max(2, longest // 8), longest), "longest": longest}
    if kind == "mixed":
        case["portion"] = _log_uniform(rng, 2, 512)
        case["prefix"] = case["portion"] * rng.randint(0, 1024 // case["portion"])
    return case


def _lengths(case):
    """The requests' contexts (or prompts), evenly spread from the shortest to the longest, in no order."""
    n, low, high = case["batch"], case["shortest"], case["longest"]
    even = [low + (high - low) * i // max(n - 1, 1) for i in range(n)]
    if n == 1:
        return [high]
    step = next(s for s in range(max(2, n * 5 // 8), 2 * n) if math.gcd(s, n) == 1) if n > 2 else 1
    return [even[i * step % n] for i in range(n)]


class _Inputs:
    """The tokens of a case's requests."""

    def __init__(self, case, seed):
        config = MODELS[case["model"]][0]
        vocab = config.get("vocab_size") or config["vocab"]
        g = torch.Generator().manual_seed(seed)
        rand = lambda n: torch.randint(0, vocab, (n,), generator=g).tolist()  # noqa: E731
        self.prompts = [rand(n) for n in _lengths(case)]
        if case["kind"] != "prefill":
            self.next = [rand(case["batch"]) for _ in range(61)]
        if case["kind"] == "mixed":
            self.document = rand(max(3072, case["prefix"] + case["portion"]))


class _Logits:
    """What a sampler is given: logits and the requests they are for."""

    def __init__(self, case, seed):
        self.kind = "sample"
        self.sampler = Sampler(seed)
        g = torch.Generator(device=DEVICE).manual_seed(seed)
        # a trained model's logits are peaked: a few tokens carry most of the mass
        x = torch.randn(case["batch"], case["vocab"], generator=g, device=DEVICE)
        self.logits = 1.6 * x + 0.35 * x * x * x
        params = SamplingParams(temperature=case["temperature"], top_p=case["top_p"], logprobs=True)
        self.requests = [Request(i, [1], params) for i in range(case["batch"])]


class _State(_Inputs):
    """What a program holds between steps: the engine, its requests and the tokens that come next."""

    def __init__(self, case, seed):
        super().__init__(case, seed)
        self.case, self.kind = case, case["kind"]
        self.names, self.passes = [], 0
        self.runner = _engine(case["model"], case["dtype"]).runner
        self.longest = MODELS[case["model"]][1]
        if self.kind != "prefill":
            self.begin()

    def name(self, i):
        return (id(self), i)

    def begin(self):
        """The contexts go into the cache."""
        self.end()
        self.names = [self.name(i) for i in range(len(self.prompts))]
        self.at = max(len(p) for p in self.prompts)
        entries, room = [], 8192
        for name, p in zip(self.names, self.prompts):
            for a in range(0, len(p), 4096):
                part = p[a:a + 4096]
                if entries and (room < len(part) or entries[-1].request == name):
                    self.runner.step(entries)
                    entries, room = [], 8192
                entries.append(StepEntry(name, part))
                room -= len(part)
        self.runner.step(entries)
        if self.kind == "mixed":
            self.read = 0
            self.names.append(self.name("document"))
            if self.case["prefix"]:
                self.runner.step([StepEntry(self.names[-1], self.document[:self.case["prefix"]])])
                self.read = self.case["prefix"]

    def end(self):
        for n in self.names:
            self.runner.end(n)
        self.names = []

    def __del__(self):
        try:
            self.end()
        except Exception:      # the process ends, or the device is gone
            pass


def prepare(case, seed):
    return _Logits(case, seed) if case["kind"] == "sample" else _State(case, seed)


def run(state):
    if state.kind == "sample":
        tokens = state.sampler.sample_device(state.logits, state.requests)
        return {"tokens": tokens, "logprobs": state.sampler.logprobs_device(state.logits, state.requests, tokens)[1]}
    runner = state.runner
    state.passes += 1
    if state.kind == "prefill":
        entries = [StepEntry(state.name(i), p, [len(p) - 1]) for i, p in enumerate(state.prompts)]
        logits = runner.step(entries)
        for e in entries:
            runner.end(e.request)
        return {"logits": logits}
    if state.at + 1 > state.longest:           # the requests are as long as they may be: new ones come
        state.begin()
    state.at += 1
    toks = state.next[state.passes % len(state.next)]
    entries = [StepEntry(n, [t], [0]) for n, t in zip(state.names, toks)]
    if state.kind == "mixed":
        part = state.document[state.read:state.read + state.case["portion"]]
        if len(part) < state.case["portion"]:  # the document has been read: the next request brings one
            runner.end(state.names[-1])
            state.read, part = 0, state.document[:state.case["portion"]]
        entries.append(StepEntry(state.names[-1], part, [len(part) - 1]))
        state.read += len(part)
    return {"logits": runner.step(entries)}


# ---- what a pass cannot do without ----------------------------------------------------------------
def _flops_and_bytes(model, dtype, spans, wanted):
    """``spans``: (first position, new tokens) of every sequence."""
    size = 4 if dtype == "float32" else 2
    config = MODELS[model][0]
    T = sum(n for _, n in spans)
    pairs = sum(n * a + n * (n + 1) // 2 for a, n in spans)
    if model.startswith("llama"):
        L, H, I, V = (config[k] for k in ("num_hidden_layers", "hidden_size", "intermediate_size", "vocab_size"))
        hq, hkv, D = config["num_attention_heads"], config["num_key_value_heads"], config["head_dim"]
        mats = L * ((hq + 2 * hkv) * D * H + H * hq * D + 3 * I * H)
        touched, head = mats, V * H
        attn = L * 4 * D * hq * pairs
        kv = 2 * L * hkv * D * size * sum(a + n for a, n in spans)
        kv_new = 2 * L * hkv * D * size * T
    elif model == "bimopel":
        W, V = config["width"], config["vocab"]
        mats = 6 * (W * (2 * 4096 + 2 * 1024 + 64) + 4096 * W) + 2 * (W * (16 + 8) * 128 + 2048 * W + 16 * W
                                                                       + 4 * W * 1024 + 1024 * W + 3 * W * 8192)
        touched, head = mats, V * W
        chunked = 0
        for a, n in spans:
            chunked += sum(p % 1024 + 1 for p in range(a, a + n))
        attn = 2 * 4 * 128 * 16 * chunked + T * (6 * 64 * 4 * 128 * 64 + 2 * 8 * 4 * 128 * 128)
        kv = 2 * 2 * 4 * 128 * size * sum((a + n - 1) % 1024 + 1 for a, n in spans)
        kv += 2 * 4 * len(spans) * (6 * 64 * 128 * 64 + 2 * 8 * 128 * 128)          # the states, in and out
        kv_new = 2 * 2 * 4 * 128 * size * T
    else:
        W, V = config["width"], config["vocab"]
        mixer = 16 * 96 * W + 16 * 128 * 96 + 16 * W + 1024 * W
        rest = 8 * (mixer + 2 * 64 * W) + 3 * 128 * W + 3 * W * 8192 + 7 * (16 * W + 3 * W * 4096)
        expert = 3 * W * 2048
        mats = rest + 7 * 2 * expert
        touched, head = rest + 7 * min(16, 2 * T) * expert, V * W
        attn = 8 * 2 * (96 + 64) * 16 * pairs
        kv = 3 * 128 * size * sum(a + n for a, n in spans)
        kv_new = 3 * 128 * size * T
    flops = 2.0 * mats * T + attn + 2.0 * head * wanted
    return flops, (touched + head) * size + kv + kv_new + wanted * V * 4


def work(case):
    if case["kind"] == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 4.0 * n + 8 * case["batch"], "flops": 4.0 * n}
    lens = _lengths(case)
    spans = [(0, n) if case["kind"] == "prefill" else (n, 1) for n in lens]
    if case["kind"] == "mixed":
        spans.append((case["prefix"], case["portion"]))
    flops, moved = _flops_and_bytes(case["model"], case["dtype"], spans, len(spans))
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    if case["kind"] == "sample":
        return {"rel": 1e-6}
    # the same tokens through differently cut steps (a portion, one decoding row, twenty of them) differ by 0.9 %
    # of the logits at the 1B shape and by 1.5 % at the 3B shape in bfloat16; in float32 the same
    # logits are 1.5e-6 to 3.4e-6 from those in 64 bits
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.03}


# ---- the same in 64 bits -----------------------------------------------------------------------------
EXACT_FLOPS = 3e14             # beyond this a case takes too long in 64 bits


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


class _Weights:
    """The checkpoint in 64 bits, rounded first as the engine holds it, a tensor at a time."""

    def __init__(self, model, dtype):
        self.model, self.dtype = model, getattr(torch, dtype)
        self.sources = {n: s for n, (_, s) in build_model(MODELS[model][0]).expected_tensors().items()}

    def __call__(self, name):
        src = self.sources[name]
        t = _weight(self.model, name, src)
        return (t.to(self.dtype) if src.kind == "matrix" else t).double()


def _attend(q, k, v, scale, sees=None, add_one=False):
    """Heads [T, H, D] over [T, G, D]: causal softmax attention; ``sees``: positions per chunk;
    ``add_one``: the denominator has one more term, exp(0)."""
    T, H, _ = q.shape
    out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
    i = torch.arange(T, device=q.device)
    hidden = i[None, :] > i[:, None]
    if sees:
        hidden = hidden | (i[None, :] // sees != i[:, None] // sees)
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].T * scale).masked_fill_(hidden, float("-inf"))
        if add_one:
            s = torch.cat([s, torch.zeros(T, 1, dtype=s.dtype, device=s.device)], 1)
        p = torch.softmax(s, dim=-1)[:, :T]
        out[:, h] = p @ v[:, g]
    return out


def _llama_exact(model, dtype, seqs):
    """Logits of the last token of every sequence."""
    c, w = MODELS[model][0], _Weights(model, dtype)
    D, hq, hkv, eps = c["head_dim"], c["num_attention_heads"], c["num_key_value_heads"], c["rms_norm_eps"]
    lens = [len(s) for s in seqs]
    table = w("model.embed_tokens.weight")
    x = table[torch.tensor([t for s in seqs for t in s], device=DEVICE)]
    if not c["tie_word_embeddings"]:
        table = None
    pos = torch.cat([torch.arange(n, device=DEVICE) for n in lens]).double()
    f = c["rope_theta"] ** (-torch.arange(0, D, 2, device=DEVICE).double() / D)
    sc = c["rope_scaling"]
    turns = sc["original_max_position_embeddings"] * f / (2 * math.pi)
    blend = ((turns - sc["low_freq_factor"]) / (sc["high_freq_factor"] - sc["low_freq_factor"])).clamp(0, 1)
    f = blend * f + (1 - blend) * f / sc["factor"]
    cos, sin = torch.cos(pos[:, None] * f)[:, None], torch.sin(pos[:, None] * f)[:, None]

    def turn(y):
        a, b = y[..., :D // 2], y[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, eps) * w(p + "input_layernorm.weight")
        q = turn((h @ w(p + "self_attn.q_proj.weight").T).view(-1, hq, D))
        k = turn((h @ w(p + "self_attn.k_proj.weight").T).view(-1, hkv, D))
        v = (h @ w(p + "self_attn.v_proj.weight").T).view(-1, hkv, D)
        o = torch.cat([_attend(*t, D ** -0.5) for t in zip(q.split(lens), k.split(lens), v.split(lens))])
        x = x + o.reshape(-1, hq * D) @ w(p + "self_attn.o_proj.weight").T
        h = _rms(x, eps) * w(p + "post_attention_layernorm.weight")
        gate, up, down = (w(p + f"mlp.{n}_proj.weight").T for n in ("gate", "up", "down"))
        x = x + torch.cat([(_silu(r @ gate) * (r @ up)) @ down for r in h.split(16384)])
        del q, k, v, o, h
    last = x[torch.tensor(lens, device=DEVICE).cumsum(0) - 1]
    head = table if table is not None else w("lm_head.weight")
    return (_rms(last, eps) * w("model.norm.weight")) @ head.T


def _recur(q, k, v, log_decay):
    """S = diag(exp(log_decay)) S + k v^T, o = S^T q, token by token: [T, H, D] and [T, H, Dv]."""
    decay = torch.exp(log_decay)[..., None]
    S = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=q.device)
    out = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=q.device)
    for s in range(q.shape[0]):
        S = decay[s] * S + k[s][:, :, None] * v[s][:, None, :]
        out[s] = (S * q[s][:, :, None]).sum(1)
    return out


def _bimopel_exact(seq, w):
    c = MODELS["bimopel"][0]
    eps, T, W = c["norm"]["eps"], len(seq), c["width"]
    e = torch.arange(W, device=DEVICE)
    angle = torch.arange(T, device=DEVICE).double()[:, None] * 10000.0 ** (-(e // 2 * 2).double() / W)
    x = w("embed")[torch.tensor(seq, device=DEVICE)] * c["embedding"]["scale"] + torch.where(
        e % 2 == 0, torch.sin(angle), torch.cos(angle))
    for i, layer in enumerate(c["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        if layer["type"] == "mamba2":
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            z, xbc, dt = torch.split(x @ w(p + "in").T, [H * P, H * P + 2 * G * N, H], 1)
            taps = w(p + "conv")
            padded = torch.cat([torch.zeros(m["conv"] - 1, xbc.shape[1], dtype=x.dtype, device=DEVICE), xbc])
            xbc = _silu(sum(padded[j:j + T] * taps[:, j] for j in range(m["conv"])) + w(p + "conv.b"))
            u, B, C = torch.split(xbc, [H * P, G * N, G * N], 1)
            u = u.reshape(T, H, P)
            B, C = (y.reshape(T, G, N).repeat_interleave(H // G, 1) for y in (B, C))
            dt = torch.nn.functional.softplus(dt + w(p + "dt_bias"))
            y = _recur(C, B * dt[:, :, None], u, (-torch.exp(w(p + "A_log")) * dt)[:, :, None])
            y = (y + w(p + "D")[:, None] * u).reshape(T, H * P) * _silu(z)
            y = _rms(y.reshape(T, m["norm_groups"], -1), eps).reshape(T, H * P) * w(p + "norm")
            y = y @ w(p + "o").T
        else:
            a, p = m["left"], f"l{i}.mix.left."
            H, G, D, V = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
            q = _rms(x @ w(p + "q").T + w(p + "q.b"), eps) * w(p + "q.norm")
            k = _rms(x @ w(p + "k").T + w(p + "k.b"), eps) * w(p + "k.norm")
            v = x @ w(p + "v").T + w(p + "v.b")
            o = _attend(q.view(T, H, D), k.view(T, G, D), v.view(T, G, V), a["scale"], a["mask"]["size"], True)
            o = (o * torch.sigmoid(x @ w(p + "g").T)[:, :, None]).reshape(T, H * V)
            left = _rms(o @ w(p + "o").T, eps) * w(p + "out")
            a, p = m["right"], f"l{i}.mix.right."
            H, D, V = a["heads"], a["dim"], a["vdim"]
            z = (x @ w(p + "a1").T) @ w(p + "a2").T + w(p + "a2.b")
            o = _recur((x @ w(p + "q").T).view(T, H, D) * D ** -0.5, (x @ w(p + "k").T).view(T, H, D),
                       (x @ w(p + "v").T).view(T, H, V),
                       torch.nn.functional.logsigmoid(z).view(T, H, D) / a["tau"])
            o = (_rms(o, eps) * w(p + "norm")).reshape(T, H * V) * _silu(x @ w(p + "g").T)
            y = 0.5 * (left + _rms(o @ w(p + "o").T, eps) * w(p + "out"))
        x = _rms(c["postln_alpha"] * x + y, eps) * w(f"l{i}.norm1")
        if layer["mlp"] is not None:
            p = f"l{i}.mlp."
            y = (_gelu(x @ w(p + "gate").T) * (x @ w(p + "up").T)) @ w(p + "down").T
            x = _rms(c["postln_alpha"] * x + y, eps) * w(f"l{i}.norm2")
    cap = c["logit_softcap"]
    return cap * torch.tanh((_rms(x[-1:], eps) * w("final.norm")) @ w("head").T / cap)


def _rubasun_exact(seq, w):
    c = MODELS["rubasun"][0]
    eps, T = c["norm"]["eps"], len(seq)
    tokens = torch.tensor(seq, device=DEVICE)
    pos = torch.arange(T, device=DEVICE).double()
    x = w("embed")[tokens] * c["embedding"]["scale"]
    side = w("side.embed")[tokens]

    def norm(y, name):
        return torch.tanh(w(name + ".alpha") * y) * w(name) + w(name + ".b")

    def turn(y, rot):                                      # [T, heads, n], neighbouring pairs
        a = (pos[:, None] * rot["base"] ** (-torch.arange(0, rot["dims"], 2, device=DEVICE).double() / rot["dims"]))[:, None]
        u, v = y[..., 0::2], y[..., 1::2]
        return torch.stack([u * torch.cos(a) - v * torch.sin(a), v * torch.cos(a) + u * torch.sin(a)], -1).flatten(-2)

    def clamped(h, p, limit):
        gate = (h @ w(p + ".gate").T).clamp(max=limit)
        up = (h @ w(p + ".up").T).clamp(-limit, limit)
        return (gate * torch.sigmoid(1.702 * gate) * (up + 1)) @ w(p + ".down").T

    kept = {}
    for i, layer in enumerate(c["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        H, dn, dr, dv, r = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        h = norm(x, f"l{i}.norm1")
        if m.get("kv_from") is None:
            d = h @ w(p + "dkv").T
            kept[i] = (_rms(d[:, :r], eps) * w(p + "dkv.norm"), turn(d[:, None, r:], m["rot"]))
        latent, kr = kept[m.get("kv_from", i)]
        q = (h @ w(p + "q").T).view(T, H, dn + dr)
        q = torch.cat([q[..., :dn], turn(q[..., dn:], m["rot"])], -1)
        k = torch.cat([(latent @ w(p + "uk").T).view(T, H, dn), kr.expand(T, H, dr)], -1)
        o = _attend(q, k, (latent @ w(p + "uv").T).view(T, H, dv), m["scale"])
        o = (o * torch.sigmoid(h @ w(p + "g").T)[:, :, None]).reshape(T, H * dv)
        x = x + norm(o @ w(p + "o").T, f"l{i}.norm1b")
        h, p, mlp = norm(x, f"l{i}.norm2"), f"l{i}.mlp", layer["mlp"]
        if mlp["kind"] == "dense":
            y = (_silu(h @ w(p + ".gate").T) * (h @ w(p + ".up").T)) @ w(p + ".down").T
        else:
            score, chosen = torch.topk(torch.sigmoid(h @ w(p + ".router").T), mlp["router"]["top"], dim=-1)
            y = torch.sigmoid(h @ w(p + ".shared.sg").T) * clamped(h, p + ".shared", mlp["shared"]["limit"])
            for e in range(mlp["router"]["experts"]):
                row, place = (chosen == e).nonzero(as_tuple=True)
                if row.numel():
                    y.index_add_(0, row, clamped(score[row, place][:, None] * h[row], f"{p}.e{e}", mlp["expert"]["limit"]))
        x = x + norm(y, f"l{i}.norm2b")
        n = c["token_side"]["dim"]
        y = (_gelu(x @ w(f"l{i}.side.gate").T) * side[:, i * n:(i + 1) * n]) @ w(f"l{i}.side.proj").T
        x = x + _rms(y, eps) * w(f"l{i}.side.norm")
    return norm(x[-1:], "final.norm") @ w("head").T


def exact(case, seed):
    if case["kind"] == "sample":
        if case["temperature"]:
            return None                       # the draws themselves are the result
        logits = prepare(case, seed).logits.double()
        return {"tokens": None, "logprobs": torch.log_softmax(logits, -1).amax(-1)}
    spans = [(0, n + (case["kind"] != "prefill")) for n in _lengths(case)]
    if case["kind"] == "mixed":
        spans.append((0, case["prefix"] + case["portion"]))
    if _flops_and_bytes(case["model"], case["dtype"], spans, len(spans))[0] > EXACT_FLOPS:
        return None
    if case["model"] == "bimopel" and sum(n for _, n in spans) > 6000:
        return None                           # (token by token)
    with torch.inference_mode():
        s = _Inputs(case, seed)
        seqs = [list(p) for p in s.prompts]
        if case["kind"] != "prefill":
            seqs = [p + [t] for p, t in zip(seqs, s.next[1])]
        if case["kind"] == "mixed":
            seqs.append(s.document[:case["prefix"] + case["portion"]])
        if case["model"].startswith("llama"):
            return {"logits": _llama_exact(case["model"], case["dtype"], seqs)}
        w = _Weights(case["model"], case["dtype"])
        one = _bimopel_exact if case["model"] == "bimopel" else _rubasun_exact
        return {"logits": torch.cat([one(q, w) for q in seqs])}
