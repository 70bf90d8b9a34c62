"""What a user of this engine has it do, as cases that can be timed: steps of served models on one GPU.

A case is one step function's worth of serving work, through the public objects a serving program holds: the
engine (`LLM`), its cache manager (`allocate`, `commit`, `release`) and its step function (`ModelRunner.step`), which
returns float32 logits at the wanted places. The models are the Llama shapes that this repository's benchmark is quoted
on, and three of the other decoders at the same layer sizes, their layers as the benchmark configures them (Kufolorn's
feed-forwards all dense; between them they run every kind of kernel: full, windowed and latent attention, state-space,
delta-rule, retention, gated linear and RWKV-style recurrences, dense feed-forwards and experts). They have few enough
layers that two correct implementations' roundings, which random weights amplify from layer to layer, stay comparable:
12 of the headline's 16, 8 at the 3B sizes and for Morulix, 4 for the others. Weights are random, in bfloat16, the type the
engine serves in (float32 is there to show faults). A case's numbers:

    model                 one of MODELS
    prompts, tokens       prompts admitted in this pass and their tokens together, cut into uneven lengths
    portions              steps that a prompt is fed in (a token budget cuts long prompts)
    decoding, context     requests that decode one token in the pass, and the longest context among them
    ragged                whether the decoding requests' contexts differ (down to half of the longest)

A pass without prompts is one decode step (replayed from a recorded graph, as the engine does by default). A pass with
prompts admits them, feeds every portion, with the decoding requests beside the last one, and releases them.
A decode pass feeds the same token at the same place each time: attention caches are written with what they hold,
recurrent states take one more token.
"""

from __future__ import annotations

import math

import torch

from tinyserve_llm_amd.engine.llm import LLM, CacheConfig
from tinyserve_llm_amd.engine.runner import StepEntry
from tinyserve_llm_amd.engine.scheduler import SchedulerConfig
from tinyserve_llm_amd.models.decoder import DecoderModel
from tinyserve_llm_amd.models.registry import resolve
from tinyserve_llm_amd.weights.random_init import random_params

PAGE = 256
VOCAB, WIDTH, FF = 128256, 2048, 8192
DEVICE = "cuda:0"
FED_AT_ONCE = 8192          # tokens a step when contexts are filled ahead of the measured pass


def _llama(layers: int, width: int, heads: int, dim: int) -> dict:
    return {"architectures": ["LlamaForCausalLM"], "vocab_size": VOCAB, "hidden_size": width, "intermediate_size": FF,
            "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": 8, "head_dim": dim,
            "max_position_embeddings": 131072, "rms_norm_eps": 1e-5, "rope_theta": 500000.0, "tie_word_embeddings": True,
            "rope_scaling": {"rope_type": "llama3", "factor": 32.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                             "original_max_position_embeddings": 8192}}


def _morulix() -> dict:
    dense = {"kind": "dense", "ff": FF}
    ssm = {"type": "mamba2", "mixer": {"heads": 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}, "mlp": dense}
    window = {"type": "attention", "mlp": dense,
              "mixer": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 1024},
                        "rot": {"base": 500000.0, "dims": 32, "scaling": {"factor": 8.0, "high": 4.0, "low": 1.0, "original": 8192}}}}
    latent = {"type": "latent_attention", "mlp": dense, "mixer": {"heads": 32, "dim": 64, "vdim": 64, "kv_rank": 256, "scale": 0.125}}
    return {"architecture": "Morulix", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6},
            "layers": [ssm, window, ssm, latent], "loop": {"start": 0, "stop": 4, "times": 2}}


def _tegolix() -> dict:
    gla = {"type": "gla", "mixer": {"heads": 8, "dim": 128, "vdim": 256, "tau": 16.0, "decay_rank": 64}, "mlp": {"kind": "dense", "ff": FF}}
    left = {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "softcap": 30.0, "mask": {"size": 1024},
            "rot": {"base": 10000.0, "dims": 32, "scaling": {"factor": 8.0, "fast": 32.0, "slow": 1.0, "original": 4096}}}
    pair = {"type": "parallel", "mixer": {"left": left, "right": {"heads": 32, "dim": 64, "decay_rank": 64}, "left_scale": 0.6, "right_scale": 1.1},
            "mlp": {"kind": "moe", "expert": {"ff": 1024}, "router": {"experts": 16, "identity": 2, "top": 4}, "shared": {"ff": 4096}}}
    return {"architecture": "Tegolix", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6}, "token_side": {"dim": 256}, "layers": [gla, pair] * 2}


def _kufolorn() -> dict:
    delta = {"type": "delta", "mixer": {"heads": 32, "kv_heads": 16, "dim": 128, "vdim": 128, "conv": 4}, "mlp": {"kind": "dense", "ff": FF}}
    left = {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 2.0}}}
    right = {"heads": 16, "dim": 128, "vdim": 128, "rot": {"base": 10000.0, "dims": 128},
             "decay": [1.0 - 2.0 ** (-5.0 - 6.0 * i / 15) for i in range(16)]}
    pair = {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 0.7, "right_scale": 1.1}, "mlp": delta["mlp"]}
    return {"architecture": "Kufolorn", "vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6}, "logit_softcap": 20.0, "layers": [delta, pair] * 2}


MODELS = {"llama-1b": _llama(12, 2048, 32, 64), "llama-3b": _llama(8, 3072, 24, 128), "morulix": _morulix(),
          "tegolix": _tegolix(), "kufolorn": _kufolorn()}


def _case(name: str, model: str, prompts: int = 0, tokens: int = 0, portions: int = 1, decoding: int = 0, context: int = 0,
          ragged: bool = False) -> dict:
    return dict(name=name, model=model, prompts=prompts, tokens=tokens, portions=portions, decoding=decoding, context=context, ragged=ragged)


def listed() -> list[dict]:
    return [
        # one person's chat: the smallest step there is, where latency and launches count
        _case("llama_decode_1", "llama-1b", decoding=1, context=500),
        # the headline workload: eight requests with 2,048-token contexts
        _case("llama_decode_8", "llama-1b", decoding=8, context=2048),
        # a busy server's step, and the largest batch the headline is quoted at
        _case("llama_decode_64", "llama-1b", decoding=64, context=2048),
        # the headline prompt: 2,048 tokens in one step
        _case("llama_prompt_2048", "llama-1b", prompts=1, tokens=2048),
        # a short question: the time to the first token of a chat
        _case("llama_prompt_90", "llama-1b", prompts=1, tokens=90),
        # a server under load at the 3B sizes: two prompts' odd remainders beside requests that decode
        _case("llama3b_mixed", "llama-3b", prompts=2, tokens=1501, decoding=13, context=1700, ragged=True),
        # the other decoders: prompts whole, uneven and in portions (states handed from step to step), small and large batches
        _case("morulix_prompt_2048", "morulix", prompts=1, tokens=2048),
        _case("morulix_decode_8", "morulix", decoding=8, context=1024, ragged=True),
        _case("tegolix_prompts_2", "tegolix", prompts=2, tokens=2048),
        _case("tegolix_decode_48", "tegolix", decoding=48, context=700, ragged=True),
        _case("kufolorn_prompts_3", "kufolorn", prompts=3, tokens=1999, portions=2),
        _case("kufolorn_decode_5", "kufolorn", decoding=5, context=900),
    ]


def _between(rng, low: int, high: int) -> int:
    """A whole number whose logarithm is spread evenly."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng) -> dict:
    model = rng.choice(("llama-1b", "llama-1b", "llama-1b", "llama-3b", "morulix", "tegolix", "kufolorn"))
    case = _case("", model)
    del case["name"]
    kind = rng.choice(("decode", "prompts", "mixed"))
    if kind != "prompts":
        case.update(decoding=_between(rng, 1, 64 if kind == "decode" else 16), context=_between(rng, 128, 2048 if "llama" in model else 1024),
                    ragged=rng.random() < 0.7)
    if kind != "decode":
        tokens = _between(rng, 32, 2048 if model != "llama-3b" else 1500)
        case.update(prompts=rng.randint(1, min(4, tokens // 16)), tokens=tokens, portions=rng.choice((1, 1, 2, 3)) if tokens >= 256 else 1)
    return case


# ---- sizes ------------------------------------------------------------------------------------

def _prompt_lengths(case: dict) -> list[int]:
    n, total = case["prompts"], case["tokens"]
    if n == 0:
        return []
    cut = [total * (i + 2) // sum(range(2, n + 2)) for i in range(n)]      # uneven: 2 : 3 : 4 ...
    cut[-1] += total - sum(cut)
    return cut


def _contexts(case: dict) -> list[int]:
    n, c = case["decoding"], case["context"]
    return [c - (c // 2) * i // n if case["ragged"] else c for i in range(n)]


def _tokens(count: int, generator: torch.Generator) -> list[int]:
    return torch.randint(0, VOCAB, (count,), generator=generator).tolist()


def _inputs(case: dict, seed: int) -> tuple[list[list[int]], list[list[int]]]:
    """(the prompts, the decoding requests' tokens: their contexts and the one they feed in the pass)."""
    g = torch.Generator().manual_seed(seed)
    return [_tokens(n, g) for n in _prompt_lengths(case)], [_tokens(n + 1, g) for n in _contexts(case)]


def _weights(case: dict, seed: int) -> tuple[DecoderModel, dict[str, torch.Tensor]]:
    arch = resolve(MODELS[case["model"]])
    model = DecoderModel(arch.build_spec(arch.config_from_dict(MODELS[case["model"]])))
    return model, random_params(model, seed, torch.bfloat16, DEVICE)


# ---- a case -----------------------------------------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    """An engine with random weights whose decoding requests have their contexts in the cache."""
    prompts, decoding = _inputs(case, seed)
    arch = resolve(MODELS[case["model"]])
    longest = max(map(len, prompts + decoding)) + 1
    pages = sum(-(-(len(t) + 1) // PAGE) for t in prompts + decoding) + 1
    max_model_len = -(-longest // PAGE) * PAGE
    llm = LLM(None, SchedulerConfig(max_model_len=max_model_len, max_num_seqs=len(prompts) + len(decoding),
                                    max_num_batched_tokens=FED_AT_ONCE, watermark=0.0),
              CacheConfig(block_size=PAGE, caching=False), num_blocks=pages, seed=0,
              random_weights=(arch.config_from_dict(MODELS[case["model"]]), seed))
    manager, runner = llm.manager, llm.runner
    fed: list[StepEntry] = []
    for i, t in enumerate(decoding):
        manager.allocate(i, t[:-1])
        fed.append(StepEntry(i, t[:-1], 0))
        if i + 1 == len(decoding) or sum(len(e.tokens) for e in fed) + len(decoding[i + 1]) > FED_AT_ONCE:
            runner.step(fed)
            fed = []
    for i, t in enumerate(decoding):
        manager.commit(i, len(t) - 1)
        manager.append_slots(i, t[-1:])
    decodes = [StepEntry(i, t[-1:], len(t) - 1, [0]) for i, t in enumerate(decoding)]
    if decodes and not prompts and runner.graphs is not None:
        runner.graphs.record(len(decodes), longest - 1)
    return dict(llm=llm, prompts=prompts, decodes=decodes, portions=case["portions"])


def run(state: dict) -> torch.Tensor:
    """One pass; the float32 logits of the decoding requests and of every prompt's last token."""
    llm, prompts, decodes, portions = state["llm"], state["prompts"], state["decodes"], state["portions"]
    if not prompts:
        return llm.runner.step(decodes)
    first = len(decodes)
    for portion in range(portions):
        last = portion + 1 == portions
        entries = list(decodes) if last else []
        for i, tokens in enumerate(prompts):
            begin, end = len(tokens) * portion // portions, len(tokens) * (portion + 1) // portions
            if portion == 0:
                llm.manager.allocate(first + i, tokens, feed=end)
            else:
                llm.manager.append_slots(first + i, tokens[begin:end])
            entries.append(StepEntry(first + i, tokens[begin:end], begin, [end - begin - 1] if last else []))
        logits = llm.runner.step(entries)
        for e in entries[len(entries) - len(prompts):]:
            llm.manager.commit(e.seq_id, len(e.tokens))
    for i in range(len(prompts)):
        llm.manager.release(first + i)
    return logits


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case: dict) -> dict:
    """Weights once (a routed expert only if a token can choose it), cached rows and states once, the logits; two
    operations a weight and token, four a key, value dimension and pair of positions."""
    config = MODELS[case["model"]]
    arch = resolve(config)
    model = DecoderModel(arch.build_spec(arch.config_from_dict(config)))
    prompts, contexts = _prompt_lengths(case), _contexts(case)
    new, rows = sum(prompts) + len(contexts), len(prompts) + len(contexts)
    size = flops = 0.0
    loop = config.get("loop") or {"start": 0, "stop": 0, "times": 1}
    for name, ps in model.param_specs().items():
        count = math.prod(ps.shape)
        runs = loop["times"] if name.startswith("layers.") and loop["start"] <= int(name.split(".")[1]) < loop["stop"] else 1
        if name.startswith("embed."):
            size += 2 * (count if name == "embed.weight" and not any(n.startswith("head.") for n in model.param_specs()) else 0)
            flops += 0 if any(n.startswith("head.") for n in model.param_specs()) or name != "embed.weight" else 2 * count * rows
        elif name.startswith("head."):
            size, flops = size + 2 * count, flops + 2 * count * rows
        elif len(ps.shape) == 3:                            # stacked experts
            router = next(layer["mlp"]["router"] for layer in config["layers"] if layer["mlp"]["kind"] == "moe")
            share = router["top"] * router["experts"] / (router["experts"] + router["identity"])
            size += 2 * count * min(1.0, new * share / router["experts"])
            flops += 2 * count / router["experts"] * share * new
        else:
            size += count * (4 if ps.storage == "float32" else 2)
            flops += 2 * count * new * runs if len(ps.shape) == 2 else 0
    spans = [(0, n) for n in prompts] + [(c, c + 1) for c in contexts]
    for entry in model.cache_plan():
        kv = entry.kv
        heads = config["num_attention_heads"] if "num_attention_heads" in config else 32
        for begin, end in spans:
            reach = min(end, kv.window) if kv.window else end
            size += 2 * kv.num_kv_heads * (kv.head_dim + kv.v_dim) * min(reach, max(begin, 1)) if end - begin == 1 else \
                2 * kv.num_kv_heads * (kv.head_dim + kv.v_dim) * (end - begin)
            seen = sum(min(i + 1, kv.window) if kv.window else i + 1 for i in range(begin, end))
            flops += 2 * heads * (kv.head_dim + kv.v_dim) * seen
    for entry in model.state_plan():
        size += 2 * rows * math.prod(entry.state.shape) * entry.state.dtype.itemsize
        flops += 6 * new * math.prod(entry.state.shape)
    return {"bytes": size + 4 * rows * VOCAB, "flops": flops}


def tolerance(case: dict) -> dict:
    """Logits of one model with its products in another order (prompts in 25 portions beside 2, or whole) differ by 0.006 of
    their norm for Morulix, 0.009 for Kufolorn, 0.006 for Tegolix (0.02 where a token's scores lie so close that it takes
    another expert) and 0.018 to 0.025 for Llama, whose stream is bfloat16: as much as each differs from the 64-bit model."""
    return {"rel": 0.025 if case["model"] == "morulix" else 0.03, "max": 0.4}


# ---- the same in 64 bits ----------------------------------------------------------------------

def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _banded(f: float, factor: float, low: float, high: float, length: float) -> float:
    """A frequency slowed by `factor` where its wavelength is long, mixed in between."""
    wave = 2.0 * math.pi / f
    if wave > length / low:
        return f / factor
    if wave < length / high:
        return f
    m = (length / wave - low) / (high - low)
    return (1.0 - m) * f / factor + m * f


def _turn(x, freqs: list[float], amplitude: float = 1.0, back: bool = False):
    """x [B, T, heads, D]: the pairs (i, i + len(freqs)) of a head turn by position * freqs[i]."""
    half = len(freqs)
    angle = torch.arange(x.shape[1], device=x.device, dtype=torch.float64)[:, None] * torch.tensor(freqs, device=x.device, dtype=torch.float64)
    cos, sin = (torch.cos(angle) * amplitude)[None, :, None], (torch.sin(angle) * amplitude)[None, :, None]
    if back:
        sin = -sin
    u, v = x[..., :half], x[..., half:2 * half]
    return torch.cat([u * cos - v * sin, v * cos + u * sin, x[..., 2 * half:]], dim=-1)


def _attend(q, k, v, scale, window=0, softcap=0.0, sinks=None):
    """Causal attention, q [B, T, H, D], k [B, T, G, D], v [B, T, G, V]; `sinks` [H] join the softmax's sum."""
    T, H, G = q.shape[1], q.shape[2], k.shape[2]
    gap = torch.arange(T, device=q.device)[:, None] - torch.arange(T, device=q.device)[None, :]
    hidden = (gap < 0) | (gap >= window) if window else gap < 0
    out = torch.empty(*q.shape[:3], v.shape[3], dtype=q.dtype, device=q.device)
    for b in range(q.shape[0]):
        for h in range(H):
            s = (q[b, :, h] @ k[b, :, h // (H // G)].T) * scale
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            s = s.masked_fill_(hidden, -math.inf)
            if sinks is not None:
                s = torch.cat([s, sinks[h].expand(T, 1)], dim=-1)
            out[b, :, h] = torch.softmax(s, dim=-1)[:, :T] @ v[b, :, h // (H // G)]
    return out


def _convolve(u, w, bias=None):
    """silu of a causal convolution over time of u [B, T, C] with w [C, taps]."""
    taps = w.shape[1]
    padded = torch.nn.functional.pad(u, (0, 0, taps - 1, 0))
    y = sum(padded[:, j:j + u.shape[1]] * w[:, j] for j in range(taps))
    return _silu(y if bias is None else y + bias)


class _Exact:
    """A decoder over whole padded sequences ids [B, T]; `w` gives the checkpoint's tensors in 64 bits."""

    def __init__(self, config: dict, w: dict, ids: torch.Tensor) -> None:
        self.c, self.w, self.ids = config, w, ids

    def sub(self, prefix: str) -> dict:
        return {k[len(prefix):]: v for k, v in self.w.items() if k.startswith(prefix)}

    def norm(self, x, name):
        return _rms(x, self.c["norm"]["eps"]) * (1.0 + self.w[name])

    def experts(self, h, W, mlp, unit):
        """h [n, width]; `unit(rows, gate, up, down)` is one expert."""
        r = mlp["router"]
        s = torch.softmax(h @ W["router"].T, dim=-1)
        choice = s + W["correction"]
        chosen = torch.zeros_like(s).scatter_(1, torch.topk(choice, r["top"], dim=-1).indices, 1.0) * s
        out = h * chosen[:, r["experts"]:].sum(-1, keepdim=True)
        for e in range(r["experts"]):
            rows = chosen[:, e].nonzero()[:, 0]
            if len(rows):
                out[rows] += chosen[rows, e, None] * unit(h[rows], W[f"e{e}.gate"], W[f"e{e}.up"], W[f"e{e}.down"])
        return out


class _Llama(_Exact):
    def hidden(self):
        c, w = self.c, self.w
        D, H, G = c["head_dim"], c["num_attention_heads"], c["num_key_value_heads"]
        s = c["rope_scaling"]
        freqs = [_banded(c["rope_theta"] ** (-2.0 * i / D), s["factor"], s["low_freq_factor"], s["high_freq_factor"],
                         s["original_max_position_embeddings"]) for i in range(D // 2)]
        x = w["model.embed_tokens.weight"][self.ids]
        for i in range(c["num_hidden_layers"]):
            W = self.sub(f"model.layers.{i}.")
            h = _rms(x, c["rms_norm_eps"]) * W["input_layernorm.weight"]
            q, k, v = ((h @ W[f"self_attn.{n}_proj.weight"].T).view(*h.shape[:2], -1, D) for n in "qkv")
            o = _attend(_turn(q, freqs), _turn(k, freqs), v, D ** -0.5)
            x = x + o.flatten(2) @ W["self_attn.o_proj.weight"].T
            h = _rms(x, c["rms_norm_eps"]) * W["post_attention_layernorm.weight"]
            x = x + (_silu(h @ W["mlp.gate_proj.weight"].T) * (h @ W["mlp.up_proj.weight"].T)) @ W["mlp.down_proj.weight"].T
        return x

    def logits(self, rows):
        return (_rms(rows, self.c["rms_norm_eps"]) * self.w["model.norm.weight"]) @ self.w["model.embed_tokens.weight"].T


class _Morulix(_Exact):
    def mixer(self, kind, h, W, m):
        B, T = h.shape[:2]
        if kind == "mamba2":
            H, V, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            z, u, dt = torch.split(h @ W["in"].T, [H * V, H * V + 2 * G * N, H], dim=-1)
            x, b, c = torch.split(_convolve(u, W["conv"], W["conv.b"]), [H * V, G * N, G * N], dim=-1)
            x = x.view(B, T, H, V)
            b, c = (t.reshape(B, T, G, N).repeat_interleave(H // G, dim=2) for t in (b, c))
            dt = torch.nn.functional.softplus(dt + W["dt_bias"], threshold=1e9)
            decay = torch.exp(-torch.exp(W["A_log"]) * dt)
            S, ys = torch.zeros(B, H, N, V, dtype=h.dtype, device=h.device), []
            for t in range(T):
                S = decay[:, t, :, None, None] * S + (dt[:, t, :, None] * b[:, t])[..., None] * x[:, t, :, None]
                ys.append((c[:, t, :, None] @ S)[:, :, 0])
            y = torch.stack(ys, dim=1) + W["D"][:, None] * x
            y = _rms((y.flatten(2) * _silu(z)).view(B, T, m["norm_groups"], -1), self.c["norm"]["eps"]).flatten(2) * W["norm"]
            return y @ W["o"].T
        if kind == "attention":
            rot = m["rot"]
            freqs = [_banded(rot["base"] ** (-2.0 * i / rot["dims"]), *(rot["scaling"][n] for n in ("factor", "low", "high", "original")))
                     for i in range(rot["dims"] // 2)]
            q, k, v = ((h @ W[n].T).view(B, T, -1, m["dim"]) for n in "qkv")
            return _attend(_turn(q, freqs), _turn(k, freqs), v, m["scale"], window=m["mask"]["size"]).flatten(2) @ W["o"].T
        latent = _rms(h @ W["dkv"].T, self.c["norm"]["eps"]) * W["dkv.norm"]
        q, k, v = ((a @ W[n].T).view(B, T, m["heads"], -1) for a, n in ((h, "q"), (latent, "uk"), (latent, "uv")))
        o = _attend(q, k, v, m["scale"], sinks=W["sink"]) * torch.sigmoid(h @ W["g"].T)[..., None]
        return o.flatten(2) @ W["o"].T

    def hidden(self):
        c, w, loop = self.c, self.w, self.c["loop"]
        x = x0 = w["embed"][self.ids]
        passes = [list(range(loop["start"], loop["stop"]))] * loop["times"]
        for t, layers in enumerate(passes):                # (every layer of these sizes is in the loop)
            x = torch.cat([x, x0], dim=-1) @ w["loop.in"].T + w["loop.step"][t]
            for i in layers:
                layer, F = c["layers"][i], self.sub(f"l{i}.mlp.")
                h = self.norm(x, f"l{i}.norm1")
                x = x + self.mixer(layer["type"], h, self.sub(f"l{i}.mix."), layer["mixer"]) + (_silu(h @ F["gate"].T) * (h @ F["up"].T)) @ F["down"].T
        return x

    def logits(self, rows):
        return self.norm(rows, "final.norm") @ self.w["head"].T


class _Tegolix(_Exact):
    def gla(self, h, W, m):
        B, T = h.shape[:2]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        q, k, v = (h @ W["q"].T).view(B, T, H, D) * D ** -0.5, (h @ W["k"].T).view(B, T, H, D), (h @ W["v"].T).view(B, T, H, V)
        alpha = torch.exp(torch.nn.functional.logsigmoid(h @ W["a1"].T @ W["a2"].T + W["a2.b"]) / m["tau"]).view(B, T, H, D)
        S, ys = torch.zeros(B, H, D, V, dtype=h.dtype, device=h.device), []
        for t in range(T):
            S = alpha[:, t, ..., None] * S + k[:, t, ..., None] * v[:, t, :, None]
            ys.append((q[:, t, :, None] @ S)[:, :, 0])
        o = (_rms(torch.stack(ys, dim=1), self.c["norm"]["eps"]) * W["norm"]).flatten(2)
        return (o * _silu(h @ W["g"].T)) @ W["o"].T

    def left(self, h, W, m):
        B, T = h.shape[:2]
        eps, rot, sc = self.c["norm"]["eps"], m["rot"], m["rot"]["scaling"]
        dims = rot["dims"]

        def turns(t):
            return dims * math.log(sc["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(rot["base"]))
        lo, hi = max(math.floor(turns(sc["fast"])), 0), min(math.ceil(turns(sc["slow"])), dims - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
        freqs = [rot["base"] ** (-2.0 * i / dims) * (r / sc["factor"] + 1.0 - r) for i, r in enumerate(ramp)]
        amplitude = 0.1 * math.log(sc["factor"]) + 1.0
        vfreqs = [rot["base"] ** (-2.0 * i / m["vdim"]) for i in range(m["vdim"] // 2)]
        q, k, v = ((h @ W[n].T).view(B, T, -1, d) for n, d in (("q", m["dim"]), ("k", m["dim"]), ("v", m["vdim"])))
        q, k = _turn(_rms(q, eps) * W["q.norm"], freqs, amplitude), _turn(_rms(k, eps) * W["k.norm"], freqs, amplitude)
        o = _attend(q, k, _turn(v, vfreqs), m["scale"], window=m["mask"]["size"], softcap=m["softcap"])
        return (_turn(o, vfreqs, back=True) * torch.sigmoid(h @ W["g"].T)[..., None]).flatten(2) @ W["o"].T

    def right(self, h, W, m):
        B, T = h.shape[:2]
        H, D = m["heads"], m["dim"]
        before = torch.nn.functional.pad(h, (0, 0, 1, 0))[:, :T]
        r, k, v, g, w = (h + (before - h) * W[f"mu.{n}"] for n in "rkvgw")
        r, k, v = ((a @ W[n].T).view(B, T, H, D) for a, n in ((r, "r"), (k, "k"), (v, "v")))
        w = torch.exp(-torch.exp(torch.tanh(w @ W["w1"].T) @ W["w2"].T + W["w0"])).view(B, T, H, D)
        S, ys = torch.zeros(B, H, D, D, dtype=h.dtype, device=h.device), []
        for t in range(T):
            kv = k[:, t, ..., None] * v[:, t, :, None]
            ys.append((r[:, t, :, None] @ (S + W["u"][..., None] * kv))[:, :, 0])
            S = w[:, t, ..., None] * S + kv
        o = _rms(torch.stack(ys, dim=1), self.c["norm"]["eps"]).flatten(2) * W["norm"]
        return (o * _silu(g @ W["g"].T)) @ W["o"].T

    def hidden(self):
        c, w, side = self.c, self.w, self.c["token_side"]["dim"]
        x = w["embed"][self.ids]
        for i, layer in enumerate(c["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = self.norm(x, p + "norm1")
            y = self.gla(h, self.sub(p + "mix."), m) if layer["type"] == "gla" else \
                m["left_scale"] * self.left(h, self.sub(p + "mix.left."), m["left"]) + m["right_scale"] * self.right(h, self.sub(p + "mix.right."), m["right"])
            x = x + self.norm(y, p + "norm1b") * w[p + "ls1"]
            h, F = self.norm(x, p + "norm2"), self.sub(p + "mlp.")
            if mlp["kind"] == "dense":
                y = (torch.relu(h @ F["gate"].T) * (h @ F["up"].T)) @ F["down"].T
            else:
                y = self.experts(h.flatten(0, 1), F, mlp, lambda a, gate, up, down: (_silu(a @ gate.T) * (a @ up.T)) @ down.T).view_as(h)
                shared = (_silu(h @ F["shared.gate"].T) * (h @ F["shared.up"].T)) @ F["shared.down"].T
                y = y + shared * torch.sigmoid(h @ F["shared.sg"].T)
            x = x + self.norm(y, p + "norm2b") * w[p + "ls2"]
            e = w["side.embed"][:, i * side:(i + 1) * side][self.ids]
            x = x + _rms((_gelu(x @ w[p + "side.gate"].T) * e) @ w[p + "side.proj"].T, c["norm"]["eps"]) * w[p + "side.norm"]
        return x

    def logits(self, rows):
        return self.norm(rows, "final.norm") @ self.w["head"].T


class _Kufolorn(_Exact):
    def delta(self, h, W, m):
        B, T = h.shape[:2]
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (_convolve(h @ W[n].T, W[f"{n}.conv"]).view(B, T, -1, D) for n in "qkv")
        q, k = ((t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, dim=2) for t in (q, k))
        q = q * D ** -0.5
        beta = torch.sigmoid(h @ W["b"].T)
        decay = torch.exp(-torch.exp(W["A_log"]) * torch.nn.functional.softplus(h @ W["a"].T + W["dt_bias"], threshold=1e9))
        S, ys = torch.zeros(B, H, D, D, dtype=h.dtype, device=h.device), []
        for t in range(T):
            S = decay[:, t, :, None, None] * S
            u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
            S = S + k[:, t, ..., None] * u[:, :, None]
            ys.append((q[:, t, :, None] @ S)[:, :, 0])
        o = _rms(torch.stack(ys, dim=1), self.c["norm"]["eps"]) * W["norm"] * _silu(h @ W["g"].T).view(B, T, H, -1)
        return o.flatten(2) @ W["o"].T

    def left(self, h, W, m):
        B, T = h.shape[:2]
        eps, rot = self.c["norm"]["eps"], m["rot"]
        freqs = [rot["base"] ** (-2.0 * i / rot["dims"]) / rot["scaling"]["factor"] for i in range(rot["dims"] // 2)]
        q = (_rms(h @ W["q"].T + W["q.b"], eps) * W["q.norm"]).view(B, T, m["heads"], -1)
        k = (_rms(h @ W["k"].T + W["k.b"], eps) * W["k.norm"]).view(B, T, m["kv_heads"], -1)
        v = (h @ W["v"].T + W["v.b"]).view(B, T, m["kv_heads"], -1)
        o = _attend(_turn(q, freqs), _turn(k, freqs), v, m["scale"], sinks=W["sink"])
        return (o * torch.sigmoid(h @ W["g"].T)[..., None]).flatten(2) @ W["o"].T

    def right(self, h, W, m):
        B, T = h.shape[:2]
        H, D, rot = m["heads"], m["dim"], m["rot"]
        freqs = [rot["base"] ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)]
        q, k = (_turn((h @ W[n].T).view(B, T, H, D), freqs) for n in "qk")
        v = (h @ W["v"].T).view(B, T, H, -1)
        decay = torch.tensor(m["decay"], dtype=h.dtype, device=h.device)[:, None, None]
        S, ys = torch.zeros(B, H, D, v.shape[-1], dtype=h.dtype, device=h.device), []
        for t in range(T):
            S = decay * S + (k[:, t, ..., None] * D ** -0.5) * v[:, t, :, None]
            ys.append((q[:, t, :, None] @ S)[:, :, 0])
        o = _rms(torch.stack(ys, dim=1), self.c["norm"]["eps"]).flatten(2)
        return (o * _silu(h @ W["g"].T)) @ W["o"].T

    def hidden(self):
        c, w = self.c, self.w
        x = w["embed"][self.ids]
        for i, layer in enumerate(c["layers"]):
            m, F = layer["mixer"], self.sub(f"l{i}.mlp.")
            y = self.delta(x, self.sub(f"l{i}.mix."), m) if layer["type"] == "delta" else \
                m["left_scale"] * self.left(x, self.sub(f"l{i}.mix.left."), m["left"]) + m["right_scale"] * self.right(x, self.sub(f"l{i}.mix.right."), m["right"])
            x = x + self.norm(y, f"l{i}.norm1")
            y = (_gelu(x @ F["gate"].T) * (x @ F["up"].T)) @ F["down"].T
            x = x + self.norm(y, f"l{i}.norm2")
        return x

    def logits(self, rows):
        cap = self.c["logit_softcap"]
        return cap * torch.tanh(self.norm(rows, "final.norm") @ self.w["embed"].T / cap)


EXACT = {"llama-1b": _Llama, "llama-3b": _Llama, "morulix": _Morulix, "tegolix": _Tegolix, "kufolorn": _Kufolorn}
EXACT_TOKENS = 16384        # tokens that go through the 64-bit model together (its products and scores must fit the memory)


@torch.no_grad()
def exact(case: dict, seed: int) -> torch.Tensor:
    """The logits of the first pass over these inputs, from whole sequences in 64 bits."""
    prompts, decoding = _inputs(case, seed)
    model, params = _weights(case, seed)
    w = {}
    for name, dest in model.spec.checkpoint.items():
        t = dest.view(params[dest.param])
        w[name] = (t.t() if dest.transpose else t).to(torch.float64)
    sequences = decoding + prompts
    out = []
    while sequences:
        most = max(1, EXACT_TOKENS // max(map(len, sequences)))
        part, sequences = sequences[:most], sequences[most:]
        ids = torch.zeros(len(part), max(map(len, part)), dtype=torch.long)
        for i, t in enumerate(part):
            ids[i, :len(t)] = torch.tensor(t)              # (what follows a sequence's end is seen by nothing before it)
        net = EXACT[case["model"]](MODELS[case["model"]], w, ids.to(DEVICE))
        x = net.hidden()
        out.append(net.logits(torch.stack([x[i, len(t) - 1] for i, t in enumerate(part)])))
    return torch.cat(out)
