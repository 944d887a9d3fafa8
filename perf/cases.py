"""The work that a user has this engine do, as measurable cases: steps of the model through ``ModelRunner.step``, the one
function that the scheduler, the command line, the Python entry points and the trace replay all call.

A case is a model, its requests and a kind of pass:

  decode  every request holds ``context`` tokens in the cache (``ragged``: from a sixteenth of that up) and brings one more;
          a pass is one step.  The requests grow by a token a pass and go back to where they began every RENEW passes.
  feed    prompts are fed from nothing in portions under the engine's budget of 2,048 tokens a step, beside single tokens of
          the requests whose prompt is done, until each has had ``new`` further tokens (0: the prompts alone); then every
          request ends.  A pass is all of these steps.  ``score``: the logits of every prompt token are wanted, not of the last.

The tokens that follow a prompt are given and not sampled, so that an output is a function of the inputs alone.  Layer sizes
are those of ``bench.py``: the Qwen3 family's (with fewer layers where a whole model says no more) and, for the six other
designs, its width 2,048 and 4,096.  What random weights of one spread do not give a model is given to it here: gates and
decays that remember from a few to a thousand tokens, and routers that are sure of their choice (``topics``).
"""
from __future__ import annotations

import hashlib
import math
from typing import Dict, List

import torch
import torch.nn.functional as F

import bench
from lucciola_amd import models  # noqa: F401  (registers the architectures)
from lucciola_amd.config.engine_config import EngineConfig
from lucciola_amd.config.registry import architecture_for
from lucciola_amd.engine.batch import StepEntry
from lucciola_amd.engine.runner import ModelRunner
from lucciola_amd.models.causal_lm import CausalLM
from lucciola_amd.weights.loader import DictSource

PAGE = 16
BUDGET = 2048          # tokens a step, the engine's default
RENEW = 256            # decode passes after which the requests go back to the context that they began with
F64 = torch.float64
QWEN = ("0.6b", "1.7b", "4b", "8b")
DESIGNS = ("pubodra", "larupel", "kikunex", "rununex", "vasanex", "nogosun")
DESIGN_CONFIGS = {"larupel": bench.larupel_design_config, "kikunex": bench.kikunex_design_config,
                  "rununex": bench.rununex_design_config, "vasanex": bench.vasanex_design_config,
                  "nogosun": bench.nogosun_design_config}


# ---------------------------------------------------------------------------------------------- the cases
def _case(name, model, size, kind, requests, context, layers=0, dtype="bfloat16", ragged=False, new=0, score=False):
    case = {"model": model, "size": size, "layers": layers, "dtype": dtype, "kind": kind, "requests": requests,
            "context": context, "ragged": ragged, "new": new, "score": score}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one person's reply from the smallest model, token by token: launches and latency
        _case("reply, one request", "qwen3", "0.6b", "decode", 1, 300, layers=28),
        # continuous batching: prompts of uneven length in portions beside the tokens of those that are done
        _case("serving, mixed steps", "qwen3", "0.6b", "feed", 12, 900, layers=28, ragged=True, new=12),
        # the headline: eight long conversations
        _case("decode, 8 x 8192", "qwen3", "8b", "decode", 8, 8192, layers=8),
        # the headline's prompt
        _case("prompt of 2048", "qwen3", "8b", "feed", 1, 2048, layers=8),
        # a trace replayed in 32 bits: logits wanted at every place of a few short prompts
        _case("trace in 32 bits", "qwen3", "0.6b", "feed", 3, 333, layers=28, dtype="float32", ragged=True, score=True),
        # a full batch that reads a latent cache, routed experts
        _case("pubodra decode", "pubodra", "w2048", "decode", 64, 2047),
        # a long document, two portions, latent attention
        _case("pubodra document", "pubodra", "w2048", "feed", 1, 4001),
        # three prompts in one step through both delta rules and routed experts
        _case("larupel prompts", "larupel", "w2048", "feed", 3, 1200, ragged=True),
        # a small batch: a state per request beside latent rows, few tokens over many experts
        _case("kikunex decode", "kikunex", "w2048", "decode", 8, 2047),
        # a prompt through differential attention, the state space and experts in every layer
        _case("rununex prompt", "rununex", "w2048", "feed", 1, 2048),
        # the larger width: a full batch of uneven requests, matrix memory and windowed attention
        _case("vasanex decode", "vasanex", "w4096", "decode", 64, 2047, ragged=True),
        # a prompt of an odd length: capped attention, gated linear attention, the delta rule by channel, experts
        _case("nogosun prompt", "nogosun", "w2048", "feed", 1, 1523),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _cost(case) -> float:
    """Seconds, roughly: bytes at half of the memory's rate or flops at a fifth of the matrix cores', and its steps' launches."""
    need = work(case)
    steps = len(schedule(case)) if case["kind"] == "feed" else 1
    return max(need["bytes"] / 4e12, need["flops"] / (5e14 if case["dtype"] == "bfloat16" else 5e13)) + steps * 1e-3


def draw(rng):
    """Another model, kind and set of requests of the same ranges, that costs no more than the largest of the list."""
    most = max(_cost(case) for case in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


def _draw(rng):
    qwen = rng.random() < 0.35
    model, size = ("qwen3", rng.choice(QWEN)) if qwen else (rng.choice(DESIGNS), rng.choice(("w2048", "w2048", "w4096")))
    layers = rng.choice((4, 6, 8)) if qwen else 0
    ragged = rng.random() < 0.5
    if rng.random() < 0.45:
        requests = _spread(rng, 1, 64)
        context = _spread(rng, 17, max(18, min(8000, 130000 // requests)))
        return _case("", model, size, "decode", requests, context, layers, ragged=ragged)
    requests = _spread(rng, 1, 12)
    context = _spread(rng, 16, max(17, min(4000, 5000 // requests)))
    if qwen and rng.random() < 0.25:
        return _case("", model, "0.6b", "feed", min(requests, 4), min(context, 400), layers, dtype="float32", ragged=ragged, score=True)
    return _case("", model, size, "feed", requests, context, layers, ragged=ragged, new=rng.choice((0, 0, rng.randint(2, 12))))


def config_of(case) -> dict:
    if case["model"] == "qwen3":
        return dict(bench.SIZES[case["size"]], architectures=["Qwen3ForCausalLM"], num_hidden_layers=case["layers"])
    if case["model"] == "pubodra":
        return bench.design_configs(case["size"], True)[1]
    return DESIGN_CONFIGS[case["model"]](case["size"])


def lengths_of(case) -> List[int]:
    """Tokens of each request: the context, or (ragged) from a sixteenth of it to the whole, spread over the logarithm."""
    n, most = case["requests"], case["context"]
    if not case["ragged"]:
        return [most] * n
    return [most] + [max(1, int(most * 16.0 ** -((i * 0.6180339887498949) % 1.0))) for i in range(1, n)]


def schedule(case):
    """The steps of a feed pass: lists of (request, first token, token behind the last, wanted places)."""
    lengths, new = lengths_of(case), case["new"]
    fed, steps = [0] * len(lengths), []
    while any(f < n + new for f, n in zip(fed, lengths)):
        step, room = [], BUDGET
        for r, n in enumerate(lengths):         # single tokens first
            if n <= fed[r] < n + new:
                step.append((r, fed[r], fed[r] + 1, [0]))
                room -= 1
        for r, n in enumerate(lengths):         # then portions, in the order of arrival
            if fed[r] < n and room > 0:
                take = min(room, n - fed[r])
                last = [take - 1] if fed[r] + take == n else []
                step.append((r, fed[r], fed[r] + take, list(range(take)) if case["score"] else last))
                room -= take
        for r, _, end, _ in step:
            fed[r] = end
        steps.append(step)
    return steps


def tokens_of(case, seed, vocab) -> List[List[int]]:
    """Every request's tokens: its prompt and what follows."""
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 11)
    more = 2 if case["kind"] == "decode" else case["new"]
    return [torch.randint(0, vocab, (n + more,), generator=gen).tolist() for n in lengths_of(case)]


# ---------------------------------------------------------------------------------------------- weights
def _key(seed, name) -> int:
    return int.from_bytes(hashlib.sha256(f"{seed} {name}".encode()).digest()[:7], "little")


def declared(cfg) -> Dict[str, tuple]:
    """Every tensor of the model: name -> (shape, how it is filled)."""
    out: Dict[str, tuple] = {}
    if "num_hidden_layers" in cfg:
        W, I, d = cfg["hidden_size"], cfg["intermediate_size"], cfg["head_dim"]
        nq, nk = cfg["num_attention_heads"] * d, cfg["num_key_value_heads"] * d
        out["model.embed_tokens.weight"] = ((cfg["vocab_size"], W), "matrix")
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            for n, shape in (("q", (nq, W)), ("k", (nk, W)), ("v", (nk, W)), ("o", (W, nq))):
                out[f"{p}self_attn.{n}_proj.weight"] = (shape, "matrix")
            for n in ("self_attn.q_norm", "self_attn.k_norm"):
                out[f"{p}{n}.weight"] = ((d,), "norm")
            for n, shape in (("gate", (I, W)), ("up", (I, W)), ("down", (W, I))):
                out[f"{p}mlp.{n}_proj.weight"] = (shape, "matrix")
            for n in ("input_layernorm", "post_attention_layernorm"):
                out[f"{p}{n}.weight"] = ((W,), "norm")
        out["model.norm.weight"] = ((W,), "norm")
        if not cfg["tie_word_embeddings"]:
            out["lm_head.weight"] = ((cfg["vocab_size"], W), "matrix")
        return out

    kind, W = cfg["architecture"].lower(), cfg["width"]

    def add(name, shape, fill="matrix"):
        out[name] = (tuple(shape), fill)

    def norm(name):
        if kind == "kikunex":
            add(name, (), "norm")
        elif kind == "vasanex":
            add(name, (W,), "small")
        else:
            add(name, (W,), "norm")
        if kind in ("pubodra", "larupel"):
            add(name + ".b", (W,), "small")
        if kind == "pubodra":
            add(name + ".alpha", (), "alpha")

    def heads(p, m, biases="", norms=""):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        maps = 2 if m.get("diff") else 1
        for n, shape in (("q", (H * d * maps, W)), ("k", (G * d * maps, W)), ("v", (G * dv, W)), ("o", (W, H * dv))):
            add(p + n, shape)
        for n, rows in (("q", H * d), ("k", G * d), ("v", G * dv), ("o", W)):
            if n in biases:
                add(f"{p}{n}.b", (rows,), "small")
        for n, rows in (("q", H), ("k", G)):
            if norms:
                add(f"{p}{n}.norm", (d if norms == "head" else rows * d,), "norm")
        if m.get("conv"):
            for n, rows in (("q", H * d * maps), ("k", G * d * maps), ("v", G * dv)):
                add(f"{p}{n}.conv", (rows, m["conv"]), "taps")

    add("embed", (cfg["vocab"], W), "embed")
    if kind == "kikunex":
        add("embed.norm", (), "norm")
    for i, layer in enumerate(cfg["layers"]):
        if layer.get("weights_of") is not None:
            continue
        p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
        x, what = p + "mix.", layer["type"]
        if what == "latent_attention":
            H, rank = m["heads"], m["kv_rank"]
            if m.get("q_rank"):
                add(x + "dq", (m["q_rank"], W))
                add(x + "dq.norm", (m["q_rank"],), "norm")
                add(x + "uq", (H * (m["dim"] + m["rot_dim"]), m["q_rank"]))
                add(x + "g", (H, W))
                add(x + "sink", (H,), "sink")
            else:
                add(x + "q", (H * (m["dim"] + m["rot_dim"]), W))
                add(x + "g", (H * m["vdim"], W))
            add(x + "dkv", (rank + m["rot_dim"], W))
            add(x + "dkv.norm", (rank,), "norm")
            add(x + "uk", (H * m["dim"], rank))
            add(x + "uv", (H * m["vdim"], rank))
            add(x + "o", (W, H * m["vdim"]))
        elif what == "attention" and kind == "larupel":
            heads(x, m, norms="head")
            if m.get("kv_from") is not None:
                for n in ("k", "v", "k.norm"):
                    del out[x + n]
            add(x + "temp", (m["heads"],), "norm")
        elif what == "attention" and kind == "rununex":
            heads(x, m)
            for n in ("lq1", "lk1", "lq2", "lk2"):
                add(x + n, (m["dim"],), "lambda")
        elif what == "attention" and kind == "vasanex":
            heads(x, m, biases="qkvo", norms="row")
            add(x + "sink", (m["heads"],), "sink")
            add(x + "vmix", (), "mix")
        elif what == "attention":
            heads(x, m, biases="qk")
            del out[x + "v"]
        elif what == "general_delta":
            n = m["heads"] * m["dim"]
            for name in ("r", "k", "v", "g", "a"):
                add(x + name, (n, W))
            add(x + "a.b", (n,), "small")
            add(x + "w1", (16, W))
            add(x + "w2", (n, 16), "wide")
            add(x + "w0", (n,), "forget")
            add(x + "norm", (n,), "norm")
            add(x + "o", (W, n))
        elif what in ("delta", "channel_delta"):
            H, nk, nv = m["heads"], m["kv_heads"] * m["dim"], m["heads"] * m["vdim"]
            for name, rows in (("q", nk), ("k", nk), ("v", nv)):
                add(x + name, (rows, W))
                add(f"{x}{name}.conv", (rows, m["conv"]), "taps")
            add(x + "b", (H, W))
            add(x + "A_log", (H,), "rate")
            add(x + "norm", (m["vdim"],), "norm")
            add(x + "o", (W, nv))
            if what == "delta":
                add(x + "a", (H, W))
                add(x + "dt_bias", (H,), "step")
                add(x + "g", (nv, W))
            else:
                add(x + "a1", (m["dim"], W))
                add(x + "a2", (H * m["dim"], m["dim"]))
                add(x + "dt_bias", (H * m["dim"],), "step")
                add(x + "g1", (m["vdim"], W))
                add(x + "g2", (nv, m["vdim"]), "wide")
        elif what == "lightning":
            H = m["heads"]
            for name, rows in (("q", H * m["dim"]), ("k", H * m["dim"]), ("v", H * m["vdim"]), ("g", H * m["vdim"])):
                add(x + name, (rows, W))
            add(x + "norm", (H * m["vdim"],), "norm")
            add(x + "o", (W, H * m["vdim"]))
        elif what == "mlstm":
            H = m["heads"]
            for name, rows in (("q", H * m["dim"]), ("k", H * m["dim"]), ("v", H * m["vdim"]), ("g", H * m["vdim"]),
                               ("i", H), ("f", H)):
                add(x + name, (rows, W))
            add(x + "i.b", (H,), "small")
            add(x + "f.b", (H,), "remember")
            add(x + "norm", (H * m["vdim"],), "norm")
            add(x + "o", (W, H * m["vdim"]))
        elif what == "parallel" and kind == "rununex":
            left, right = m["left"], m["right"]
            heads(x + "left.", left)
            add(x + "left.r1", (left["heads"],), "norm")
            add(x + "left.r2", (left["heads"],), "norm")
            add(x + "left.sink", (left["heads"],), "sink")
            add(x + "left.g", (left["heads"] * left["vdim"], W))
            inner, both = right["heads"] * right["vdim"], 2 * right["groups"] * right["state"]
            add(x + "right.in", (2 * inner + both + right["heads"], W))
            add(x + "right.conv", (inner + both, right["conv"]), "taps")
            add(x + "right.conv.b", (inner + both,), "small")
            add(x + "right.dt_bias", (right["heads"],), "step")
            add(x + "right.A_log", (right["heads"],), "rate")
            add(x + "right.D", (right["heads"],), "norm")
            add(x + "right.norm", (inner,), "norm")
            add(x + "right.o", (W, inner))
        else:
            left, right = m["left"], m["right"]
            heads(x + "left.", left, biases="qkv", norms="head")
            add(x + "left.g", (left["heads"] * left["vdim"], W))
            H = right["heads"]
            for name, rows in (("q", H * right["dim"]), ("k", H * right["dim"]), ("v", H * right["vdim"]), ("g", H * right["vdim"])):
                add(x + "right." + name, (rows, W))
            add(x + "right.a1", (16, W))
            add(x + "right.a2", (H * right["dim"], 16), "wide")
            add(x + "right.a2.b", (H * right["dim"],), "keep")
            add(x + "right.norm", (right["vdim"],), "norm")
            add(x + "right.o", (W, H * right["vdim"]))
        x = p + "mlp."
        gated = kind in ("larupel", "rununex", "vasanex")
        units = [(x, mlp["ff"])] if mlp["kind"] == "dense" else \
            [(f"{x}e{e}.", mlp["expert"]["ff"]) for e in range(mlp["router"]["experts"])]
        if mlp.get("shared"):
            units.append((x + "shared.", mlp["shared"]["ff"]))
        for prefix, ff in units:
            if gated:
                add(prefix + "gate", (ff, W))
            add(prefix + "up", (ff, W))
            add(prefix + "down", (W, ff))
        if mlp["kind"] == "moe":
            add(x + "router", (mlp["router"]["experts"], W), "router")
            if kind == "larupel":
                add(x + "router.b", (mlp["router"]["experts"],), "zero")
                add(x + "shared.sg", (1, W))
            if kind == "kikunex":
                add(x + "correction", (mlp["router"]["experts"],), "zero")
        elif kind == "kikunex":
            add(x + "act", (2,), "act")
        norm(p + "norm1")
        norm(p + "norm2")
        if kind == "larupel":
            norm(p + "norm1b")
            norm(p + "norm2b")
        if kind == "kikunex":
            add(p + "shift", (W,), "unit")
    norm("final.norm")
    if kind not in ("pubodra", "vasanex"):
        add("head", (cfg["vocab"], W))
    return out


UNIFORM = {"forget": (-6.0, -1.0), "remember": (3.0, 6.0), "keep": (-2.0, 4.0), "unit": (0.0, 1.0), "mix": (0.2, 0.4),
           "act": (0.3, 0.8), "alpha": (0.45, 0.55)}
NORMAL = {"matrix": 0.02, "small": 0.02, "embed": 0.02, "wide": 0.2, "taps": 0.3, "sink": 1.0, "lambda": 0.1}


def topics(cfg, w, seed) -> None:
    """Routers that are sure, as trained ones mostly are: a token's embedding marks the four experts that suit it in the
    first coordinates, no branch writes there, and a layer's router reads them in an order of its own.  Two of the four are
    neighbours of one group of eight and two of another.  (With routers of noise, a last bit decides between two experts.)"""
    routed = [i for i, layer in enumerate(cfg["layers"]) if layer["mlp"]["kind"] == "moe" and layer.get("weights_of") is None]
    if not routed:
        return
    E = cfg["layers"][routed[0]]["mlp"]["router"]["experts"]
    dev = w["embed"].device
    gen = torch.Generator(device=dev).manual_seed(_key(seed, "topics"))
    groups = torch.rand((cfg["vocab"], E // 8), device=dev, generator=gen).argsort(1)[:, :2]
    inside = torch.rand((cfg["vocab"], 2, 8), device=dev, generator=gen).argsort(2)[:, :, :2]
    chosen = (groups[:, :, None] * 8 + inside).reshape(-1, 4)
    scale = {"pubodra": 1.0, "larupel": 1.0, "kikunex": 50.0}.get(cfg["architecture"].lower()) or cfg["embedding"]["scale"]
    marks = torch.zeros((cfg["vocab"], E), device=dev)
    marks.scatter_(1, chosen, torch.tensor([6.0, 5.1, 4.2, 3.3], device=dev).expand(cfg["vocab"], 4) / scale)
    w["embed"][:, :E] = marks.to(w["embed"].dtype)
    for name in w:
        if name.endswith((".o", ".down", ".o.b")) or ".norm1b" in name or ".norm2b" in name:
            w[name][:E] = 0
    for i in routed:
        order = torch.randperm(E // 8, device=dev, generator=gen)[:, None] * 8 + torch.randperm(8, device=dev, generator=gen)[None]
        w[f"l{i}.mlp.router"][:, :E] = torch.eye(E, device=dev)[order.reshape(-1)].to(w["embed"].dtype) * 2.0


def weights_of(cfg, seed, device="cuda") -> Dict[str, torch.Tensor]:
    w = {}
    for name, (shape, fill) in declared(cfg).items():
        gen = torch.Generator(device=device).manual_seed(_key(seed, name))
        if fill == "zero":
            t = torch.zeros(shape, device=device)
        elif fill == "router":
            t = torch.randn(shape, device=device, generator=gen) * 0.002
        elif fill in UNIFORM:
            low, high = UNIFORM[fill]
            t = torch.rand(shape, device=device, generator=gen) * (high - low) + low
        elif fill == "rate":        # log of 1 to 16
            t = torch.log(torch.rand(shape, device=device, generator=gen) * 15.0 + 1.0)
        elif fill == "step":        # softplus of it: 0.001 to 0.1, spread over the logarithm
            dt = torch.exp(torch.rand(shape, device=device, generator=gen) * math.log(100.0) + math.log(0.001))
            t = dt + torch.log(-torch.expm1(-dt))
        elif fill == "norm":
            t = torch.randn(shape, device=device, generator=gen) * 0.02 + 1.0
        else:
            t = torch.randn(shape, device=device, generator=gen) * NORMAL[fill]
        w[name] = t.to(torch.bfloat16)
    if "architecture" in cfg:
        topics(cfg, w, seed)
    return w


# ---------------------------------------------------------------------------------------------- what is measured
class State:
    def __init__(self, runner, case, tokens):
        self.runner, self.case, self.tokens = runner, case, tokens
        self.names = [f"request {r}" for r in range(len(tokens))]
        self.steps, self.held, self.passes = [], [], 0


def prepare(case, seed):
    cfg = config_of(case)
    arch = architecture_for(cfg)
    model = CausalLM(arch.model_spec(arch.read_config(cfg)), DictSource(weights_of(cfg, seed)),
                     torch.float32 if case["dtype"] == "float32" else torch.bfloat16, "cuda:0")
    lengths = lengths_of(case)
    spare = RENEW + 8 if case["kind"] == "decode" else case["new"] + 8
    blocks = sum(-(-(n + spare) // PAGE) for n in lengths) + 8
    runner = ModelRunner(model, EngineConfig(dtype=case["dtype"], block_size=PAGE, max_blocks=blocks, max_seqs=len(lengths) + 1))
    state = State(runner, case, tokens_of(case, seed, model.vocab_size))
    if case["kind"] == "feed":
        state.steps = [[StepEntry(state.names[r], state.tokens[r][a:b], want) for r, a, b, want in step]
                       for step in schedule(case)]
        return state
    # a conversation under way: the prompts have been fed and a first token decoded
    for step in schedule(dict(case, kind="feed", new=0, score=False)):
        runner.step([StepEntry(state.names[r], state.tokens[r][a:b], want) for r, a, b, want in step])
    runner.step([StepEntry(n, t[-2:-1], [0]) for n, t in zip(state.names, state.tokens)])
    state.held = [n + 1 for n in lengths]
    state.steps = [[StepEntry(n, t[-1:], [0]) for n, t in zip(state.names, state.tokens)]]
    return state


def run(state):
    runner = state.runner
    if state.case["kind"] == "feed":
        logits = [runner.step(step) for step in state.steps]
        for name in state.names:
            runner.finish(name)
        return [out for out in logits if out.shape[0]]
    if state.passes == RENEW:
        for name, held in zip(state.names, state.held):
            runner.finish(name)
            runner.cache.admit(name)
            runner.cache.reserve(name, held)
            runner.cache.commit(name)
        state.passes = 0
    state.passes += 1
    return runner.step(state.steps[0])


# ---------------------------------------------------------------------------------------------- what it cannot do without
def _mixer_work(cfg, layer) -> tuple:
    """(bytes a token leaves in the cache, bytes of state a request has, flops a query spends on a key, flops a token spends on
    the state, the most keys a query sees) of one layer, in entries of the case's type for the cache and of 32 bits for states."""
    if layer is None:
        G, H, d = cfg["num_key_value_heads"], cfg["num_attention_heads"], cfg["head_dim"]
        return 2 * G * d, 0, 4 * H * d, 0, None
    m, what = layer["mixer"], layer["type"]
    if what == "parallel":
        left = _mixer_work(cfg, {"mixer": m["left"], "type": "attention"})
        r = m["right"]
        entries = r["heads"] * r["vdim"] * (r["state"] if "state" in r else r["dim"])
        return left[0], entries, left[2], 5 * entries, left[4]
    most = (m.get("mask") or {}).get("size")
    if what == "latent_attention":
        row = m["kv_rank"] + m["rot_dim"]
        return row, 0, 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), 0, most
    if what == "attention":
        maps = 2 if m.get("diff") else 1
        flops = 2 * m["heads"] * maps * (m["dim"] + m["vdim"])
        stored = 0 if m.get("kv_from") is not None else m["kv_heads"] * (maps * m["dim"] + m["vdim"])
        return stored, 0, flops, 0, most
    entries = m["heads"] * m["dim"] * m.get("vdim", m["dim"])
    return 0, entries, 0, (9 if "delta" in what else 5) * entries, None


def work(case):
    """Each step reads every weight that its tokens need once, the cache of its requests once and their states, and writes the
    new rows, the states and its logits."""
    cfg = config_of(case)
    size = 4 if case["dtype"] == "float32" else 2
    layers = cfg.get("layers") or [None] * cfg["num_hidden_layers"]
    lengths = lengths_of(case)
    steps = schedule(case) if case["kind"] == "feed" else [[(r, n + 1, n + 2, [0]) for r, n in enumerate(lengths)]]
    plain, expert, experts, top, vocab, width = 0, [0] * len(layers), 0, 0, 0, 0
    for name, (shape, fill) in declared(cfg).items():
        n = math.prod(shape)
        if fill == "embed" or name == "model.embed_tokens.weight":
            vocab, width = shape
        elif name in ("head", "lm_head.weight"):
            pass
        elif ".mlp.e" in name:
            expert[int(name[1:name.index(".")])] += n
        else:
            plain += n
    for i, layer in enumerate(layers):
        if layer and layer["mlp"]["kind"] == "moe":
            experts, top = layer["mlp"]["router"]["experts"], layer["mlp"]["router"]["top"]
    bytes_, flops = 0.0, 0.0
    for step in steps:
        tokens, wanted = sum(b - a for _, a, b, _ in step), sum(len(w) for _, _, _, w in step)
        bytes_ += plain * 2 + (vocab * width * 2 if wanted else 0) + tokens * width * 2 + wanted * vocab * 4
        flops += 2.0 * tokens * plain + 2.0 * wanted * vocab * width
        for i, layer in enumerate(layers):
            runs = 1 + sum(1 for other in layers if other and other.get("weights_of") == i)
            if expert[i]:
                bytes_ += expert[i] * 2 * (1.0 - (1.0 - top / experts) ** tokens)
                flops += 2.0 * runs * tokens * expert[i] * top / experts
            row, entries, per_key, per_state, most = _mixer_work(cfg, layer)
            for _, a, b, _ in step:
                bytes_ += (min(b, most or b) + (b - a)) * row * size + 2 * entries * 4
                pairs = sum(min(p + 1, most or p + 1) for p in ((a + b - 1) / 2,)) * (b - a)
                flops += pairs * per_key + (b - a) * per_state
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """32-bit sums (9e-7 off the 64-bit logits where measured), or activations rounded to bfloat16 from layer to layer: 0.0014
    off for Pubodra, whose norms are tanh, and 0.006 to 0.019 for the others."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5}
    return {"rel": 0.006 if case["model"] == "pubodra" else 0.03}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
class Exact:
    """Whole sequences through the model in float64, every formula written out; rows of all sequences lie one behind the
    other, ``spans`` says where each begins and ends."""

    def __init__(self, cfg, w, sequences):
        self.cfg, self.w, self.dev = cfg, w, "cuda"
        ends = torch.tensor([len(s) for s in sequences]).cumsum(0).tolist()
        self.spans = list(zip([0] + ends[:-1], ends))
        self.ids = torch.tensor([t for s in sequences for t in s], device=self.dev)
        self.positions = torch.cat([torch.arange(b - a, device=self.dev, dtype=F64) for a, b in self.spans])
        self.eps = float(cfg["norm"]["eps"] if "norm" in cfg else cfg["rms_norm_eps"])

    # ---- pieces
    def t(self, name):
        return self.w[name].to(F64)

    def linear(self, x, name):
        return x @ self.t(name).T

    def rms(self, x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.eps)

    def layer_norm(self, x, name, bias=True):
        dev = x - x.mean(-1, keepdim=True)
        y = dev / torch.sqrt((dev * dev).mean(-1, keepdim=True) + self.eps) * self.t(name)
        return y + self.t(name + ".b") if bias else y

    @staticmethod
    def unit(x):
        return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)

    def rotate(self, x, rot, interleaved=False):
        """x [T, heads, n]: the first ``dims`` entries turn in pairs (neighbours, or halves apart)."""
        dims, base, scaling = rot["dims"], float(rot["base"]), rot.get("scaling")
        f = base ** (-2.0 * torch.arange(dims // 2, dtype=F64) / dims)
        size = 1.0
        if scaling and "fast" in scaling:
            def pair(turns):
                return dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
            low, high = max(math.floor(pair(scaling["fast"])), 0), min(math.ceil(pair(scaling["slow"])), dims - 1)
            ramp = ((torch.arange(dims // 2, dtype=F64) - low) / max(high - low, 0.001)).clamp(0, 1)
            f, size = f / scaling["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0
        elif scaling:
            wave = 2 * math.pi / f
            s = (scaling["original"] / wave - scaling["low"]) / (scaling["high"] - scaling["low"])
            s = s.clamp(0, 1)       # 1: shorter than original / high, kept; 0: longer than original / low, divided
            f = (1 - s) * f / scaling["factor"] + s * f
        angle = self.positions[:, None, None] * f.to(self.dev)
        cos, sin = angle.cos() * size, angle.sin() * size
        y = x.clone()
        one, two = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, dims // 2), slice(dims // 2, dims))
        y[..., one], y[..., two] = x[..., one] * cos - x[..., two] * sin, x[..., two] * cos + x[..., one] * sin
        return y

    def attend(self, q, k, v, scale, chunk=None, window=None, first=0, sink=None, cap=None, bias=None, one_more=False):
        """q [T, H, d], k [T, G, d], v [T, G, dv] of all sequences -> [T, H, dv]; scale: a number or one a head."""
        H, G = q.shape[1], k.shape[1]
        out = torch.empty((q.shape[0], H, v.shape[2]), dtype=F64, device=self.dev)
        scale = torch.as_tensor(scale, dtype=F64, device=self.dev).expand(H)
        for a, b in self.spans:
            n = b - a
            at = max(1, min(n, (1 << 28) // (H * n)))
            keys, values = k[a:b].permute(1, 2, 0), v[a:b].transpose(0, 1)
            for c in range(0, n, at):
                rows = min(at, n - c)
                part = (q[a + c:a + c + rows] * scale[:, None]).view(rows, G, H // G, -1).permute(1, 2, 0, 3)
                s = (part.reshape(G, H // G * rows, -1) @ keys).view(H, rows, n)
                i = torch.arange(c, c + rows, device=self.dev)[:, None]
                j = torch.arange(n, device=self.dev)[None]
                seen = j <= i
                if window:
                    seen &= (i - j < window) | (j < first)
                if chunk:
                    seen &= i // chunk == j // chunk
                if cap:
                    s = cap * torch.tanh(s / cap)
                if bias is not None:
                    s = s - bias[0][:, None, None] * torch.log1p(bias[1][:, None, None] * (i - j).clamp(min=0))
                s = s.masked_fill(~seen, -math.inf)
                more = sink[:, None, None] if sink is not None else torch.zeros((), dtype=F64, device=self.dev) if one_more else None
                top = s.amax(-1, keepdim=True)
                top = top if more is None else torch.maximum(top, more)
                e = torch.exp(s - top)
                e = e / (e.sum(-1, keepdim=True) + (0.0 if more is None else torch.exp(more - top)))
                o = e.view(G, H // G * rows, n) @ values
                out[a + c:a + c + rows] = o.view(G, H // G, rows, -1).permute(2, 0, 1, 3).reshape(rows, H, -1)
        return out

    def conv(self, x, taps, bias=0.0):
        out, K = torch.empty_like(x), taps.shape[1]
        for a, b in self.spans:
            padded = torch.cat([x.new_zeros((K - 1, x.shape[1])), x[a:b]])
            out[a:b] = sum(padded[j:j + b - a] * taps[:, j] for j in range(K)) + bias
        return out

    def scan(self, decay, write, v, read, probe=None, removal=None):
        """S <- diag(decay) S - removal (probe^T S) + write v^T;  o = S^T read; planes [T, H, d], v [T, H, dv]."""
        R, most = len(self.spans), max(b - a for a, b in self.spans)
        H, dv = v.shape[1:]

        def by_time(x):
            y = x.new_zeros((most, R) + x.shape[1:])
            for r, (a, b) in enumerate(self.spans):
                y[:b - a, r] = x[a:b]
            return y.view(most, R * H, -1)
        decay, write, v, read = by_time(decay), by_time(write), by_time(v), by_time(read)
        if probe is not None:
            probe, removal = by_time(probe), by_time(removal)
        S, out = v.new_zeros((R * H, write.shape[2], dv)), torch.empty_like(v)
        for t in range(most):
            held = torch.bmm(probe[t, :, None], S) if probe is not None else None
            S *= decay[t, :, :, None]
            if held is not None:
                S.baddbmm_(removal[t, :, :, None], held, alpha=-1.0)
            S.baddbmm_(write[t, :, :, None], v[t, :, None])
            out[t] = torch.bmm(read[t, :, None], S)[:, 0]
        out = out.view(most, R, H, dv)
        return torch.cat([out[:b - a, r] for r, (a, b) in enumerate(self.spans)])

    # ---- mixers
    def qkv(self, h, p, m, biases=""):
        q, k = self.linear(h, p + "q"), self.linear(h, p + "k") if p + "k" in self.w else None
        v = self.linear(h, p + "v") if p + "v" in self.w else None
        q = q + self.t(p + "q.b") if "q" in biases else q
        k = k + self.t(p + "k.b") if "k" in biases else k
        v = v + self.t(p + "v.b") if "v" in biases else v
        return q, k, v

    def latent(self, h, p, m):
        T, H, dim, rank = h.shape[0], m["heads"], m["dim"], m["kv_rank"]
        if m.get("q_rank"):
            q = self.linear(self.rms(self.linear(h, p + "dq")) * self.t(p + "dq.norm"), p + "uq")
        else:
            q = self.linear(h, p + "q")
        q, down = q.view(T, H, -1), self.linear(h, p + "dkv")
        near = self.cfg["architecture"] == "Pubodra"
        c = self.rms(down[:, :rank]) * self.t(p + "dkv.norm")
        turned_q = self.rotate(q[..., dim:], m["rot"], near)
        turned_k = self.rotate(down[:, None, rank:], m["rot"], near).expand(T, H, -1)
        q = torch.cat([q[..., :dim], turned_q], -1)
        k = torch.cat([self.linear(c, p + "uk").view(T, H, dim), turned_k], -1)
        v = self.linear(c, p + "uv").view(T, H, -1)
        sink = self.t(p + "sink") if p + "sink" in self.w else None
        o = self.attend(q, k, v, m["scale"], window=m["mask"]["size"], sink=sink)
        gate = torch.sigmoid(self.linear(h, p + "g"))
        o = o * gate[:, :, None] if m.get("q_rank") else o * gate.view(T, H, -1)
        return self.linear(o.reshape(T, -1), p + "o")

    def differential(self, h, p, m):
        T, H, G, d = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.conv(x, self.t(p + n + ".conv")) for x, n in zip(self.qkv(h, p, m), "qkv"))
        q, k = self.rotate(q.view(T, 2 * H, d), m["rot"], True), self.rotate(k.view(T, 2 * G, d), m["rot"], True)
        v = v.view(T, G, -1)
        one, two = (self.attend(q[:, i::2], k[:, i::2], v, m["scale"], chunk=m["mask"]["size"]) for i in (0, 1))
        lam = (torch.exp((self.t(p + "lq1") * self.t(p + "lk1")).sum())
               - torch.exp((self.t(p + "lq2") * self.t(p + "lk2")).sum()) + m["diff"])
        o = self.rms(one - lam * two) * (1.0 - m["diff"])
        return self.linear(o.reshape(T, -1), p + "o")

    def general_delta(self, h, p, m):
        T, H = h.shape[0], m["heads"]
        r, k, v = (self.linear(h, p + n).view(T, H, -1) for n in "rkv")
        inner = torch.tanh(self.linear(h, p + "w1"))
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(self.linear(inner, p + "w2") + self.t(p + "w0"))).view(T, H, -1)
        a = torch.sigmoid(self.linear(h, p + "a") + self.t(p + "a.b")).view(T, H, -1)
        u = self.unit(k)
        o = self.rms(self.scan(decay, k, v, r, u, a * u)).reshape(T, -1) * self.t(p + "norm")
        return self.linear(o * torch.sigmoid(self.linear(h, p + "g")), p + "o")

    def delta(self, h, p, m):
        T, H, G, d = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (F.silu(self.conv(self.linear(h, p + n), self.t(p + n + ".conv"))) for n in "qkv")
        q, k = (self.unit(x.view(T, G, d)).repeat_interleave(H // G, 1) for x in (q, k))
        beta = torch.sigmoid(self.linear(h, p + "b"))[:, :, None]
        rate = torch.exp(self.t(p + "A_log"))[:, None]
        if p + "a1" in self.w:
            step = F.softplus(self.linear(self.linear(h, p + "a1"), p + "a2") + self.t(p + "dt_bias")).view(T, H, d)
            gate = torch.sigmoid(self.linear(self.linear(h, p + "g1"), p + "g2"))
        else:
            step = F.softplus(self.linear(h, p + "a") + self.t(p + "dt_bias"))[:, :, None]
            gate = F.silu(self.linear(h, p + "g"))
        g = torch.exp(-rate * step).expand(T, H, d)
        o = self.scan(g, beta * k, v.view(T, H, -1), q * d ** -0.5, g * k, beta * k)
        return self.linear((self.rms(o) * self.t(p + "norm")).reshape(T, -1) * gate, p + "o")

    def lightning(self, h, p, m):
        T, H = h.shape[0], m["heads"]
        q, k, v = (F.silu(self.linear(h, p + n)).view(T, H, -1) for n in "qkv")
        # the model's constants are kept in 32 bits
        decay = torch.tensor(m["decay"], dtype=torch.float32, device=self.dev).to(F64)[:, None].expand(T, H, k.shape[2])
        o = self.rms(self.scan(decay, k, v, q).reshape(T, -1)) * self.t(p + "norm")
        return self.linear(o * torch.sigmoid(self.linear(h, p + "g")), p + "o")

    def matrix_memory(self, h, p, m):
        T, H, d, cap = h.shape[0], m["heads"], m["dim"], m["gate_cap"]
        q, k, v = (self.linear(h, p + n).view(T, H, -1) for n in "qkv")
        log_in = cap * torch.tanh((self.linear(h, p + "i") + self.t(p + "i.b")) / cap)
        log_keep = F.logsigmoid(cap * torch.tanh((self.linear(h, p + "f") + self.t(p + "f.b")) / cap))
        top = torch.zeros_like(log_in)
        for a, b in self.spans:         # m_t = max(f_t + m_(t-1), i_t) from 0: sums of f and a running maximum
            total = log_keep[a:b].cumsum(0)
            best = torch.cat([torch.zeros_like(total[:1]), log_in[a:b] - total]).cummax(0).values[1:]
            top[a:b] = total + best
        before = torch.cat([torch.zeros_like(top[:1]), top[:-1]])
        before[[a for a, _ in self.spans]] = 0.0
        keep, write = torch.exp(log_keep + before - top), torch.exp(log_in - top)
        ones = torch.cat([v, torch.ones_like(v[..., :1])], -1)      # the normaliser rides along as one more value
        o = self.scan(keep[:, :, None].expand(T, H, d), write[:, :, None] * k, ones, q * d ** -0.5)
        bottom = torch.maximum(o[..., -1:].abs(), torch.exp(-top)[:, :, None]) + 1e-6
        o = self.rms(o[..., :-1] / bottom).reshape(T, -1) * self.t(p + "norm")
        return self.linear(o * torch.sigmoid(self.linear(h, p + "g")), p + "o")

    def state_space(self, h, p, m):
        T, H, dv, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * dv
        z, xbc, dt = self.linear(h, p + "in").split([inner, inner + 2 * G * N, H], -1)
        xbc = F.silu(self.conv(xbc, self.t(p + "conv"), self.t(p + "conv.b")))
        x, B, C = xbc.split([inner, G * N, G * N], -1)
        x, B, C = x.view(T, H, dv), *(u.view(T, G, N).repeat_interleave(H // G, 1) for u in (B, C))
        dt = F.softplus(dt + self.t(p + "dt_bias"))
        decay = torch.exp(-torch.exp(self.t(p + "A_log")) * dt)[:, :, None].expand(T, H, N)
        y = self.scan(decay, dt[:, :, None] * B, x, C) + self.t(p + "D")[:, None] * x
        y = (y.reshape(T, inner) * F.silu(z)).view(T, m["norm_groups"], -1)
        return self.linear(self.rms(y).reshape(T, inner) * self.t(p + "norm"), p + "o")

    def mixer(self, kind, h, p, m, kept):
        arch, T = self.cfg["architecture"], h.shape[0]
        if kind == "latent_attention":
            return self.latent(h, p, m)
        if kind == "general_delta":
            return self.general_delta(h, p, m)
        if kind in ("delta", "channel_delta"):
            return self.delta(h, p, m)
        if kind == "lightning":
            return self.lightning(h, p, m)
        if kind == "mlstm":
            return self.matrix_memory(h, p, m)
        if arch == "Rununex" and kind == "attention":
            return self.differential(h, p, m)
        if kind == "parallel":
            left, right = m["left"], m["right"]
            H, G = left["heads"], left["kv_heads"]
            if arch == "Rununex":
                q, k, v = (x.view(T, n, -1) for x, n in zip(self.qkv(h, p + "left.", left), (H, G, G)))
                o = self.attend(self.rms(q), self.rms(k), v, left["scale"], chunk=left["mask"]["size"],
                                sink=self.t(p + "left.sink"), bias=(self.t(p + "left.r1"), self.t(p + "left.r2")))
                other = self.state_space(h, p + "right.", right)
            else:
                q, k, v = (x.view(T, n, -1) for x, n in zip(self.qkv(h, p + "left.", left, "qkv"), (H, G, G)))
                q, k = self.rms(q) * self.t(p + "left.q.norm"), self.rms(k) * self.t(p + "left.k.norm")
                temp = 1.0 + left["q_temp"]["coef"] * torch.log(torch.floor((self.positions + 1) / left["q_temp"]["every"]) + 1)
                o = self.attend(q * temp[:, None, None], k, v, left["scale"], cap=left["softcap"], one_more=True)
                R = right["heads"]
                rq, rk, rv = (self.linear(h, f"{p}right.{n}").view(T, R, -1) for n in "qkv")
                z = self.linear(self.linear(h, p + "right.a1"), p + "right.a2") + self.t(p + "right.a2.b")
                keep = (torch.sigmoid(z) ** (1.0 / right["tau"])).view(T, R, -1)
                y = self.rms(self.scan(keep, rk, rv, rq * right["dim"] ** -0.5)) * self.t(p + "right.norm")
                other = self.linear(y.reshape(T, -1) * F.silu(self.linear(h, p + "right.g")), p + "right.o")
            own = self.linear(o.reshape(T, -1) * torch.sigmoid(self.linear(h, p + "left.g")), p + "left.o")
            return m["left_scale"] * own + m["right_scale"] * other
        H, G = m["heads"], m["kv_heads"]
        if arch == "Larupel":
            q, k, v = self.qkv(h, p, m)
            q = self.rms(q.view(T, H, -1)) * self.t(p + "q.norm")
            if m.get("kv_from") is None:
                kept[p] = self.rms(k.view(T, G, -1)) * self.t(p + "k.norm"), v.view(T, G, -1)
            k, v = kept[p if m.get("kv_from") is None else f"l{m['kv_from']}.mix."]
            o = self.attend(q, k, v, m["scale"] * self.t(p + "temp"))
        elif arch == "Vasanex":
            q, k, v = self.qkv(h, p, m, "qkv")
            q = (self.rms(q) * self.t(p + "q.norm")).view(T, H, -1)
            k, v = (self.rms(k) * self.t(p + "k.norm")).view(T, G, -1), v.view(T, G, -1)
            first = kept.setdefault("values", v)
            v = v if first is v else (1.0 - self.t(p + "vmix")) * v + self.t(p + "vmix") * first
            o = self.attend(self.rotate(q, m["rot"]), self.rotate(k, m["rot"]), v, m["scale"], window=m["mask"]["size"],
                            sink=self.t(p + "sink"))
            return self.linear(o.reshape(T, -1), p + "o") + self.t(p + "o.b")
        else:
            q, k, _ = self.qkv(h, p, m, "qk")
            q, k = q.view(T, H, -1), k.view(T, G, -1)
            o = self.attend(self.rotate(q, m["rot"]), self.rotate(k, m["rot"]), k, m["scale"], window=m["mask"]["size"],
                            first=m["mask"]["keep_first"])
        return self.linear(o.reshape(T, -1), p + "o")

    # ---- feed-forwards
    def unit_ff(self, h, p, dense):
        """One expert, or a dense feed-forward, of the model's kind."""
        arch = self.cfg["architecture"]
        up = self.linear(h, p + "up")
        if arch == "Pubodra":
            z = F.gelu(up, approximate="tanh") if dense else F.relu(up) ** 2
        elif arch == "Kikunex" and dense:
            a, b = F.softplus(self.t(p + "act"))
            z = torch.where(up > 0, a * up * up, (0.5 + b) * (torch.expm1(up.clamp(max=0)) - up.clamp(max=0))) + 0.5 * up
        elif arch == "Kikunex":
            z = F.relu(up) ** 2
        elif arch == "Nogosun":
            z = F.gelu(up)
        elif arch == "Vasanex":
            limit = self.cfg["layers"][0]["mlp"]["limit"]
            gate, up = self.linear(h, p + "gate").clamp(max=limit), up.clamp(-limit, limit)
            z = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
        else:
            gate = self.linear(h, p + "gate")
            z = (F.gelu(gate, approximate="tanh") if arch == "Larupel" and dense else F.silu(gate)) * up
        return self.linear(z, p + "down")

    def feed_forward(self, h, p, mlp):
        if mlp["kind"] == "dense":
            return torch.cat([self.unit_ff(part, p, True) for part in h.split(16384)])
        arch, top = self.cfg["architecture"], mlp["router"]["top"]
        z = self.linear(h, p + "router")
        if arch == "Larupel":
            best = (z + self.t(p + "router.b")).topk(top, -1)
            chosen, share = best.indices, best.values.softmax(-1)
        elif arch == "Kikunex":
            score = torch.sigmoid(z)
            choice, groups = score + self.t(p + "correction"), mlp["router"]["groups"]
            per = choice.view(len(z), groups["count"], -1)
            keep = per.topk(2, -1).values.sum(-1).topk(groups["keep"], -1).indices
            out = torch.ones(per.shape[:2], dtype=torch.bool, device=self.dev).scatter_(1, keep, False)
            chosen = per.masked_fill(out[:, :, None], -math.inf).view_as(z).topk(top, -1).indices
            share = score.gather(1, chosen) * mlp["router"]["scale"]
        else:
            score = torch.sigmoid(z) if arch == "Rununex" else z.softmax(-1)
            share, chosen = score.topk(top, -1)
            if arch == "Pubodra":
                share = share / (share.sum(-1, keepdim=True) + 1e-20)
        y = torch.zeros_like(h)
        for e in range(z.shape[1]):
            row, k = (chosen == e).nonzero(as_tuple=True)
            s = share[row, k][:, None]
            if arch == "Rununex":
                y.index_add_(0, row, self.unit_ff(s * h[row], f"{p}e{e}.", False))
            else:
                y.index_add_(0, row, s * self.unit_ff(h[row], f"{p}e{e}.", False))
        if mlp.get("shared"):
            shared = self.unit_ff(h, p + "shared.", False)
            y = y + (torch.sigmoid(self.linear(h, p + "shared.sg")) * shared if arch == "Larupel" else shared)
        return y

    # ---- models
    def norm(self, x, name):
        arch = self.cfg["architecture"]
        if arch == "Pubodra":
            return torch.tanh(self.t(name + ".alpha") * x) * self.t(name) + self.t(name + ".b")
        if arch in ("Larupel", "Rununex"):
            return self.layer_norm(x, name, bias=arch == "Larupel")
        return self.rms(x) * (self.t(name) + (1.0 if arch == "Vasanex" else 0.0))

    def design(self, rows):
        cfg, arch, kept = self.cfg, self.cfg["architecture"], {}
        x = self.w["embed"][self.ids].to(F64) * float((cfg.get("embedding") or {}).get("scale", 1.0))
        if arch == "Larupel":
            W = x.shape[1]
            angle = self.positions[:, None] * 10000.0 ** (-2.0 * torch.arange(W // 2, device=self.dev, dtype=F64) / W)
            x = x + torch.stack([angle.sin(), angle.cos()], -1).view(-1, W)
        elif arch == "Kikunex":
            x = self.rms(x) * self.t("embed.norm")
        mult = cfg.get("residual_mult", 1.0)
        for i, layer in enumerate(cfg["layers"]):
            p = f"l{i if layer.get('weights_of') is None else layer['weights_of']}."
            h = self.norm(x, p + "norm1")
            if arch == "Kikunex":
                before = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
                before[[a for a, _ in self.spans]] = 0.0
                h = h + (before - h) * self.t(p + "shift")
            y = self.mixer(layer["type"], h, p + "mix.", layer["mixer"], kept)
            if arch == "Nogosun":
                x = x + y + self.feed_forward(self.norm(x, p + "norm2"), p + "mlp.", layer["mlp"])
                continue
            x = x + mult * (self.norm(y, p + "norm1b") if arch == "Larupel" else y)
            y = self.feed_forward(self.norm(x, p + "norm2"), p + "mlp.", layer["mlp"])
            x = x + mult * (self.norm(y, p + "norm2b") if arch == "Larupel" else y)
        x = self.norm(x[rows], "final.norm")
        return self.linear(x, "head" if "head" in self.w else "embed") * float(cfg.get("logit_scale", 1.0))

    def qwen3(self, rows):
        cfg, T = self.cfg, len(self.ids)
        rot = {"dims": cfg["head_dim"], "base": cfg["rope_theta"]}
        x = self.w["model.embed_tokens.weight"][self.ids].to(F64)
        for i in range(cfg["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.rms(x) * self.t(p + "input_layernorm.weight")
            q, k, v = (self.linear(h, f"{p}self_attn.{n}_proj.weight").view(T, -1, cfg["head_dim"]) for n in "qkv")
            q, k = (self.rotate(self.rms(u) * self.t(f"{p}self_attn.{n}_norm.weight"), rot) for u, n in ((q, "q"), (k, "k")))
            x = x + self.linear(self.attend(q, k, v, cfg["head_dim"] ** -0.5).reshape(T, -1), p + "self_attn.o_proj.weight")
            del h, q, k, v
            x = torch.cat([u + self.linear(F.silu(self.linear(z, p + "mlp.gate_proj.weight")) * self.linear(z, p + "mlp.up_proj.weight"),
                                           p + "mlp.down_proj.weight")
                           for u in x.split(16384)
                           for z in (self.rms(u) * self.t(p + "post_attention_layernorm.weight"),)])
        x = self.rms(x[rows]) * self.t("model.norm.weight")
        return self.linear(x, "lm_head.weight" if "lm_head.weight" in self.w else "model.embed_tokens.weight")


def exact(case, seed):
    cfg = config_of(case)
    sequences = tokens_of(case, seed, cfg.get("vocab") or cfg["vocab_size"])
    if work(dict(case, kind="feed", new=0, score=False))["flops"] > 4e14:       # minutes in 64 bits
        return None
    if case["kind"] == "decode":
        steps = [[(r, len(s) - 1, len(s), [0]) for r, s in enumerate(sequences)]]
    else:
        steps = [s for s in schedule(case) if any(want for _, _, _, want in s)]
    model = Exact(cfg, weights_of(cfg, seed), sequences)
    rows = [[model.spans[r][0] + a + place for r, a, _, want in step for place in want] for step in steps]
    forward = model.qwen3 if case["model"] == "qwen3" else model.design
    logits = forward(torch.tensor([row for step in rows for row in step], device="cuda"))
    parts = list(logits.split([len(step) for step in rows]))
    return parts[0] if case["kind"] == "decode" else parts
