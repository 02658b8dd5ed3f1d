"""What the engine's speed is measured on: steps and generations of models this repository's benchmark names, through
``Engine.step``, ``Engine.run`` and ``LLM.generate``, at sizes from one short prompt to dozens of long contexts.

A case is plain numbers.  ``kind`` says what one pass is:

``prompt``    one step that brings whole prompts, the logits of each one's last token wanted; then they are released.
              What a request waits for before its first token.
``decode``    one step of one token each for live requests, as the generation loop launches it (``Engine.run`` on pages
              that are reserved): what a token costs.
``mixed``     the same beside one portion of a longer prompt: what the scheduler makes of requests that arrive while
              others run.
``answer``    prompts in one step, then one step a token; then they are released.  A short answer to short prompts from
              its first launch to its last.  The tokens are given, so that logits can be compared.
``generate``  ``LLM.generate`` in true 32-bit, greedy, with log-probabilities: what the engine's results are checked with.

Lengths of several requests are spread between ``low`` and ``high`` (over their logarithm); the tokens are drawn from the
seed.  The weights are the framework's random ones, the layers of each model repeat, and a case runs a few of them: over
dozens of layers of random weights two correct implementations in bfloat16 drift apart by more than can be told from a fault.
One engine serves all states of a case, as a server's does; a state is its live requests or its prompts.
"""
import gc
import itertools
import math
import weakref

import numpy as np
import torch

from prelude_amd import LLM
from prelude_amd.config import EngineConfig
from prelude_amd.engine import Engine, StepEntry
from prelude_amd.weights import random_tensors_on_device

WEIGHTS_SEED = 0
CHUNK = 2048            # tokens a request's context is filled by at a time
STATES = 4              # states that live at the same time, at most


# ---- the models -------------------------------------------------------------------------------------------------------
def _qwen3(layers, hidden, ff, heads, tied):
    return dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", vocab_size=151936, hidden_size=hidden,
                intermediate_size=ff, num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=8,
                head_dim=128, attention_bias=False, max_position_embeddings=40960, sliding_window=None,
                max_window_layers=layers, tie_word_embeddings=tied, rope_theta=1000000.0, rms_norm_eps=1e-6,
                use_sliding_window=False, hidden_act="silu", eos_token_id=151645)


def _libodra(layers):
    mixer = dict(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, q_rank=768, rot=dict(base=10000.0, dims=64),
                 scale=192 ** -0.5)
    dense = dict(kind="dense", ff=8192, limit=7.0)
    moe = dict(kind="moe", expert=dict(ff=1408), router=dict(experts=64, top=6), shared=dict(ff=2816))
    return dict(architecture="Libodra", vocab=65536, width=2048, norm=dict(eps=1e-6),
                layers=[dict(type="latent_attention", mixer=mixer, mlp=dense if i % 3 == 0 else moe) for i in range(layers)])


def _pogorax(layers):
    dense = dict(kind="dense", ff=5504)
    mamba = dict(heads=64, vdim=64, state=128, groups=8, conv=4, norm_groups=8)
    attention = dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=128 ** -0.5)
    griffin = dict(left=dict(attention, rot=dict(base=1000000.0, dims=64)), right=dict(width=2048, blocks=8, conv=4))
    xlstm = dict(left=dict(attention, mask=dict(size=1024)), right=dict(heads=8, dim=128, vdim=256, gate_cap=15.0))
    period = (("mamba2", mamba, None), ("parallel_2", griffin, dense), ("mamba2", mamba, None), ("parallel", xlstm, dense))
    return dict(architecture="Pogorax", vocab=65536, width=2048, norm=dict(eps=1e-5), embedding=dict(scale=2048 ** 0.5),
                layers=[dict(type=period[i % 4][0], mixer=period[i % 4][1], mlp=period[i % 4][2]) for i in range(layers)])


def _raw(case):
    n = case["layers"]
    return {"qwen3-0.6b": lambda: _qwen3(n, 1024, 3072, 16, True), "qwen3-4b": lambda: _qwen3(n, 2560, 9728, 32, True),
            "qwen3-8b": lambda: _qwen3(n, 4096, 12288, 32, False), "libodra": lambda: _libodra(n),
            "pogorax": lambda: _pogorax(n)}[case["model"]]()


LAYERS = {"qwen3-0.6b": 28, "qwen3-4b": 8, "qwen3-8b": 6, "libodra": 12, "pogorax": 12}


def _case(kind, model, requests, low, high, portion=0, behind=0, new=0, dtype="bfloat16", layers=None, **name):
    return dict(name, kind=kind, model=model, layers=layers or LAYERS[model], dtype=dtype, requests=requests, low=low,
                high=high, portion=portion, behind=behind, new=new)


# ---- the cases --------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one short prompt to a small model: nothing but launches and short kernels
        _case("prompt", "qwen3-0.6b", 1, 128, 128, name="0.6b_prompt_128"),
        # four clients of a small model, short questions and short answers
        _case("answer", "qwen3-0.6b", 4, 128, 128, new=32, name="0.6b_answer_4x128+32"),
        # one interactive user
        _case("decode", "qwen3-4b", 1, 1003, 1003, name="4b_decode_1"),
        # the benchmark's batch: eight users with long contexts
        _case("decode", "qwen3-4b", 8, 4096, 4096, name="4b_decode_8x4096"),
        # a busy server: requests of all lengths
        _case("decode", "qwen3-8b", 48, 61, 4096, name="8b_decode_48_ragged"),
        # the prompt of the request workload, and the benchmark's
        _case("prompt", "qwen3-4b", 1, 512, 512, name="4b_prompt_512"),
        _case("prompt", "qwen3-4b", 1, 2048, 2048, name="4b_prompt_2048"),
        # a portion in the middle of a long prompt beside users who wait for their next token
        _case("mixed", "qwen3-8b", 31, 100, 3000, portion=1500, behind=2500, name="8b_mixed_1500+31"),
        # experts and attention through a latent: a long prompt, and a batch of users
        _case("prompt", "libodra", 1, 2048, 2048, name="libodra_prompt_2048"),
        _case("decode", "libodra", 8, 4096, 4096, name="libodra_decode_8x4096"),
        # recurrences beside attention: several prompts of odd lengths in one step and the first tokens of their answers
        _case("answer", "pogorax", 3, 211, 1303, new=8, name="pogorax_answer_3_ragged+8"),
        # the 32-bit engine, through the Python entry point
        _case("generate", "qwen3-0.6b", 3, 25, 150, new=6, dtype="float32", name="0.6b_f32_generate_3"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "decode", "decode", "mixed", "answer", "generate"])
    if kind == "prompt":
        n = rng.choice([1, 1, 2, 3])
        high = _log(rng, 16, 2048 // n)
        return _case(kind, rng.choice(["qwen3-0.6b", "qwen3-4b", "qwen3-8b", "libodra", "pogorax"]), n, max(2, high // rng.randint(1, 4)), high)
    if kind == "decode":
        n = _log(rng, 1, 48)
        high = _log(rng, 64, 4096)
        return _case(kind, rng.choice(["qwen3-0.6b", "qwen3-4b", "qwen3-8b", "libodra"]), n, max(16, high // rng.randint(1, 16)), high)
    if kind == "mixed":
        high = _log(rng, 64, 3000)
        return _case(kind, rng.choice(["qwen3-4b", "qwen3-8b", "libodra"]), _log(rng, 1, 31), max(16, high // rng.randint(1, 16)), high,
                     portion=_log(rng, 16, 1500), behind=_log(rng, 16, 2500))
    if kind == "answer":
        high = _log(rng, 16, 400)
        return _case(kind, rng.choice(["qwen3-0.6b", "pogorax"]), rng.randint(1, 5), max(2, high // rng.randint(1, 4)), high, new=rng.randint(2, 32))
    high = _log(rng, 16, 150)
    return _case(kind, "qwen3-0.6b", rng.randint(1, 3), max(2, high // rng.randint(1, 6)), high, new=rng.randint(1, 6), dtype="float32")


def _lengths(case):
    """The requests' lengths: spread between low and high, in no order."""
    n, lo, hi = case["requests"], case["low"], case["high"]
    if n == 1:
        return [hi]
    order = sorted(range(n), key=lambda i: (i * 0.6180339887) % 1.0)
    return [int(round(lo * (hi / lo) ** (order[i] / (n - 1)))) for i in range(n)]


def _vocab(case):
    return 151936 if case["model"].startswith("qwen3") else 65536


def _inputs(case, seed):
    """Every request's tokens from its first on; the portion's request, where there is one, last."""
    rng = np.random.default_rng(seed)
    lengths = _lengths(case)
    extra = {"decode": 1, "mixed": 1, "answer": max(case["new"] - 1, 0)}.get(case["kind"], 0)
    sizes = [n + extra for n in lengths]
    if case["kind"] == "mixed":
        sizes.append(case["behind"] + case["portion"])
    return [rng.integers(0, _vocab(case), size=n).tolist() for n in sizes]


# ---- the engine: one at a time ------------------------------------------------------------------------------------------
_held = {}
_ids = itertools.count()


def _let_go():
    gc.collect()
    torch.cuda.empty_cache()


def _engine(case):
    pages = sum(-(-len(t) // 16) + 1 for t in _inputs(case, 0)) + case["requests"] * (1 + case["new"] // 16)
    slots = STATES * (case["requests"] + 1)
    which = (case["model"], case["layers"], case["dtype"])
    if _held.get("model") != which:
        _held.clear()
        _let_go()
    if _held.get("size") != (pages, slots):
        config = EngineConfig(dtype=case["dtype"], max_cache_tokens=STATES * pages * 16, max_state_slots=slots)
        old = _held.pop("engine", None)
        engine = Engine.from_config(_raw(case), config, seed=WEIGHTS_SEED) if old is None else Engine(old.model, config, old.raw_config)
        del old
        _let_go()
        _held.update(model=which, size=(pages, slots), engine=engine)
    return _held["engine"]


class State:
    """A case's requests on the engine; what they hold goes back with it."""

    def __init__(self, case, seed):
        self.case = case
        self.engine = _engine(case)
        self.tokens = _inputs(case, seed)
        self.ids = [next(_ids) for _ in self.tokens]
        weakref.finalize(self, _release, self.engine, list(self.ids))


def _release(engine, ids):
    for i in ids:
        engine.release(i)


def prepare(case, seed):
    state = State(case, seed)
    engine = state.engine
    if case["kind"] == "generate":
        state.llm = LLM.from_engine(engine)
    if case["kind"] in ("decode", "mixed"):
        state.starts = [len(t) - 1 for t in state.tokens]
        if case["kind"] == "mixed":
            state.starts[-1] = case["behind"]
        for i, tokens, start in zip(state.ids, state.tokens, state.starts):
            for at in range(0, start, CHUNK):
                engine.step([StepEntry(i, tokens[at:min(start, at + CHUNK)], [])])
            engine.tables.reserve(i, len(tokens))
    return state


def run(state):
    case, engine, tokens = state.case, state.engine, state.tokens
    kind = case["kind"]
    if kind in ("decode", "mixed"):
        entries = [StepEntry(i, t[s:], [len(t) - s - 1]) for i, t, s in zip(state.ids, tokens, state.starts)]
        return engine.run(entries, state.starts)
    if kind == "prompt":
        logits = engine.step([StepEntry(i, t, [len(t) - 1]) for i, t in zip(state.ids, tokens)])
        _release(engine, state.ids)
        return logits
    if kind == "answer":
        lengths = _lengths(case)
        out = [engine.step([StepEntry(i, t[:n], [n - 1]) for i, t, n in zip(state.ids, tokens, lengths)])]
        for j in range(case["new"] - 1):
            out.append(engine.step([StepEntry(i, t[n + j:n + j + 1], [0]) for i, t, n in zip(state.ids, tokens, lengths)]))
        _release(engine, state.ids)
        return out
    results = state.llm.generate(tokens, max_tokens=case["new"], temperature=0.0, logprobs=0)
    return {"tokens": [np.array(r.token_ids) for r in results], "logprobs": [np.array(r.token_logprobs) for r in results]}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------
def _sizes(case):
    """(matrix elements every token goes through in one layer of each kind with their counts, attention and cache sizes)."""
    raw, n = _raw(case), case["layers"]
    if case["model"].startswith("qwen3"):
        h, f, heads = raw["hidden_size"], raw["intermediate_size"], raw["num_attention_heads"]
        per = (heads + 16) * 128 * h + heads * 128 * h + 3 * h * f
        return dict(matrices=n * per, experts=0, attention=[(n, heads, 128, 128, None)], cached=n * 2 * 8 * 128, state=0, width=h)
    if case["model"] == "libodra":
        dense = -(-n // 3)
        per = 2048 * 768 + 768 * 16 * 192 + 2048 * 576 + 512 * 16 * 256 + 2048 * 2048
        return dict(matrices=n * per + dense * 3 * 2048 * 8192 + (n - dense) * 2 * 2048 * 2816, experts=n - dense,
                    attention=[(n, 16, 192, 128, None)], cached=n * 576, state=0, width=2048)
    m, g, x = -(-n // 2), (n + 2) // 4, n // 4
    att = 2048 * (2048 + 512 + 512) + 2048 * 2048
    matrices = m * (2048 * (2 * 4096 + 2048 + 64) + 4096 * 2048) + g * (att + 3 * 2048 * 2048 + 2 * 2048 * 256) \
        + x * (att + 2048 * 2048 + 2048 * (2 * 1024 + 2 * 2048 + 16) + 2048 * 2048) + (g + x) * 3 * 2048 * 5504
    return dict(matrices=matrices, experts=0, attention=[(g, 16, 128, 128, None), (x, 16, 128, 128, 1024)],
                cached=(g + x) * 2 * 4 * 128, state=m * 64 * 64 * 128 + x * 8 * 128 * 256, width=2048)


def _step_work(case, spans, rows):
    """One step: ``spans`` are (first position, tokens) of its requests, ``rows`` the logits wanted."""
    s, el, vocab = _sizes(case), 4 if case["dtype"] == "float32" else 2, _vocab(case)
    tokens = sum(n for _, n in spans)
    bytes_ = s["matrices"] * el + vocab * s["width"] * el + rows * vocab * 4 + tokens * s["width"] * el
    flops = 2.0 * s["matrices"] * tokens + 2.0 * vocab * s["width"] * rows
    if s["experts"]:
        touched = 64 * (1 - (1 - 6 / 64) ** tokens)
        bytes_ += s["experts"] * touched * 2 * 2048 * 1408 * el
        flops += s["experts"] * tokens * 6 * 2 * 2 * 2048 * 1408
    for start, n in spans:
        bytes_ += (start + n) * s["cached"] * el + 2 * 4 * s["state"] * (0.5 if start == 0 else 1)
        flops += 6.0 * n * s["state"]
        for layers, heads, dim, vdim, chunk in s["attention"]:
            seen = n * start + n * (n + 1) / 2.0 if chunk is None else n * chunk / 2.0
            flops += 2.0 * layers * heads * (dim + vdim) * seen
    return bytes_, flops


def work(case):
    lengths, kind = _lengths(case), case["kind"]
    if kind == "decode":
        steps = [([(n, 1) for n in lengths], len(lengths))]
    elif kind == "mixed":
        steps = [([(n, 1) for n in lengths] + [(case["behind"], case["portion"])], len(lengths) + 1)]
    else:
        steps = [([(0, n) for n in lengths], len(lengths))]
        steps += [([(n + j, 1) for n in lengths], len(lengths)) for j in range(max(case["new"], 1) - 1)]
    parts = [_step_work(case, *s) for s in steps]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """Measured: bfloat16 logits of the same tokens in other portions differ by up to 0.020 of their size (0.12 of their
    root mean square at one place), and lie 0.009 to 0.022 off the 64-bit ones; 32-bit log-probabilities lie 1e-7 off."""
    if case["dtype"] == "float32":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    return {"rel": 0.03, "max": 0.5}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------
def _rms(x, w, eps):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


class _Weights(dict):
    def mul(self, x, name):
        return x @ self[name].double().T


def _spans(lengths):
    at = 0
    for n in lengths:
        yield slice(at, at + n)
        at += n


def _attend(q, k, v, scale, sink=None, chunk=None):
    """q [T, H, d], k [T, G, d], v [T, G, e] of one sequence, causal; ``chunk``: keys of the query's own chunk only."""
    n, heads, group = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    out = torch.empty(n, heads, v.shape[2], dtype=q.dtype, device=q.device)
    at = torch.arange(n, device=q.device)
    see = at[:, None] >= at[None, :]
    if chunk:
        see &= (at[:, None] // chunk) == (at[None, :] // chunk)
    for h in range(heads):
        s = (q[:, h] @ k[:, h // group].T).mul_(scale).masked_fill_(~see, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].double().expand(n, 1)], dim=1)
        out[:, h] = torch.softmax(s, dim=-1)[:, :n] @ v[:, h // group]
    return out.reshape(n, -1)


def _positions(lengths, device):
    return torch.cat([torch.arange(n, device=device) for n in lengths])


def _exact_qwen3(raw, w, x, lengths, tokens):
    eps, heads = raw["rms_norm_eps"], raw["num_attention_heads"]
    n = x.shape[0]
    inv = 1.0 / (torch.tensor(raw["rope_theta"], dtype=torch.float64).pow(torch.arange(0, 128, 2, dtype=torch.float64) / 128)).float()
    angle = (_positions(lengths, x.device).float()[:, None] * inv.to(x.device)[None, :]).double()[:, None, :]
    cos, sin = torch.cos(angle), torch.sin(angle)

    def turned(z, name):
        z = _rms(z.reshape(n, -1, 128), w[name].double(), eps)
        a, b = z[..., :64], z[..., 64:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for i in range(raw["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _rms(x, w[p + "input_layernorm.weight"].double(), eps)
        q = turned(w.mul(h, p + "self_attn.q_proj.weight"), p + "self_attn.q_norm.weight")
        k = turned(w.mul(h, p + "self_attn.k_proj.weight"), p + "self_attn.k_norm.weight")
        v = w.mul(h, p + "self_attn.v_proj.weight").reshape(n, -1, 128)
        o = torch.cat([_attend(q[s], k[s], v[s], 128 ** -0.5) for s in _spans(lengths)])
        x = x + w.mul(o, p + "self_attn.o_proj.weight")
        h = _rms(x, w[p + "post_attention_layernorm.weight"].double(), eps)
        g = w.mul(h, p + "mlp.gate_proj.weight")
        x = x + w.mul(g * torch.sigmoid(g) * w.mul(h, p + "mlp.up_proj.weight"), p + "mlp.down_proj.weight")
    return _rms(x, w["model.norm.weight"].double(), eps)


def _turn_pairs(x, positions, rot):
    """The first dims of the last axis in pairs (2i, 2i + 1); x [T, heads, d]."""
    dims = rot["dims"]
    f = float(rot["base"]) ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=x.device) / dims)
    angle = positions.double()[:, None, None] * f
    c, s = torch.cos(angle), torch.sin(angle)
    out = x.clone()
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    out[..., 0:dims:2], out[..., 1:dims:2] = u * c - v * s, v * c + u * s
    return out


def _exact_libodra(raw, w, x, lengths, tokens):
    eps, n = raw["norm"]["eps"], x.shape[0]
    positions = _positions(lengths, x.device)
    for i, layer in enumerate(raw["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        h = _rms(x, 1.0 + w[p + "norm1"].double(), eps)
        q = w.mul(_rms(w.mul(h, p + "mix.dq"), w[p + "mix.dq.norm"].double(), eps), p + "mix.uq").reshape(n, 16, 192)
        low = w.mul(h, p + "mix.dkv")
        c = _rms(low[:, :512], w[p + "mix.dkv.norm"].double(), eps)
        shared = _turn_pairs(low[:, None, 512:], positions, m["rot"]).expand(n, 16, 64)
        k = torch.cat([w.mul(c, p + "mix.uk").reshape(n, 16, 128), shared], -1)
        q = torch.cat([q[..., :128], _turn_pairs(q[..., 128:].contiguous(), positions, m["rot"])], -1)
        v = w.mul(c, p + "mix.uv").reshape(n, 16, 128)
        o = torch.cat([_attend(q[s], k[s], v[s], m["scale"], w[p + "mix.sink"]) for s in _spans(lengths)])
        x = x + w.mul(o, p + "mix.o")
        h = _rms(x, 1.0 + w[p + "norm2"].double(), eps)
        if f["kind"] == "dense":
            g = w.mul(h, p + "mlp.gate").clamp(max=f["limit"])
            u = w.mul(h, p + "mlp.up").clamp(min=-f["limit"], max=f["limit"])
            x = x + w.mul(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "mlp.down")
            continue
        top, chosen = f["router"]["top"], w[p + "mlp.table"][tokens]
        y = w.mul(w.mul(h, p + "mlp.shared.up").relu().square(), p + "mlp.shared.down")
        for e in range(f["router"]["experts"]):
            mine = (chosen == e).any(dim=1).nonzero()[:, 0]
            if mine.numel():
                y[mine] += w.mul(w.mul(h[mine], f"{p}mlp.e{e}.up").relu().square(), f"{p}mlp.e{e}.down") / top
        x = x + y
    return _rms(x, 1.0 + w["final.norm"].double(), eps)


def _conv(x, w, b):
    taps = w.shape[1]
    padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    return sum(padded[j:j + x.shape[0]] * w[:, j].double() for j in range(taps)) + b.double()


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _mamba2(h, w, p, m, eps):
    heads, dv, size, groups, n = m["heads"], m["vdim"], m["state"], m["groups"], h.shape[0]
    inner = heads * dv
    z, xbc, dt = w.mul(h, p + "in").split([inner, inner + 2 * groups * size, heads], dim=1)
    xbc = torch.nn.functional.silu(_conv(xbc, w[p + "conv"], w[p + "conv.b"]))
    x, b, c = xbc.split([inner, groups * size, groups * size], dim=1)
    x = x.reshape(n, heads, dv)
    b, c = (a.reshape(n, groups, size).repeat_interleave(heads // groups, dim=1) for a in (b, c))
    dt = torch.nn.functional.softplus(dt + w[p + "dt_bias"].double())
    keep = torch.exp(-torch.exp(w[p + "A_log"].double()) * dt)[:, :, None, None]
    add = dt[:, :, None] * b
    state, y = x.new_zeros(heads, size, dv), torch.empty_like(x)
    for t in range(n):
        state = torch.addcmul(keep[t] * state, add[t][:, :, None], x[t][:, None, :])
        y[t] = (state * c[t][:, :, None]).sum(1)
    y = (y + w[p + "D"].double()[:, None] * x).reshape(n, inner) * torch.nn.functional.silu(z)
    y = _rms(y.reshape(n, m["norm_groups"], -1), None, eps).reshape(n, inner) * w[p + "norm"].double()
    return w.mul(y, p + "o")


def _mlstm(h, w, p, m, eps):
    heads, d, dv, cap, n = m["heads"], m["dim"], m["vdim"], m["gate_cap"], h.shape[0]
    q = w.mul(h, p + "q").reshape(n, heads, d) * d ** -0.5
    k, v = w.mul(h, p + "k").reshape(n, heads, d), w.mul(h, p + "v").reshape(n, heads, dv)
    i = cap * torch.tanh((w.mul(h, p + "i") + w[p + "i.b"].double()) / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh((w.mul(h, p + "f") + w[p + "f.b"].double()) / cap))
    s, z, top = h.new_zeros(heads, d, dv), h.new_zeros(heads, d), h.new_zeros(heads)
    o = torch.empty_like(v)
    for t in range(n):
        new = torch.maximum(f[t] + top, i[t])
        keep, add = torch.exp(f[t] + top - new), torch.exp(i[t] - new)
        s = torch.addcmul(keep[:, None, None] * s, (add[:, None] * k[t])[:, :, None], v[t][:, None, :])
        z, top = torch.addcmul(keep[:, None] * z, add[:, None], k[t]), new
        den = torch.maximum((z * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        o[t] = (s * q[t][:, :, None]).sum(1) / den[:, None]
    o = _rms(o, None, eps).reshape(n, -1) * w[p + "norm"].double() * torch.sigmoid(w.mul(h, p + "g"))
    return w.mul(o, p + "o")


def _griffin(h, w, p, m):
    y = _gelu(w.mul(h, p + "y") + w[p + "y.b"].double())
    u = _conv(w.mul(h, p + "x") + w[p + "x.b"].double(), w[p + "conv"], w[p + "conv.b"])
    parts = u.reshape(u.shape[0], m["blocks"], -1)

    def gate(name):
        g = torch.stack([parts[:, a] @ w[p + name][a].double().T for a in range(m["blocks"])], 1) + w[p + name + ".b"].double()
        return torch.sigmoid(g).reshape(u.shape)

    log_a = -8.0 * gate("ra") * torch.nn.functional.softplus(w[p + "lam"].double())
    a, add = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * gate("ri") * u
    state, out = u.new_zeros(u.shape[1]), torch.empty_like(u)
    for t in range(u.shape[0]):
        state = torch.addcmul(add[t], a[t], state)
        out[t] = state
    return w.mul(out * y, p + "o")


def _exact_pogorax(raw, w, x, lengths, tokens):
    eps = raw["norm"]["eps"]
    x = x * raw["embedding"]["scale"]
    for i, layer in enumerate(raw["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        normed = _rms(x, w[p + "norm1"].double(), eps)
        out = []
        for s in _spans(lengths):
            h = normed[s]
            if layer["type"] == "mamba2":
                out.append(_mamba2(h, w, p + "mix.", m, eps))
                continue
            n, a, l, r = h.shape[0], m["left"], p + "mix.left.", p + "mix.right."
            q, k, v = w.mul(h, l + "q").reshape(n, -1, 128), w.mul(h, l + "k").reshape(n, -1, 128), w.mul(h, l + "v").reshape(n, -1, 128)
            if "rot" in a:
                q, k = (_rms(_turn_pairs(z, torch.arange(n, device=z.device), a["rot"]), None, eps) for z in (q, k))
            o = _attend(q, k, v, a["scale"], chunk=a.get("mask", {}).get("size"))
            if "mask" in a:
                o = o * torch.sigmoid(w.mul(h, l + "g"))
            o = w.mul(o, l + "o")
            other = _mlstm(h, w, r, m["right"], eps) if layer["type"] == "parallel" else _griffin(h, w, r, m["right"])
            out.append(0.5 * (_rms(o, w[l + "out"].double(), eps) + _rms(other, w[r + "out"].double(), eps)))
        x = x + torch.cat(out)
        if layer["mlp"]:
            h = _rms(x, w[p + "norm2"].double(), eps)
            x = x + w.mul(_gelu(w.mul(h, p + "mlp.gate")) * w.mul(h, p + "mlp.up"), p + "mlp.down")
    return _rms(x, w["final.norm"].double(), eps)


_FORWARD = {"qwen3-0.6b": _exact_qwen3, "qwen3-4b": _exact_qwen3, "qwen3-8b": _exact_qwen3, "libodra": _exact_libodra,
            "pogorax": _exact_pogorax}


def _exact_logits(case, w, sequences, wanted):
    """Logits in 64 bits at the positions ``wanted[i]`` of ``sequences[i]``, one tensor [positions, vocab] each."""
    raw = _raw(case)
    lengths = [len(t) for t in sequences]
    tokens = torch.tensor([t for seq in sequences for t in seq], device="cuda")
    qwen = case["model"].startswith("qwen3")
    embed = w["model.embed_tokens.weight" if qwen else "embed"]
    x = _FORWARD[case["model"]](raw, w, embed[tokens].double(), lengths, tokens)
    head = ("model.embed_tokens.weight" if raw.get("tie_word_embeddings") else "lm_head.weight") if qwen else "head"
    rows = torch.cat([x[s][list(at)] for s, at in zip(_spans(lengths), wanted)])
    return w.mul(rows, head).split([len(at) for at in wanted])


def exact(case, seed):
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    w = _Weights(random_tensors_on_device(_raw(case), WEIGHTS_SEED, "cuda", dtype=dtype))
    tokens, kind = _inputs(case, seed), case["kind"]
    with torch.no_grad():
        if kind in ("decode", "mixed", "prompt"):
            return torch.cat(_exact_logits(case, w, tokens, [[len(t) - 1] for t in tokens]))
        lengths = _lengths(case)
        if kind == "answer":
            got = _exact_logits(case, w, tokens, [range(n - 1, len(t)) for t, n in zip(tokens, lengths)])
            return list(torch.stack(list(got), dim=1))
        logprobs = [[] for _ in tokens]
        for _ in range(case["new"]):
            rows = torch.log_softmax(torch.cat(_exact_logits(case, w, tokens, [[len(t) - 1] for t in tokens])), -1)
            for seq, out, row in zip(tokens, logprobs, rows):
                seq.append(int(row.argmax()))
                out.append(float(row.max()))
        return {"tokens": None, "logprobs": [np.array(r) for r in logprobs]}
