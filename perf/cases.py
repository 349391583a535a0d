"""The work that users of this library have it do, as cases that can be timed and checked.

Three kinds of call, all through the public entry points:

  prompt  the prompts of one or more sequences in one `Engine.step`, logits of each last token; with `held`, new
          turns of conversations that already hold that many tokens (rolled back behind the call)
  decode  a conversation's next tokens: a `DecodeSession` bound to sequences that hold their context, a few steps
          launched one ahead of the tokens' collection as the generation loop does it, rolled back behind the call
  reply   prompts and decode steps of new sequences, for a design whose state cannot be rolled back

Models: the Qwen2 decoder at the sizes that `bench.py` names (the library's main path, bfloat16; the 32-bit run type at
the smallest size), and the Rofizen design at the benchmark's small size (linear attention, a matrix memory, sloped
attention, experts picked by a table).  Designs whose router chooses experts by a score are not among them: a score near
a tie may rightly go either way, so two correct runs differ by a whole expert; their kernels are the same ones.

Weights are random at the scales of a freshly initialised model (the matrices that add into the stream a factor of
sqrt(2 layers) smaller, embedding rows of size one), with one thing that a trained model has: the next token is
clear.  The head's row of token (t + hop) mod vocabulary carries a share of the embedding row of t (a tied head does it
by itself, with hop 0), so that the sampled tokens do not hang on the last bit of a logit.  Prompts are uniform over
the vocabulary.
"""
import math
import random
import zlib

import torch

from minfer_amd import DecoderModel, Engine, Sampler, SamplingParams, config_from_dict

_BASE = dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", hidden_act="silu", rope_theta=1000000.0, rms_norm_eps=1e-6,
             max_position_embeddings=32768, use_sliding_window=False)


def _qwen2(layers, width, heads, kv_heads, ff, vocab, tied):
    return dict(_BASE, num_hidden_layers=layers, hidden_size=width, num_attention_heads=heads, num_key_value_heads=kv_heads,
                intermediate_size=ff, vocab_size=vocab, tie_word_embeddings=tied)


_QWEN2 = {
    "0.5b": _qwen2(24, 896, 14, 2, 4864, 151936, True),
    "1.5b": _qwen2(28, 1536, 12, 2, 8960, 151936, True),
    "3b": _qwen2(36, 2048, 16, 2, 11008, 151936, True),
    "7b": _qwen2(28, 3584, 28, 4, 18944, 152064, False),
}


def _rofizen(width=2048, layers=4, heads=16, ff=8192, dim=128, experts=8, rank=16, vocab=32768):
    gla = dict(type="gla", mixer=dict(heads=heads, dim=dim, vdim=dim, tau=16.0, rank=rank))
    ret = dict(type="retention", mixer=dict(heads=heads, dim=dim, vdim=dim, rot=dict(base=10000.0, dims=dim),
                                            decay=[1.0 - 2.0 ** (-5.0 - 3.0 * h / (heads - 1)) for h in range(heads)]))
    both = dict(type="parallel", mixer=dict(
        left=dict(heads=heads, kv_heads=heads // 4, dim=dim, vdim=dim, scale=dim ** -0.5, softcap=50.0,
                  q_temp=dict(coef=0.5, every=1024)),
        right=dict(heads=heads, dim=dim, vdim=dim, gate_cap=15.0)))
    routed = dict(kind="moe", expert=dict(ff=ff // 2), router=dict(experts=experts, top=1), shared=dict(ff=ff // 2))
    return dict(architecture="Rofizen", vocab=vocab, width=width, norm=dict(eps=1e-6), embedding=dict(scale=width ** 0.5),
                postln_alpha=(2.0 * layers) ** 0.25,
                layers=[dict((gla, both, ret, both)[i % 4], mlp=dict(kind="dense", ff=ff) if i % 4 == 0 else routed)
                        for i in range(layers)])


_ROFIZEN = {"rofizen": _rofizen()}
_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


# ------------------------------------------------------------------ the cases
def _prompt(model, batch, longest, held=0, dtype="bf16"):
    return dict(kind="prompt", model=model, dtype=dtype, batch=batch, longest=longest, held=held)


def _decode(model, batch, longest, steps, sampling="greedy", dtype="bf16"):
    return dict(kind="decode", model=model, dtype=dtype, batch=batch, longest=longest, steps=steps, sampling=sampling)


def _reply(batch, longest, steps):
    return dict(kind="reply", model="rofizen", dtype="bf16", batch=batch, longest=longest, steps=steps)


def listed():
    return [
        # one user, the smallest model, the library's default sampling (penalty, top-k, top-p): latency and launches
        dict(_decode("0.5b", 1, 150, 24, "default"), name="0.5b reply of one"),
        # the first token after a one-line question
        dict(_prompt("0.5b", 1, 37), name="0.5b prompt 37"),
        # the 32-bit run type: a reference run to compare others with
        dict(_prompt("0.5b", 1, 611, dtype="fp32"), name="0.5b prompt 611 fp32"),
        # a chat turn: a paragraph
        dict(_prompt("7b", 1, 203), name="7b prompt 203"),
        # the benchmark's prompt
        dict(_prompt("7b", 1, 2048), name="7b prompt 2048"),
        # a server's step: unequal prompts that arrived together
        dict(_prompt("7b", 8, 1500), name="7b prompts of 8"),
        # a document
        dict(_prompt("7b", 1, 12001), name="7b prompt 12001"),
        # new turns of conversations that hold thousands of tokens
        dict(_prompt("3b", 4, 180, held=5000), name="3b turns on 5000"),
        # the benchmark's decode step
        dict(_decode("7b", 8, 2048, 16), name="7b decode of 8"),
        # a busy server
        dict(_decode("7b", 64, 1024, 8), name="7b decode of 64"),
        # another design: recurrences, sloped attention, experts; its prompt and its short replies
        dict(_prompt("rofizen", 1, 2048), name="rofizen prompt 2048"),
        dict(_reply(8, 96, 32), name="rofizen replies of 8"),
    ]


def _spread(rng, low, high):
    """A whole number between the two, spread over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    while True:
        kind = rng.choice(("prompt", "prompt", "prompt", "decode", "decode", "rofizen"))
        if kind == "prompt":
            dtype = "fp32" if rng.random() < 0.1 else "bf16"
            model = rng.choice(("0.5b", "1.5b") if dtype == "fp32" else tuple(_QWEN2))
            batch = rng.choice((1, 1, 1, 2, 3, 5, 8))
            longest = _spread(rng, 20, 1000 if dtype == "fp32" else 12001)
            held = _spread(rng, 100, 5000) if rng.random() < 0.25 else 0
            case = _prompt(model, batch, longest, held, dtype)
        elif kind == "decode":
            case = _decode(rng.choice(tuple(_QWEN2)), _spread(rng, 1, 64), _spread(rng, 30, 4000), rng.choice((8, 16, 24)),
                           rng.choice(("greedy", "default")))
        elif rng.random() < 0.5:
            case = _prompt("rofizen", rng.choice((1, 1, 2, 5)), _spread(rng, 20, 3000))
        else:
            case = _reply(_spread(rng, 1, 16), _spread(rng, 20, 300), rng.choice((16, 32)))
        w = work(case)
        new = sum(_lengths(case))
        if case["dtype"] == "fp32" and w["flops"] > 3e12:
            continue
        if case["kind"] != "decode" and new > 12001:
            continue
        if case["kind"] == "decode" and (new > 34000 or w["bytes"] > 2.5e11):
            continue
        return case


def _lengths(case):
    """New tokens of each sequence (decode: context of each), the longest first, the others anything below."""
    rng = random.Random(case["batch"] * 100003 + case["longest"])
    return [case["longest"]] + [rng.randint(max(1, case["longest"] // 16), case["longest"]) for _ in range(case["batch"] - 1)]


# ------------------------------------------------------------------ weights and prompts
def _raw(case):
    return _QWEN2.get(case["model"]) or _ROFIZEN[case["model"]]


def _hop(raw):
    return 0 if raw.get("tie_word_embeddings") else 1021


def _vocab(raw):
    return raw.get("vocab_size") or raw["vocab"]


def _qwen2_tensors(c):
    """name -> (shape, scale, offset) of values scale * normal + offset."""
    h, ff, hd = c["hidden_size"], c["intermediate_size"], c["hidden_size"] // c["num_attention_heads"]
    kv, small = c["num_key_value_heads"] * hd, 0.02 / math.sqrt(2 * c["num_hidden_layers"])
    # a tied head sees rows of size one: the last norm's gain brings the logits to the size they have in earnest
    last = 2.4 / math.sqrt(h) if c["tie_word_embeddings"] else 1.0
    out = {"model.embed_tokens.weight": ((c["vocab_size"], h), 1.0, 0.0), "model.norm.weight": ((h,), 0.05 * last, last)}
    if not c["tie_word_embeddings"]:
        out["lm_head.weight"] = ((c["vocab_size"], h), 0.04, 0.0)
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        for n, rows in (("q", h), ("k", kv), ("v", kv)):
            out[f"{p}self_attn.{n}_proj.weight"] = ((rows, h), 0.02, 0.0)
            out[f"{p}self_attn.{n}_proj.bias"] = ((rows,), 0.02, 0.0)
        out[p + "self_attn.o_proj.weight"] = ((h, h), small, 0.0)
        out[p + "mlp.gate_proj.weight"] = out[p + "mlp.up_proj.weight"] = ((ff, h), 0.02, 0.0)
        out[p + "mlp.down_proj.weight"] = ((h, ff), small, 0.0)
        out[p + "input_layernorm.weight"] = out[p + "post_attention_layernorm.weight"] = ((h,), 0.05, 1.0)
    return out


def _rofizen_tensors(c):
    h, out = c["width"], {}

    def matrix(name, rows, cols, factor=1.0):
        out[name] = ((rows, cols), factor / math.sqrt(cols), 0.0)

    def gains(name, n):
        out[name] = ((n,), 0.05, 1.0)

    matrix("head", c["vocab"], h)
    out["embed"] = ((c["vocab"], h), 1.0 / c["embedding"]["scale"], 0.0)
    gains("final.norm", h)

    def experts(stem, ff):
        matrix(stem + ".gate", ff, h)
        matrix(stem + ".up", ff, h)
        matrix(stem + ".down", h, ff, 0.5)

    for i, layer in enumerate(c["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        gains(p + "norm1", h)
        gains(p + "norm2", h)
        if layer["type"] != "parallel":
            keys, values = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            for n, rows in (("q", keys), ("k", keys), ("v", values), ("g", values)):
                matrix(f"{p}mix.{n}", rows, h)
            matrix(p + "mix.o", h, values, 0.5)
            if layer["type"] == "gla":
                matrix(p + "mix.a1", m["rank"], h)
                matrix(p + "mix.a2", keys, m["rank"])
                out[p + "mix.a2.b"] = ((keys,), 0.3, 0.0)
                gains(p + "mix.norm", m["vdim"])
        else:
            lf, rg = m["left"], m["right"]
            for n, rows in (("q", lf["heads"] * lf["dim"]), ("k", lf["kv_heads"] * lf["dim"]), ("v", lf["kv_heads"] * lf["vdim"])):
                matrix(f"{p}mix.left.{n}", rows, h)
                out[f"{p}mix.left.{n}.b"] = ((rows,), 0.3, 0.0)
            gains(p + "mix.left.q.norm", lf["heads"] * lf["dim"])
            gains(p + "mix.left.k.norm", lf["kv_heads"] * lf["dim"])
            matrix(p + "mix.left.o", h, lf["heads"] * lf["vdim"], 0.5)
            out[p + "mix.left.o.b"] = ((h,), 0.02, 0.0)
            keys, values = rg["heads"] * rg["dim"], rg["heads"] * rg["vdim"]
            for n, rows in (("q", keys), ("k", keys), ("v", values), ("g", values), ("i", rg["heads"]), ("f", rg["heads"])):
                matrix(f"{p}mix.right.{n}", rows, h)
            out[p + "mix.right.i.b"] = ((rg["heads"],), 0.3, 0.0)
            out[p + "mix.right.f.b"] = ((rg["heads"],), 0.3, 3.0)          # a memory that keeps
            gains(p + "mix.right.norm", values)
            matrix(p + "mix.right.o", h, values, 0.5)
            out[p + "mix.left.out"] = out[p + "mix.right.out"] = ((h,), 0.02, 0.5)
        if f["kind"] == "dense":
            matrix(p + "mlp.up", f["ff"], h)
            matrix(p + "mlp.down", h, f["ff"], 0.5)
        else:
            for e in range(f["router"]["experts"]):
                experts(f"{p}mlp.e{e}", f["expert"]["ff"])
            experts(p + "mlp.shared", f["shared"]["ff"])
            matrix(p + "mlp.shared.sg", 1, h)
            out[p + "mlp.table"] = ((c["vocab"], f["router"]["top"]), None, f["router"]["experts"])
    return out


class _Weights:
    """The model's tensors by name, made on the GPU when asked for: rounded to bfloat16, in the run type."""

    def __init__(self, case, seed):
        self.raw, self.seed, self.dtype = _raw(case), seed, _DTYPES[case["dtype"]]
        self.rofizen = case["model"] in _ROFIZEN
        self.tensors = _rofizen_tensors(self.raw) if self.rofizen else _qwen2_tensors(self.raw)

    def _draw(self, name):
        shape, scale, offset = self.tensors[name]
        gen = torch.Generator(device="cuda")
        gen.manual_seed(((self.seed & 0x7FFFFFFF) << 32) ^ zlib.crc32(name.encode()))
        if scale is None:
            return torch.randint(0, offset, shape, generator=gen, device="cuda", dtype=torch.int32)
        t = torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16).mul_(scale)
        return t.add_(offset) if offset else t

    def get(self, name):
        t = self._draw(name)
        if name in ("lm_head.weight", "head"):
            table = self._draw("embed" if self.rofizen else "model.embed_tokens.weight")
            share = 0.02 if not self.rofizen else 0.012 * self.raw["embedding"]["scale"]
            t.add_(torch.roll(table, _hop(self.raw), 0), alpha=share)
        return t.to(self.dtype) if t.is_floating_point() else t


def _tokens(case, seed, vocab):
    rng = torch.Generator().manual_seed(seed * 7919 + 17)
    take = lambda n: torch.randint(0, vocab, (n,), generator=rng).tolist()  # noqa: E731
    new = [take(n) for n in _lengths(case)]
    held = [take(case["held"] - 3 * i) for i in range(case["batch"])] if case.get("held") else None
    start = [take(1)[0] for _ in new]                # decode: the token that each sequence goes on from
    return new, held, start


def _next(token, raw):
    return (token + _hop(raw)) % _vocab(raw)


def _params(case):
    return SamplingParams() if case["sampling"] == "default" else SamplingParams.greedy()


# ------------------------------------------------------------------ what a program has in hand
class _State:
    pass


def _pages(n):
    return (n + 63) // 64 * 64


def prepare(case, seed):
    """A loaded model with its engine, prompts as lists of ids and, where the call goes on from something, the sequences
    that hold it.  Decode: the program has been serving, so its session has taken its steps before."""
    raw, s = _raw(case), _State()
    config = config_from_dict(raw)
    model = DecoderModel(config.model_spec(), _DTYPES[case["dtype"]], "cuda:0")
    model.config = config
    model.load(_Weights(case, seed).get)
    s.new, held, s.start = _tokens(case, seed, _vocab(raw))
    room = [len(t) + case.get("held", 0) + case.get("steps", 0) + 8 for t in s.new]
    s.case, s.engine = case, Engine(model, max_tokens=sum(_pages(n) for n in room), max_seqs=case["batch"])
    s.slots, s.cap = None, max(room)
    if case["kind"] == "decode" or held:
        s.slots = [s.engine.new_sequence() for _ in s.new]
        for slot, tokens in zip(s.slots, held or s.new):
            s.engine.step([slot], [tokens], [[]])
    if case["kind"] != "prompt":
        s.sampler = Sampler(_params(case)) if case["kind"] == "decode" else Sampler(SamplingParams.greedy())
        s.steps, steps = 4, case["steps"]
        run(s)
        s.steps = steps
    return s


def _decode_steps(s, slots, start, windows):
    """`steps` decode steps as the generation loop runs them: tokens [steps][sequences] and the last step's logits."""
    session = s.engine.decode_session(len(slots), s.cap, s.sampler)
    session.bind(slots, start, list(range(len(slots))), [1] * len(slots))
    if s.sampler.params.has_penalties:
        session.set_windows(windows)
    tokens, pending = [], session.launch()
    for _ in range(s.steps - 1):
        ahead = session.launch()
        tokens.append(session.collect(pending))
        pending = ahead
    tokens.append(session.collect(pending))
    return dict(tokens=torch.tensor(tokens), logits=session.last_logits)


def run(s):
    eng, kind = s.engine, s.case["kind"]
    if kind == "decode":
        out = _decode_steps(s, s.slots, s.start, [p[-63:] + [t] for p, t in zip(s.new, s.start)])
        for slot, p in zip(s.slots, s.new):
            eng.truncate(slot, len(p))
        return out
    if kind == "prompt" and s.slots is not None:
        before = [eng.length(slot) for slot in s.slots]
        logits = eng.step(s.slots, s.new, "last")
        for slot, n in zip(s.slots, before):
            eng.truncate(slot, n)
        return logits
    slots = [eng.new_sequence() for _ in s.new]
    logits = eng.step(slots, s.new, "last")
    out = logits
    if kind == "reply":
        first = torch.argmax(logits, dim=-1).tolist()
        out = dict(_decode_steps(s, slots, first, None), first=logits)
    for slot in slots:
        eng.end_sequence(slot)
    return out


# ------------------------------------------------------------------ what the path cannot do without
def _qwen2_work(c):
    """(values of a layer's matrices, values a token leaves in a layer's cache, width of all heads)."""
    h, hd = c["hidden_size"], c["hidden_size"] // c["num_attention_heads"]
    kv = c["num_key_value_heads"] * hd
    return 2 * h * h + 2 * h * kv + 3 * c["intermediate_size"] * h, 2 * kv, h


def work(case):
    raw, elem = _raw(case), 2 if case["dtype"] == "bf16" else 4
    lens, batch, steps = _lengths(case), case["batch"], case.get("steps", 0)
    flops = nbytes = 0.0
    if case["model"] in _QWEN2:
        per_layer, row, heads = _qwen2_work(raw)
        L, head = raw["num_hidden_layers"], raw["vocab_size"] * raw["hidden_size"]
        weights = (L * per_layer + head) * elem
        if case["kind"] == "decode":
            for k in range(steps):
                seen = sum(n + k + 1 for n in lens)
                nbytes += weights + seen * L * row * elem + batch * raw["vocab_size"] * 4
                flops += 2.0 * batch * (L * per_layer + head) + 4.0 * L * heads * seen
        else:
            had = [case["held"] - 3 * i if case["held"] else 0 for i in range(batch)]
            pairs = sum(n * a + n * (n + 1) / 2 for n, a in zip(lens, had))
            nbytes = weights + (sum(lens) + sum(had)) * L * row * elem + batch * raw["vocab_size"] * 4
            flops = 2.0 * (sum(lens) * L * per_layer + batch * head) + 4.0 * L * heads * pairs
        return {"bytes": nbytes, "flops": flops}
    h = raw["width"]
    passes = [(n, 1, [0]) for n in lens] + [(1, batch, lens)] * steps     # (new tokens, sequences, before them)
    matrices = experts = state = kv = 0
    for layer in raw["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        for side in ([m["left"], m["right"]] if layer["type"] == "parallel" else [m]):
            keys, values = side["heads"] * side["dim"], side["heads"] * side["vdim"]
            if "kv_heads" in side:
                matrices += h * (keys + values) + h * side["kv_heads"] * (side["dim"] + side["vdim"])
                kv += side["kv_heads"] * (side["dim"] + side["vdim"])
            else:
                matrices += h * (2 * keys + 3 * values)
                state += keys * side["vdim"]
        if f["kind"] == "dense":
            matrices += 2 * h * f["ff"]
        else:
            matrices += 3 * h * f["shared"]["ff"]
            experts += 3 * h * f["expert"]["ff"]
    attn = sum(4.0 * y["mixer"]["left"]["heads"] * y["mixer"]["left"]["dim"] for y in raw["layers"] if y["type"] == "parallel")
    some = 8.0
    prompt_passes = passes[:batch]
    nbytes += (matrices + some * (1 - (1 - 1 / some) ** sum(lens)) * experts + raw["vocab"] * h) * elem + batch * raw["vocab"] * 4
    for n, _, _ in prompt_passes:
        flops += 2.0 * n * (matrices + experts) + 2.0 * raw["vocab"] * h + attn * n * (n + 1) / 2 + 4.0 * n * state
        nbytes += n * kv * elem + 4 * state
    for k in range(steps):
        seen = sum(n + k + 1 for n in lens)
        nbytes += (matrices + some * (1 - (1 - 1 / some) ** batch) * experts + raw["vocab"] * h) * elem
        nbytes += seen * kv * elem + 8 * state * batch + batch * raw["vocab"] * 4
        flops += 2.0 * batch * (matrices + experts + raw["vocab"] * h) + attn * seen + 4.0 * batch * state
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # four times the distance from `exact` that was measured: 3e-7 in the 32-bit run type; 0.0018 (24 layers of 896) to
    # 0.0055 (28 layers of 3,584) in bfloat16, where every layer rounds its activations
    if case["dtype"] == "fp32":
        return {"rel": 1.5e-6, "max": 3e-5}
    return {"rel": 2e-2, "max": 0.15}


# ------------------------------------------------------------------ the same in 64 bits
def _rms(x, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt()


def _turn(x, base, dims):
    """Values i and i + dims / 2 of every head of x [tokens][heads][width] turned by position * base^(-2 i / dims)."""
    half = dims // 2
    a = torch.arange(x.shape[0], dtype=torch.float64, device=x.device)[:, None] * \
        base ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / dims)
    c, s, u, v = a.cos()[:, None], a.sin()[:, None], x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], -1)


def _causal(q, k, v, scale, first=0, cap=None, slopes=None):
    """Softmax attention of queries [tokens][heads][width], which begin at position `first`, over keys and values
    [tokens][kv heads][width]."""
    out, group = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=q.device), q.shape[1] // k.shape[1]
    at = torch.arange(k.shape[0], device=q.device)
    for hd in range(q.shape[1]):
        kk, vv = k[:, hd // group].t().contiguous(), v[:, hd // group].contiguous()
        for a in range(0, q.shape[0], 4096):
            s = (q[a:a + 4096, hd].contiguous() @ kk) * scale
            gap = (at[first + a:first + a + s.shape[0]])[:, None] - at[None, :]
            if cap is not None:
                s = cap * torch.tanh(s / cap)
            if slopes is not None:
                s = s - slopes[hd] * gap
            out[a:a + 4096, hd] = torch.softmax(s.masked_fill_(gap < 0, -math.inf), -1) @ vv
    return out


def _exact_qwen2(w, sequences):
    """Logits of each sequence's last token."""
    c = w.raw
    H, G = c["num_attention_heads"], c["num_key_value_heads"]
    D, eps = c["hidden_size"] // H, c["rms_norm_eps"]
    wide = lambda name: w.get(name).double()  # noqa: E731
    ends = [0]
    for t in sequences:
        ends.append(ends[-1] + len(t))
    table = w.get("model.embed_tokens.weight")
    x = table[torch.tensor([t for q in sequences for t in q], device="cuda")].double()
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        y = _rms(x, eps) * wide(p + "input_layernorm.weight")
        q, k, v = (y @ wide(f"{p}self_attn.{n}_proj.weight").t() + wide(f"{p}self_attn.{n}_proj.bias") for n in "qkv")
        o = torch.empty_like(q)
        for a, b in zip(ends, ends[1:]):
            qs, ks = (_turn(t[a:b].view(b - a, -1, D), c["rope_theta"], D) for t in (q, k))
            o[a:b] = _causal(qs, ks, v[a:b].view(b - a, G, D), D ** -0.5).reshape(b - a, H * D)
        x = x + o @ wide(p + "self_attn.o_proj.weight").t()
        y = _rms(x, eps) * wide(p + "post_attention_layernorm.weight")
        g = y @ wide(p + "mlp.gate_proj.weight").t()
        g = g.mul_(torch.sigmoid(g)).mul_(y @ wide(p + "mlp.up_proj.weight").t())
        x = x + g @ wide(p + "mlp.down_proj.weight").t()
    x = x[torch.tensor(ends[1:], device="cuda") - 1]
    head = table.double() if c["tie_word_embeddings"] else wide("lm_head.weight")
    return (_rms(x, eps) * wide("model.norm.weight")) @ head.t()


def _layer_norm(x, gain, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / (d.square().mean(-1, keepdim=True) + eps).sqrt() * gain


def _walk(q, k, v, keep, take=None):
    """o_t = S_t^T q_t with S_t = keep_t S_(t-1) + take_t k_t v_t^T, and n_t . q_t of the same sum over the keys alone;
    q, k [tokens][heads][keys], v [tokens][heads][values], keep and take [tokens][heads][keys or 1]."""
    T, H, D = q.shape
    v = torch.cat([v, torch.ones(T, H, 1, dtype=v.dtype, device=v.device)], -1)
    S, o = torch.zeros(H, D, v.shape[2], dtype=v.dtype, device=v.device), torch.empty_like(v)
    k = k if take is None else k * take
    for t in range(T):
        S = torch.addcmul(S * keep[t][:, :, None], k[t][:, :, None], v[t][:, None, :])
        o[t] = (S * q[t][:, :, None]).sum(1)
    return o[..., :-1], o[..., -1]


def _exact_rofizen(w, tokens, places):
    """Logits [places][vocab] of one sequence at the given offsets."""
    c = w.raw
    eps, alpha, T = c["norm"]["eps"], c["postln_alpha"], len(tokens)
    wide = lambda name: w.get(name).double()  # noqa: E731
    ids = torch.tensor(tokens, device="cuda")

    def expert(y, stem):
        g = y @ wide(stem + ".gate").t()
        return (g * torch.sigmoid(g) * (y @ wide(stem + ".up").t())) @ wide(stem + ".down").t()

    x = w.get("embed")[ids].double() * c["embedding"]["scale"]
    for i, layer in enumerate(c["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        split = lambda name, heads: (x @ wide(p + name).t()).view(T, heads, -1)  # noqa: E731
        if layer["type"] == "parallel":
            lf, rg = m["left"], m["right"]
            q, k, v = (x @ wide(f"{p}mix.left.{n}").t() + wide(f"{p}mix.left.{n}.b") for n in "qkv")
            q, k = _rms(q, eps) * wide(p + "mix.left.q.norm"), _rms(k, eps) * wide(p + "mix.left.k.norm")
            at = torch.arange(T, dtype=torch.float64, device="cuda")
            warm = 1.0 + lf["q_temp"]["coef"] * torch.log(torch.floor((at + 1) / lf["q_temp"]["every"]) + 1.0)
            q = q.view(T, lf["heads"], -1) * warm[:, None, None]
            left = _causal(q, k.view(T, lf["kv_heads"], -1), v.view(T, lf["kv_heads"], -1), lf["scale"], cap=lf["softcap"],
                           slopes=[2.0 ** (-8.0 * (hd + 1) / lf["heads"]) for hd in range(lf["heads"])])
            left = left.reshape(T, -1) @ wide(p + "mix.left.o").t() + wide(p + "mix.left.o.b")
            H = rg["heads"]
            gi, gf = (rg["gate_cap"] * torch.tanh((x @ wide(f"{p}mix.right.{n}").t() + wide(f"{p}mix.right.{n}.b")) / rg["gate_cap"])
                      for n in "if")
            gf = torch.nn.functional.logsigmoid(gf)
            # the running maximum of the gates, from 0: max over the starts of what has decayed since
            run = gf.cumsum(0)
            top = torch.maximum(torch.cummax(gi - run, 0).values, torch.zeros_like(gi)) + run
            was = torch.cat([torch.zeros_like(top[:1]), top[:-1]])
            o, n = _walk(split("mix.right.q", H) * rg["dim"] ** -0.5, split("mix.right.k", H), split("mix.right.v", H),
                         torch.exp(gf + was - top)[..., None], torch.exp(gi - top)[..., None])
            o = o / (torch.maximum(n.abs(), torch.exp(-top)) + 1e-6)[..., None]
            o = _rms(o, eps).reshape(T, -1) * wide(p + "mix.right.norm") * torch.sigmoid(x @ wide(p + "mix.right.g").t())
            right = o @ wide(p + "mix.right.o").t()
            y = 0.5 * (_rms(left, eps) * wide(p + "mix.left.out") + _rms(right, eps) * wide(p + "mix.right.out"))
        else:
            H = m["heads"]
            q, k, v = (split("mix." + n, H) for n in "qkv")
            if layer["type"] == "gla":
                z = x @ wide(p + "mix.a1").t() @ wide(p + "mix.a2").t() + wide(p + "mix.a2.b")
                keep = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, H, -1)
                o = _rms(_walk(q * m["dim"] ** -0.5, k, v, keep)[0], eps) * wide(p + "mix.norm")
            else:
                q, k = _turn(q, m["rot"]["base"], m["rot"]["dims"]), _turn(k, m["rot"]["base"], m["rot"]["dims"])
                keep = torch.tensor(m["decay"], dtype=torch.float64, device="cuda")[None, :, None].expand(T, H, 1)
                o = _rms(_walk(q, k * m["dim"] ** -0.5, v, keep)[0], eps)
            g = x @ wide(p + "mix.g").t()
            y = (o.reshape(T, -1) * g * torch.sigmoid(g)) @ wide(p + "mix.o").t()
        x = _layer_norm(alpha * x + y, wide(p + "norm1"), eps)
        if f["kind"] == "dense":
            y = torch.relu(x @ wide(p + "mlp.up").t()).square() @ wide(p + "mlp.down").t()
        else:
            y = torch.sigmoid(x @ wide(p + "mlp.shared.sg").t()) * expert(x, p + "mlp.shared")
            chosen = w.get(p + "mlp.table")[ids].long()
            for e in range(f["router"]["experts"]):
                rows, _ = torch.where(chosen == e)
                if rows.numel():
                    y.index_add_(0, rows, expert(x[rows], f"{p}mlp.e{e}") / f["router"]["top"])
        x = _layer_norm(alpha * x + y, wide(p + "norm2"), eps)
    x = _layer_norm(x[torch.tensor(places, device="cuda")], wide("final.norm"), eps)
    return x @ wide("head").t()


def exact(case, seed):
    if work(case)["flops"] > 3e14 or (case["kind"] == "decode" and sum(_lengths(case)) * work(_prompt(case["model"], 1, 1))["flops"] > 3e14):
        return None
    raw, w = _raw(case), _Weights(case, seed)
    new, held, start = _tokens(case, seed, _vocab(raw))
    if case["kind"] == "prompt":
        whole = [a + b for a, b in zip(held, new)] if held else new
        if case["model"] in _QWEN2:
            return _exact_qwen2(w, whole)
        return torch.cat([_exact_rofizen(w, t, [len(t) - 1]) for t in whole])
    if case["kind"] == "reply":
        out = []
        for t in new:
            fed, first = list(t), len(t) - 1
            token = t[-1]
            for _ in range(case["steps"]):
                token = _next(token, raw)
                fed.append(token)
            out.append(_exact_rofizen(w, fed, [first, len(fed) - 1]))
        return dict(tokens=None, first=torch.stack([o[0] for o in out]), logits=torch.stack([o[1] for o in out]))
    fed = []
    for t, s in zip(new, start):
        chain = [s]
        for _ in range(case["steps"] - 1):
            chain.append(_next(chain[-1], raw))
        fed.append(chain)
    logits = _exact_qwen2(w, [a + b for a, b in zip(new, fed)])
    p = _params(case)
    if p.has_penalties:                              # in the window: the prompt's end and what was fed since
        for row, t, chain in zip(logits, new, fed):
            seen = torch.tensor(sorted(set((t[-63:] + chain)[-64:])), device="cuda")
            row[seen] = torch.where(row[seen] > 0, row[seen] / p.repeat_penalty, row[seen] * p.repeat_penalty)
    return dict(tokens=None, logits=logits)
