"""The work that programs have this engine do, as cases to be timed.

A case is one of four kinds, each a pass through ``Model.step`` / ``Model.decode_greedy`` and the
cache manager, as the scheduler, ``bin/trace_run`` and ``bench.py`` call them:

``prefill``   one prompt, whole or in portions, with the logits of its last token;
``decode``    requests that find their context in the cache (as a hit in the prefix cache does)
              take ``steps`` single-token steps, every step's logits kept;
``mixed``     one step of continuous batching: requests that decode beside prompt portions, some of
              which go on with a context that is already cached;
``generate``  whole requests: prompts in, then single tokens until they end; greedy through the
              device-side loop where the arithmetic is 32-bit, else a given continuation.

The tokens that a decoding request brings are given (a recorded continuation, what ``bin/trace_run``
replays) rather than picked: a pick between two nearly equal logits would make everything after it a
different computation.  In 32-bit arithmetic such picks are rare enough to be made.

Layer sizes are those of the presets ``qwen3-0.6b``, ``qwen3-8b`` and ``qwen3-32b`` and of the Toripel
design that ``bench.py`` measures at the first one's sizes.  Weights are normal in bfloat16 with a deviation
of 0.64 / sqrt(width) (0.02 at a width of 1,024), so that every width's layers change the stream alike; norm
weights are 1 + N(0, 0.1), token ids uniform.
"""

from __future__ import annotations

import math

import torch

from lockstep_amd.config import config_from_dict
from lockstep_amd.engine.batch import StepEntry
from lockstep_amd.engine.model import model_from_tensors

PAGE = 16
VOCAB = 151936
EPS = 1e-6
THETA = 1000000.0
F64 = torch.float64

#: layer sizes: width, feed-forward, layers, heads, kv heads, head size, whether the head is the embedding
SIZES = {
    "qwen3-0.6b": (1024, 3072, 28, 16, 8, 128, True),
    "qwen3-8b": (4096, 12288, 36, 32, 8, 128, False),
    "qwen3-32b": (5120, 25600, 64, 64, 8, 128, False),
    "toripel-0.6b": (1024, 3072, 28, 16, 8, 128, False),
}

# Toripel beside the sizes above: experts, experts a token uses, residual copies, window, taps of the
# convolutions, and the rotation of the attention over a latent
EXPERTS, TOP, STREAMS, WINDOW, TAPS = 32, 4, 4, 4096, 4
LATENT_ROT = {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}


def listed():
    return [
        # one reader at a chat window: nothing but launches, their gaps and 1.2 GB of weights a token
        dict(name="decode 1", kind="decode", model="qwen3-0.6b", layers=28, dtype="bfloat16",
             batch=1, shortest=512, longest=512, steps=32),
        # bench.py's headline: a small service
        dict(name="decode 8", kind="decode", model="qwen3-0.6b", layers=28, dtype="bfloat16",
             batch=8, shortest=512, longest=512, steps=32),
        # a full service whose conversations have all ages
        dict(name="decode 64 ragged", kind="decode", model="qwen3-0.6b", layers=28, dtype="bfloat16",
             batch=64, shortest=128, longest=4096, steps=16),
        # the larger model behind a small service, contexts of a few pages of text
        dict(name="decode 8 8b", kind="decode", model="qwen3-8b", layers=36, dtype="bfloat16",
             batch=8, shortest=1024, longest=2048, steps=24),
        # a question of a few lines: the time to its first token
        dict(name="prefill 97", kind="prefill", model="qwen3-0.6b", layers=28, dtype="bfloat16",
             tokens=97, portion=0),
        # bench.py's prompt
        dict(name="prefill 2048", kind="prefill", model="qwen3-0.6b", layers=28, dtype="bfloat16",
             tokens=2048, portion=0),
        # the same for the larger model
        dict(name="prefill 2048 8b", kind="prefill", model="qwen3-8b", layers=36, dtype="bfloat16",
             tokens=2048, portion=0),
        # a long document in portions, as a service with a token budget runs it; the last one is ragged
        dict(name="prefill 9000 portions", kind="prefill", model="qwen3-0.6b", layers=28, dtype="bfloat16",
             tokens=9000, portion=2048),
        # a step in the middle of serving the larger model: many decode, three bring prompt portions
        dict(name="mixed 8b", kind="mixed", model="qwen3-8b", layers=36, dtype="bfloat16",
             batch=21, shortest=128, longest=1536, prompts=3, tokens=311),
        # the 32-bit path that results are checked with: whole requests, greedy
        dict(name="generate float32", kind="generate", model="qwen3-0.6b", layers=28, dtype="float32",
             batch=8, tokens=250, steps=24),
        # the family whose parts the other designs share most of (delta rule, windowed and latent attention,
        # experts, several residual copies): a prompt, and whole requests
        dict(name="toripel prefill 2048", kind="prefill", model="toripel-0.6b", layers=28, dtype="bfloat16",
             tokens=2048, portion=0),
        dict(name="toripel generate 8", kind="generate", model="toripel-0.6b", layers=28, dtype="bfloat16",
             batch=8, tokens=128, steps=32),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["decode", "decode", "prefill", "prefill", "mixed", "generate"])
    # (the largest sizes with an eighth of their layers, so that no case outgrows the listed ones)
    model, layers = rng.choice([("qwen3-0.6b", 28), ("qwen3-0.6b", 28), ("qwen3-8b", 36), ("qwen3-32b", 8)])
    case = dict(kind=kind, model=model, layers=layers, dtype="bfloat16")
    if kind == "decode":
        batch = spread(1, 64)
        most = min(4096, (65536 if model == "qwen3-0.6b" else 14000) // batch)
        longest = max(64, spread(128, most))
        return dict(case, batch=batch, shortest=max(16, spread(longest // 16, longest)), longest=longest,
                    steps=rng.randint(8, 24))
    if kind == "prefill":
        if rng.random() < 0.25:
            case.update(model="toripel-0.6b", layers=28)
            return dict(case, tokens=spread(16, 2048), portion=0)
        tokens = spread(16, 9000 if model == "qwen3-0.6b" else 2047)
        return dict(case, tokens=tokens, portion=2048 if tokens > 2048 else rng.choice([0, 0, 512]))
    if kind == "mixed":
        return dict(case, batch=spread(1, 40), shortest=64, longest=spread(96, 1536), prompts=rng.randint(1, 4),
                    tokens=spread(16, 400))
    if rng.random() < 0.5:
        return dict(case, model="qwen3-0.6b", layers=28, dtype="float32", batch=rng.randint(1, 8), tokens=spread(16, 250),
                    steps=rng.randint(8, 24))
    return dict(case, model="toripel-0.6b", layers=28, batch=rng.randint(1, 8), tokens=spread(16, 128),
                steps=rng.randint(8, 32))


# -- sizes of a case -----------------------------------------------------------------------


def contexts(case):
    """Cached tokens of every decoding request: whole pages, evenly spaced in the logarithm."""
    n, lo, hi = case["batch"], case["shortest"], case["longest"]
    return [PAGE * max(1, round(lo * (hi / lo) ** (i / max(1, n - 1)) / PAGE)) for i in range(n)]


def portions(case):
    """(cached tokens, new tokens) of a mixed step's prompt portions: every second goes on with a cached part."""
    return [(PAGE * (case["tokens"] // PAGE) if i % 2 else 0, case["tokens"] + 13 * i) for i in range(case["prompts"])]


def steps_of(case):
    """A list of model steps, each a list of (tokens before, new tokens, wanted rows) by request."""
    kind = case["kind"]
    if kind == "prefill":
        n, size = case["tokens"], case["portion"] or case["tokens"]
        return [[(lo, min(size, n - lo), 1 if lo + size >= n else 0)] for lo in range(0, n, size)]
    if kind == "decode":
        return [[(c + s, 1, 1) for c in contexts(case)] for s in range(case["steps"])]
    if kind == "mixed":
        return [[(c, 1, 1) for c in contexts(case)] + [(c, n, 1) for c, n in portions(case)]]
    return [[(0, case["tokens"], 1)] * case["batch"]] + [[(case["tokens"] + s, 1, 1)] * case["batch"]
                                                         for s in range(case["steps"])]


# -- weights -------------------------------------------------------------------------------


def config_of(case):
    h, f, _, heads, kv, d, tied = SIZES[case["model"]]
    if not case["model"].startswith("toripel"):
        return dict(model_type="qwen3", hidden_size=h, intermediate_size=f, num_hidden_layers=case["layers"],
                    num_attention_heads=heads, num_key_value_heads=kv, head_dim=d, vocab_size=VOCAB, rms_norm_eps=EPS,
                    rope_theta=THETA, max_position_embeddings=40960, tie_word_embeddings=tied)
    mlp = dict(kind="moe", expert=dict(ff=f // TOP), router=dict(experts=EXPERTS, top=TOP))
    layers = []
    for i in range(case["layers"]):
        grouped = dict(heads=heads, kv_heads=kv, dim=d, vdim=d)
        latent = dict(heads=heads, dim=d, rot_dim=d // 2, vdim=d, q_rank=3 * d, kv_rank=d, scale=(d + d // 2) ** -0.5,
                      mask=dict(size=WINDOW), rot=dict(dims=d // 2, base=THETA, scaling=LATENT_ROT))
        kind, mixer = [("delta", dict(grouped, conv=TAPS)), ("attention", dict(grouped, scale=d ** -0.5, mask=dict(size=WINDOW))),
                       ("latent_attention", latent), ("latent_attention", dict(latent, kv_from=i - 1))][i % 4]
        layers.append(dict(type=kind, mixer=mixer, mlp=mlp))
    return dict(architecture="Toripel", vocab=VOCAB, width=h, embedding=dict(scale=1.0), norm=dict(eps=EPS),
                streams=STREAMS, layers=layers)


def shapes(case):
    """Every tensor's name, shape and distribution, in the order in which they are drawn."""
    h, f, _, heads, kv, d, tied = SIZES[case["model"]]
    if not case["model"].startswith("toripel"):
        yield "model.embed_tokens.weight", (VOCAB, h), "matrix"
        for i in range(case["layers"]):
            p = f"model.layers.{i}"
            yield f"{p}.input_layernorm.weight", (h,), "norm"
            for name, shape in (("q_proj", (heads * d, h)), ("k_proj", (kv * d, h)), ("v_proj", (kv * d, h)), ("o_proj", (h, heads * d))):
                yield f"{p}.self_attn.{name}.weight", shape, "matrix"
            yield f"{p}.self_attn.q_norm.weight", (d,), "norm"
            yield f"{p}.self_attn.k_norm.weight", (d,), "norm"
            yield f"{p}.post_attention_layernorm.weight", (h,), "norm"
            for name, shape in (("gate_proj", (f, h)), ("up_proj", (f, h)), ("down_proj", (h, f))):
                yield f"{p}.mlp.{name}.weight", shape, "matrix"
        yield "model.norm.weight", (h,), "norm"
        if not tied:
            yield "lm_head.weight", (VOCAB, h), "matrix"
        return
    rot, rank = d // 2, d
    yield "embed", (VOCAB, h), "matrix"
    for i in range(case["layers"]):
        p, m = f"l{i}", f"l{i}.mix"
        for half in (1, 2):
            yield f"{p}.norm{half}", (h,), "centred"
            yield f"{p}.hc{half}.in", (STREAMS,), "unit"
            yield f"{p}.hc{half}.out", (STREAMS,), "norm"
            yield f"{p}.hc{half}.mix", (STREAMS, STREAMS), "identity"
        if i % 4 == 0:
            for name, rows in (("q", kv * d), ("k", kv * d), ("v", heads * d)):
                yield f"{m}.{name}", (rows, h), "matrix"
                yield f"{m}.{name}.conv", (rows, TAPS), "unit"
            yield f"{m}.b", (heads, h), "matrix"
            yield f"{m}.a", (heads, h), "matrix"
            yield f"{m}.A_log", (heads,), "vector"
            yield f"{m}.dt_bias", (heads,), "vector"
            yield f"{m}.norm", (d,), "norm"
            yield f"{m}.g", (heads * d, h), "matrix"
        elif i % 4 == 1:
            for name, rows in (("q", heads * d), ("k", kv * d), ("v", kv * d)):
                yield f"{m}.{name}", (rows, h), "matrix"
                yield f"{m}.{name}.b", (rows,), "vector"
        else:
            yield f"{m}.dq", (3 * d, h), "matrix"
            yield f"{m}.dq.norm", (3 * d,), "norm"
            yield f"{m}.uq", (heads * (d + rot), 3 * d), "matrix"
            if i % 4 == 2:
                yield f"{m}.dkv", (rank + rot, h), "matrix"
                yield f"{m}.dkv.norm", (rank,), "norm"
            yield f"{m}.uk", (heads * d, rank), "matrix"
            yield f"{m}.uv", (heads * d, rank), "matrix"
            yield f"{m}.sink", (heads,), "vector"
        yield f"{m}.o", (h, heads * d), "matrix"
        yield f"{p}.mlp.table", (VOCAB, TOP), "table"
        for e in range(EXPERTS):
            yield f"{p}.mlp.e{e}.gate", (f // TOP, h), "matrix"
            yield f"{p}.mlp.e{e}.up", (f // TOP, h), "matrix"
            yield f"{p}.mlp.e{e}.down", (h, f // TOP), "matrix"
    yield "final.norm", (h,), "centred"
    yield "head", (VOCAB, h), "matrix"


def tensors_of(case, seed):
    """The checkpoint: a tensor by name, in bfloat16, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    spread = 0.64 / math.sqrt(SIZES[case["model"]][0])
    out = {}
    for name, shape, how in shapes(case):
        if how == "table":           # every token names TOP different experts
            first = torch.randint(0, EXPERTS, (shape[0], 1), generator=gen, device="cuda")
            stride = 2 * torch.randint(0, EXPERTS // 2, (shape[0], 1), generator=gen, device="cuda") + 1
            out[name] = ((first + stride * torch.arange(TOP, device="cuda")) % EXPERTS).to(torch.int32)
            continue
        if how == "unit":
            value = torch.rand(shape, generator=gen, device="cuda")
        else:
            std = 0.1 if how in ("norm", "centred") else spread
            value = torch.empty(shape, dtype=torch.bfloat16 if how == "matrix" else torch.float32, device="cuda")
            value.normal_(0.0, std, generator=gen)
            if how == "norm":
                value += 1.0
            if how == "identity":
                value += torch.eye(shape[0], device="cuda")
        out[name] = value.to(torch.bfloat16)
    return out


def tokens_of(case, seed):
    """Token ids by request, as many as the case's steps take in all (cached contexts included)."""
    need = {}
    for step in steps_of(case):
        for i, (before, new, _) in enumerate(step):
            need[i] = before + new
    gen = torch.Generator().manual_seed(seed)
    return [torch.randint(0, VOCAB, (need[i],), generator=gen).tolist() for i in sorted(need)]


# -- a pass --------------------------------------------------------------------------------


def prepare(case, seed):
    config = config_from_dict(config_of(case))
    model = model_from_tensors(config, tensors_of(case, seed), dtype=case["dtype"])
    tokens, steps = tokens_of(case, seed), steps_of(case)
    cached = [before for before, _, _ in steps[0]]
    pages = sum(-(-len(t) // PAGE) + 1 for t in tokens) + sum(c // PAGE for c in cached)
    longest = max(len(t) for t in tokens)
    cache = model.make_cache(num_pages=pages, page_size=PAGE, max_requests=2 * len(tokens), max_tokens_per_request=longest + PAGE)
    state = dict(model=model, cache=cache, greedy=case["kind"] == "generate" and case["dtype"] == "float32", kept={})
    # contexts that are already cached: requests of their own, which the pass's requests share the pages of
    for lo in range(0, len(tokens), 4):
        entries = []
        for i in range(lo, min(lo + 4, len(tokens))):
            if cached[i]:
                cache.open(("kept", i))
                entries.append(StepEntry(("kept", i), tokens[i][:cached[i]]))
        model.step(cache, entries)
    for i, n in enumerate(cached):
        if n:
            state["kept"][i] = (cache.request_pages(("kept", i)), n)
    state["requests"] = list(range(len(tokens)))
    state["steps"] = [[StepEntry(i, tokens[i][before:before + new], [new - 1] if want else [])
                       for i, (before, new, want) in enumerate(step)] for step in steps]
    return state


def run(state):
    model, cache, steps = state["model"], state["cache"], state["steps"]
    for i in state["requests"]:
        cache.open(i)
        if i in state["kept"]:
            pages, n = state["kept"][i]
            cache.adopt(i, pages)
            cache.commit(i, n)
    if state["greedy"]:
        prompt = model.step(cache, steps[0])
        first = prompt.argmax(dim=1).tolist()
        picked = model.decode_greedy(cache, state["requests"], first, len(steps) - 1)
        last = model.step(cache, [StepEntry(i, [int(t)], [0]) for i, t in zip(state["requests"], picked[-1])])
        out = {"prompt": prompt, "picked": picked, "last": last}
    else:
        out = [logits for logits in (model.step(cache, entries) for entries in steps) if logits is not None]
    for i in state["requests"]:
        cache.close(i)
    return out


# -- what a pass cannot do without ---------------------------------------------------------


def work(case):
    h, f, _, heads, kv, d, _ = SIZES[case["model"]]
    element = 2 if case["dtype"] == "bfloat16" else 4
    toripel = case["model"].startswith("toripel")
    total = {"bytes": 0.0, "flops": 0.0}
    steps = steps_of(case)
    if case["kind"] == "generate" and case["dtype"] == "float32":
        steps = steps + [[(b + 1, n, w) for b, n, w in steps[-1]]]       # the step whose logits are returned
    for step in steps:
        tokens, wanted = sum(n for _, n, _ in step), sum(w for _, _, w in step)
        for i in range(case["layers"]):
            # matrix elements a token multiplies with, elements a step reads, elements of cache a token holds,
            # and multiply-adds for a pair of a query and a key
            if not toripel:
                matrices = h * d * (2 * heads + 2 * kv) + 3 * h * f
                read, held, pair = matrices, 2 * kv * d, 2 * heads * d
            else:
                experts = 3 * h * (f // TOP)
                mixer = [h * d * (2 * kv + 3 * heads) + 2 * h * heads, h * d * (2 * heads + 2 * kv)][i % 4] if i % 4 < 2 else \
                    3 * d * h + heads * (d + d // 2) * 3 * d + (d + d // 2) * h * (i % 4 == 2) + 2 * heads * d * d + h * heads * d
                held = [0, 2 * kv * d, d + d // 2, 0][i % 4]
                pair = [0, 2 * heads * d, heads * (2 * d + d // 2), heads * (2 * d + d // 2)][i % 4]
                matrices, read = mixer + TOP * experts, mixer + min(EXPERTS, TOP * tokens) * experts
                if i % 4 == 0:       # the state's update and read-out, and the state itself in and out
                    total["flops"] += tokens * heads * d * d * 6.0
                    total["bytes"] += 8.0 * len(step) * heads * d * d
            pairs = sum(n * b + n * (n + 1) / 2 for b, n, _ in step)
            total["flops"] += 2.0 * tokens * matrices + 2.0 * pairs * pair
            total["bytes"] += element * (read + held * sum(b + n for b, n, _ in step))
        total["flops"] += 2.0 * wanted * h * VOCAB
        total["bytes"] += element * (h * tokens + (h * VOCAB if wanted else 0)) + 4.0 * wanted * VOCAB
    return total


def tolerance(case):
    """Four times what separates a pass from the same in 64 bits, at most 0.03 (measured: 32-bit arithmetic 1e-6;
    bfloat16 0.006 at the smallest Qwen3 sizes, 0.01 at the larger ones and for Toripel; the largest difference of a
    logit 0.04 to 0.06 of their root mean square)."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6, "max": 1e-4, "differ": 0.01}
    return {"rel": 0.025, "max": 0.16} if case["model"] == "qwen3-0.6b" else {"rel": 0.03, "max": 0.24}


# -- the same in 64 bits -------------------------------------------------------------------


def exact(case, seed):
    w, tokens, steps = tensors_of(case, seed), tokens_of(case, seed), steps_of(case)
    model = ToripelIn64(case, w) if case["model"].startswith("toripel") else Qwen3In64(case, w)
    if case["kind"] == "generate" and case["dtype"] == "float32":
        sequences, rows = [t[:case["tokens"]] for t in tokens], []
        for _ in range(case["steps"] + 2):
            ends = model.logits(sequences, [[len(s) - 1] for s in sequences])
            rows.append(torch.cat(ends))
            for s, token in zip(sequences, rows[-1].argmax(dim=1).tolist()):
                s.append(token)
        return {"prompt": rows[0], "picked": torch.tensor([[s[case["tokens"] + 1 + i] for s in sequences] for i in range(case["steps"])]),
                "last": rows[-1]}
    wanted = [[before + new - 1 for step in steps for r, (before, new, want) in enumerate(step) if r == i and want]
              for i in range(len(tokens))]
    rows = model.logits(tokens, wanted)
    out = []
    for s in range(max(len(r) for r in rows)):
        out.append(torch.stack([r[s] for r in rows]))
    return out


def rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def attend(q, k, v, scale, window=None, sink=None):
    """Causal attention of one sequence: q [T, heads, d], k and v [T, kv heads, ...]."""
    n, heads, _ = q.shape
    k, v = (x.repeat_interleave(heads // x.shape[1], dim=1).transpose(0, 1).contiguous() for x in (k, v))
    out = []
    for lo in range(0, n, 1024):         # rows at a time, so that the scores fit
        rows = q[lo:lo + 1024].transpose(0, 1)
        s = torch.matmul(rows, k[:, :lo + 1024].transpose(1, 2).contiguous()) * scale
        i, j = torch.arange(lo, lo + rows.shape[1], device=q.device)[:, None], torch.arange(s.shape[2], device=q.device)[None, :]
        hidden = j > i if window is None else (j > i) | (i - j >= window)
        s = s.masked_fill(hidden, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink[:, None, None].expand(heads, s.shape[1], 1)], dim=2)
        p = torch.softmax(s, dim=2)
        out.append(torch.matmul(p[:, :, :lo + 1024] if sink is None else p[:, :, :-1], v[:, :lo + 1024]).transpose(0, 1))
    return torch.cat(out).reshape(n, -1)


class Qwen3In64:
    def __init__(self, case, w):
        self.w, self.case = w, case
        self.h, self.f, _, self.heads, self.kv, self.d, self.tied = SIZES[case["model"]]

    def rotate(self, x):
        half = self.d // 2
        f = THETA ** (-torch.arange(half, dtype=F64, device=x.device) * 2.0 / self.d)
        angle = torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None, None] * f
        lo, hi, c, s = x[..., :half], x[..., half:], angle.cos(), angle.sin()
        return torch.cat([lo * c - hi * s, hi * c + lo * s], dim=-1)

    def logits(self, sequences, wanted):
        embed = self.w["model.embed_tokens.weight"]
        xs = [embed[torch.tensor(t, device="cuda")].to(F64) for t in sequences]
        for i in range(self.case["layers"]):
            w = {name: self.w[f"model.layers.{i}.{name}.weight"].to(F64) for name in (
                "input_layernorm", "post_attention_layernorm", "self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj",
                "self_attn.o_proj", "self_attn.q_norm", "self_attn.k_norm", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")}
            for r, x in enumerate(xs):
                y = rms(x) * w["input_layernorm"]
                q, k, v = ((y @ w[f"self_attn.{n}_proj"].T).reshape(len(x), -1, self.d) for n in "qkv")
                q, k = self.rotate(rms(q) * w["self_attn.q_norm"]), self.rotate(rms(k) * w["self_attn.k_norm"])
                x = x + attend(q, k, v, self.d ** -0.5) @ w["self_attn.o_proj"].T
                y = rms(x) * w["post_attention_layernorm"]
                gate = y @ w["mlp.gate_proj"].T
                xs[r] = x + (gate * torch.sigmoid(gate) * (y @ w["mlp.up_proj"].T)) @ w["mlp.down_proj"].T
        head = (embed if self.tied else self.w["lm_head.weight"]).to(F64)
        return [(rms(x[rows]) * self.w["model.norm.weight"].to(F64)) @ head.T for x, rows in zip(xs, wanted)]


class ToripelIn64:
    def __init__(self, case, w):
        self.w, self.case = w, case
        self.h, self.f, _, self.heads, self.kv, self.d, _ = SIZES[case["model"]]

    def t(self, name):
        return self.w[name].to(F64)

    def rotate(self, x):
        """The last axis in neighbouring pairs, with frequencies stretched along a ramp."""
        dims, positions = x.shape[-1], torch.arange(x.shape[0], dtype=F64, device=x.device)

        def turns_at(t):
            return dims * math.log(LATENT_ROT["original"] / (2.0 * math.pi * t)) / (2.0 * math.log(THETA))

        lo, hi = max(math.floor(turns_at(LATENT_ROT["fast"])), 0), min(math.ceil(turns_at(LATENT_ROT["slow"])), dims - 1)
        pair = torch.arange(dims // 2, dtype=F64, device=x.device)
        ramp = ((pair - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f = THETA ** (-2.0 * pair / dims) * (ramp / LATENT_ROT["factor"] + 1.0 - ramp)
        angle = (positions[:, None] * f).reshape((len(x),) + (1,) * (x.dim() - 2) + (dims // 2,))
        magnitude = 0.1 * math.log(LATENT_ROT["factor"]) + 1.0
        u, v, c, s = x[..., 0::2], x[..., 1::2], angle.cos() * magnitude, angle.sin() * magnitude
        return torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)

    def delta(self, p, y):
        n, d = len(y), self.d

        def convolved(name, heads):
            x, taps = y @ self.t(f"{p}.{name}").T, self.t(f"{p}.{name}.conv")
            x = torch.cat([x.new_zeros(TAPS - 1, x.shape[1]), x])
            x = sum(x[a:a + n] * taps[:, a] for a in range(TAPS))
            return (x * torch.sigmoid(x)).reshape(n, heads, d)

        q, k, v = convolved("q", self.kv), convolved("k", self.kv), convolved("v", self.heads)
        q, k = (x / torch.sqrt((x * x).sum(dim=-1, keepdim=True) + 1e-6) for x in (q, k))
        q, k = (x.repeat_interleave(self.heads // self.kv, dim=1) for x in (q * d ** -0.5, k))
        beta = torch.sigmoid(y @ self.t(f"{p}.b").T)
        decay = torch.exp(-torch.exp(self.t(f"{p}.A_log")) * torch.nn.functional.softplus(y @ self.t(f"{p}.a").T + self.t(f"{p}.dt_bias")))
        state, out = y.new_zeros(self.heads, d, d), []
        for t in range(n):
            state = decay[t][:, None, None] * state
            u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], state)[:, 0])
            state = state + k[t][:, :, None] * u[:, None, :]
            out.append(torch.bmm(q[t][:, None], state)[:, 0])
        gate = y @ self.t(f"{p}.g").T
        o = (rms(torch.stack(out)) * self.t(f"{p}.norm")).reshape(n, -1)
        return (o * gate * torch.sigmoid(gate)) @ self.t(f"{p}.o").T

    def mixer(self, i, y, latents):
        p, n, d, heads = f"l{i}.mix", len(y), self.d, self.heads
        if i % 4 == 0:
            return self.delta(p, y)
        if i % 4 == 1:
            q, k, v = ((y @ self.t(f"{p}.{a}").T + self.t(f"{p}.{a}.b")).reshape(n, -1, d) for a in "qkv")
            return attend(rms(q), rms(k), v, d ** -0.5, WINDOW) @ self.t(f"{p}.o").T
        q = ((rms(y @ self.t(f"{p}.dq").T) * self.t(f"{p}.dq.norm")) @ self.t(f"{p}.uq").T).reshape(n, heads, -1)
        q = torch.cat([q[..., :d], self.rotate(q[..., d:])], dim=-1)
        if i % 4 == 2:
            down = y @ self.t(f"{p}.dkv").T
            latents["c"], latents["rot"] = rms(down[:, :d]) * self.t(f"{p}.dkv.norm"), self.rotate(down[:, d:])
        k = (latents["c"] @ self.t(f"{p}.uk").T).reshape(n, heads, d)
        k = torch.cat([k, latents["rot"][:, None, :].expand(n, heads, d // 2)], dim=-1)
        v = (latents["c"] @ self.t(f"{p}.uv").T).reshape(n, heads, d)
        return attend(q, k, v, (d + d // 2) ** -0.5, WINDOW, self.t(f"{p}.sink")) @ self.t(f"{p}.o").T

    def feed_forward(self, i, y, tokens):
        p, out = f"l{i}.mlp", torch.zeros_like(y)
        named = self.w[f"{p}.table"][tokens]
        for e in range(EXPERTS):
            rows = (named == e).any(dim=1).nonzero()[:, 0]
            if len(rows):
                gate, up = y[rows] @ self.t(f"{p}.e{e}.gate").T, y[rows] @ self.t(f"{p}.e{e}.up").T
                out[rows] += (gate * torch.sigmoid(gate) * up) @ self.t(f"{p}.e{e}.down").T / TOP
        return out

    def logits(self, sequences, wanted):
        out = []
        for ids, rows in zip(sequences, wanted):
            tokens = torch.tensor(ids, device="cuda")
            streams = self.w["embed"][tokens].to(F64)[:, None, :].repeat(1, STREAMS, 1)
            latents = {}
            for i in range(self.case["layers"]):
                for half in (1, 2):
                    hc = f"l{i}.hc{half}"
                    y = rms((streams * self.t(f"{hc}.in")[:, None]).sum(dim=1)) * (1.0 + self.t(f"l{i}.norm{half}"))
                    y = self.mixer(i, y, latents) if half == 1 else self.feed_forward(i, y, tokens)
                    streams = torch.einsum("sr,tsw->trw", self.t(f"{hc}.mix"), streams) + self.t(f"{hc}.out")[None, :, None] * y[:, None, :]
            x = rms(streams[rows].sum(dim=1)) * (1.0 + self.t("final.norm"))
            out.append(x @ self.t("head").T)
        return out
