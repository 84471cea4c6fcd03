"""The work that users of this engine have it do, as cases that can be measured: Qwen2.5 decoders through ``LLM``, its
step function and its sampler.

The dense Qwen2.5 decoder is the architecture that the engine's entry points default to and that its published figures
are of; its layer sizes here are those of ``bench.py``, its weights seeded random ones.  A pass is what one turn of a
serving loop does:

* ``decode``: one step of ``requests`` requests that hold between ``shortest`` and ``longest`` tokens, a token each; they
  grow by that token, and begin again with their prompts once they reach the length that the pool was sized for;
* ``prefill``: prompts of between ``shortest`` and ``longest`` tokens, whole, in steps of at most BUDGET tokens, with the
  logits of their last places; then they end;
* ``mixed``: ``requests`` requests of between ``shortest`` and ``longest`` tokens decode while a prompt of ``prompt``
  tokens comes in portions of ``portion`` tokens, as continuous batching cuts it; then the prompt's request ends;
* ``sample``: the next tokens of ``requests`` rows of logits, with the options given.

Every case but ``sample`` returns float32 logits.
"""

from __future__ import annotations

import functools
import hashlib
import math

import torch

from somi_inference_amd import LLM, Qwen2Config, SamplingParams
from somi_inference_amd.engine.batch import StepEntry

DEVICE = "cuda:0"
BUDGET = 8192            # tokens of one step of a prompt at most
PAGE = 16                # tokens a cache page (the default of LLM)

# layers, width, query heads, key/value heads, head size, feed-forward, norm eps, vocabulary, tied head.  Of the 7B model's 28
# layers the first 24 and of the 14B model's 48 the first 18: behind more of them (48: 0.04) two correct orders of bfloat16 sums
# leave logits of random weights too far apart for a comparison to tell rounding from a fault; every layer costs the same.
SIZES = {
    "0.5b": (24, 896, 14, 2, 64, 4864, 1e-6, 151936, True),
    "7b": (24, 3584, 28, 4, 128, 18944, 1e-6, 152064, False),
    "14b": (18, 5120, 40, 8, 128, 13824, 1e-5, 152064, False),
}


# ------------------------------------------------------------------------------------------------------------ cases
def _decode(name, sizes, requests, shortest, longest, dtype="bfloat16"):
    return {"name": name, "kind": "decode", "sizes": sizes, "dtype": dtype, "requests": requests, "shortest": shortest,
            "longest": longest}


def _prefill(name, sizes, requests, shortest, longest, dtype="bfloat16"):
    return dict(_decode(name, sizes, requests, shortest, longest, dtype), kind="prefill")


def listed() -> list[dict]:
    return [
        # one user of a small model: the smallest step there is, launches and latencies
        _decode("decode 0.5b 1x1024", "0.5b", 1, 1024, 1024),
        # a handful of users of a 7B model at its benchmark's context: the weights' way from memory
        _decode("decode 7b 8x4096", "7b", 8, 4096, 4096),
        # a busy server: keys and values weigh as much as weights
        _decode("decode 7b 64x2048", "7b", 64, 2048, 2048),
        # a very busy one, with requests of every age; an odd number of them
        _decode("decode 7b 147 ragged", "7b", 147, 301, 1019),
        # the first token of a short question to a small model
        _prefill("prefill 0.5b 128", "0.5b", 1, 128, 128),
        # the first token of an ordinary prompt
        _prefill("prefill 7b 2048", "7b", 1, 2048, 2048),
        # a long document
        _prefill("prefill 14b 8192", "14b", 1, 8192, 8192),
        # continuous batching: a prompt comes in, portion by portion, beside requests that decode
        {"name": "mixed 14b 31+1100", "kind": "mixed", "sizes": "14b", "dtype": "bfloat16", "requests": 31, "shortest": 128,
         "longest": 2048, "prompt": 1100, "portion": 512},
        # float32 is what LLM() takes by default: a few users, a prompt, and the 32-bit check of a 7B model
        _decode("decode 0.5b f32 4x512", "0.5b", 4, 512, 512, "float32"),
        _prefill("prefill 0.5b f32 512", "0.5b", 1, 512, 512, "float32"),
        _decode("decode 7b f32 8x300", "7b", 8, 280, 320, "float32"),
        # a busy server's sampling options, all of them
        {"name": "sample 64", "kind": "sample", "requests": 64, "vocab": 152064, "temperature": 0.8, "top_k": 50, "top_p": 0.95,
         "penalty": 1.1, "history": 700},
    ]


def _spread(rng, low: int, high: int) -> int:
    """A whole number, even over the logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng) -> dict:
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "mixed", "decode f32", "prefill f32", "sample"])
    if kind == "sample":
        return {"kind": "sample", "requests": _spread(rng, 1, 200), "vocab": rng.choice([151936, 152064]),
                "temperature": rng.choice([0.0, 0.7, 0.8, 1.0]), "top_k": rng.choice([-1, 20, 50]),
                "top_p": rng.choice([1.0, 0.9, 0.95]), "penalty": rng.choice([1.0, 1.05, 1.1]), "history": _spread(rng, 20, 3000)}
    if kind == "decode f32":
        sizes = rng.choice(["0.5b", "0.5b", "7b"])
        longest = _spread(rng, 64, 1024 if sizes == "0.5b" else 400)
        return _drawn("decode", sizes, "float32", _spread(rng, 1, 16 if sizes == "0.5b" else 8), longest // 2, longest)
    if kind == "prefill f32":
        sizes = rng.choice(["0.5b", "0.5b", "7b"])
        longest = _spread(rng, 16, 2048 if sizes == "0.5b" else 600)
        return _drawn("prefill", sizes, "float32", 1, longest, longest)
    sizes = rng.choice(["0.5b", "7b", "7b", "14b"])
    if kind == "decode":
        requests = _spread(rng, 1, 192)
        longest = _spread(rng, 300, max(300, min(8000, {"0.5b": 300000, "7b": 140000, "14b": 70000}[sizes] // requests)))
        return _drawn("decode", sizes, "bfloat16", requests, rng.randint(max(1, longest // 4), longest), longest)
    if kind == "prefill":
        requests = _spread(rng, 1, 6)
        longest = _spread(rng, 16, {"0.5b": 8192, "7b": 8192, "14b": 6000}[sizes] // requests)
        return _drawn("prefill", sizes, "bfloat16", requests, rng.randint(max(1, longest // 4), longest), longest)
    requests = _spread(rng, 4, 64)
    longest = _spread(rng, 300, 2048)
    return dict(_drawn("mixed", sizes, "bfloat16", requests, longest // 8, longest), prompt=_spread(rng, 200, 2000),
                portion=rng.choice([256, 512, 1024]))


def _drawn(kind, sizes, dtype, requests, shortest, longest) -> dict:
    case = _decode("", sizes, requests, shortest, longest, dtype)
    del case["name"]
    return dict(case, kind=kind)


def _lengths(case) -> list[int]:
    """The requests' lengths: from the shortest to the longest in equal steps."""
    n, low, high = case["requests"], case["shortest"], case["longest"]
    return [high] if n == 1 else [low + (high - low) * i // (n - 1) for i in range(n)]


# ------------------------------------------------------------------------------------------------------------ inputs
def _config(case) -> Qwen2Config:
    layers, width, heads, kv_heads, head_dim, ff, eps, vocab, tied = SIZES[case["sizes"]]
    return Qwen2Config(vocab_size=vocab, hidden_size=width, intermediate_size=ff, num_hidden_layers=layers,
                       num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=head_dim, rms_norm_eps=eps,
                       rope_theta=1e6, max_position_embeddings=32768, tie_word_embeddings=tied)


def _tokens(seed: int, what: str, count: int, vocab: int) -> list[int]:
    gen = torch.Generator().manual_seed(_seed_of(seed, what))
    return torch.randint(0, vocab, (count,), generator=gen).tolist()


def _seed_of(seed: int, name: str) -> int:
    return int.from_bytes(hashlib.sha256(f"{seed}:{name}".encode()).digest()[:8], "little") & ((1 << 63) - 1)


class _Requests:
    """Requests that decode: their prompts are in the cache, each has its own tokens to come."""

    def __init__(self, llm: LLM, case, seed: int) -> None:
        self.llm, vocab = llm, llm.config.vocab_size
        self.prompts = [_tokens(seed, f"prompt {i}", n, vocab) for i, n in enumerate(_lengths(case))]
        self.to_come = [_tokens(seed, f"to come {i}", FOLLOWING, vocab) for i in range(len(self.prompts))]
        self.ids = [f"request {i}" for i in range(len(self.prompts))]
        self.room = _room(case)
        self.live = False
        self.begin()

    def begin(self) -> None:
        runner = self.llm.runner
        for rid in self.ids:
            if self.live:
                runner.end(rid)
            runner.begin(rid)
        self.live, self.grown = True, 0
        for entries in _portions(self.ids, self.prompts):
            runner.step([StepEntry(rid, tokens, []) for rid, tokens, _ in entries])

    def next_entries(self) -> list[StepEntry]:
        if self.grown >= self.room:
            self.begin()
        at, self.grown = self.grown % FOLLOWING, self.grown + 1
        return [StepEntry(rid, [tokens[at]], [0]) for rid, tokens in zip(self.ids, self.to_come)]


FOLLOWING = 61           # tokens to come that a request of a decode case takes in turn


def _room(case) -> int:
    """By how many tokens decoding requests grow before they end: to the next power of two of the longest one's length, as a
    bound on the context would have them, but not by less than a quarter."""
    longest = case["longest"]
    bound = 256
    while bound < longest + max(64, longest // 4):
        bound *= 2
    return bound - longest


def _portions(ids, prompts):
    """Steps of at most BUDGET tokens that take the prompts in: lists of (id, tokens, whether they are the prompt's last)."""
    steps, entries, used = [], [], 0
    for rid, prompt in zip(ids, prompts):
        at = 0
        while at < len(prompt):
            take = min(BUDGET - used, len(prompt) - at)
            entries.append((rid, prompt[at:at + take], at + take == len(prompt)))
            at, used = at + take, used + take
            if used == BUDGET:
                steps.append(entries)
                entries, used = [], 0
    return steps + [entries] if entries else steps


def prepare(case, seed):
    if case["kind"] == "sample":
        return _prepare_sample(case, seed)
    lengths = _lengths(case)
    grown = case["longest"] + (_room(case) if case["kind"] != "prefill" else 0) + PAGE
    pages = len(lengths) * (grown // PAGE + 1) + (case.get("prompt", 0) // PAGE + 1)
    llm = LLM(_config(case), random_seed=seed, dtype=case["dtype"], num_blocks=pages, block_size=PAGE,
              max_concurrent=len(lengths) + 1, device=DEVICE)
    state = {"llm": llm, "case": case}
    if case["kind"] == "prefill":
        state["prompts"] = [_tokens(seed, f"prompt {i}", n, llm.config.vocab_size) for i, n in enumerate(lengths)]
        state["ids"] = [f"request {i}" for i in range(len(lengths))]
        return state
    state["requests"] = _Requests(llm, case, seed)
    if case["kind"] == "mixed":
        state["prompt"] = _tokens(seed, "the prompt", case["prompt"], llm.config.vocab_size)
    llm.runner.step(state["requests"].next_entries())       # a server's decode steps have run before
    return state


def _prepare_sample(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    rows, vocab = case["requests"], case["vocab"]
    logits = torch.randn((rows, vocab), generator=gen, device=DEVICE) * 2.5
    histories = [_tokens(seed, f"history {i}", case["history"], vocab) for i in range(rows)]
    params = SamplingParams(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"],
                            repetition_penalty=case["penalty"])
    from somi_inference_amd.sampling import Sampler
    return {"sampler": Sampler(), "case": case, "logits": logits, "histories": histories, "params": [params] * rows,
            "seeds": [_seed_of(seed, f"stream {i}") for i in range(rows)], "counters": [len(h) for h in histories]}


# ------------------------------------------------------------------------------------------------------------ a pass
def run(state):
    kind = state["case"]["kind"]
    if kind == "sample":
        return state["sampler"].sample(state["logits"], state["params"], token_histories=state["histories"],
                                       seeds=state["seeds"], counters=state["counters"])
    runner = state["llm"].runner
    if kind == "decode":
        return runner.step(state["requests"].next_entries())
    if kind == "prefill":
        for rid in state["ids"]:
            runner.begin(rid)
        outputs = []
        for entries in _portions(state["ids"], state["prompts"]):
            outputs.append(runner.step([StepEntry(rid, tokens, [len(tokens) - 1] if last else []) for rid, tokens, last in entries]))
        for rid in state["ids"]:
            runner.end(rid)
        return outputs
    prompt, portion, outputs = state["prompt"], state["case"]["portion"], []
    runner.begin("prompt")
    for at in range(0, len(prompt), portion):
        tokens = prompt[at:at + portion]
        entries = state["requests"].next_entries()
        entries.append(StepEntry("prompt", tokens, [len(tokens) - 1] if at + portion >= len(prompt) else []))
        outputs.append(runner.step(entries))
    runner.end("prompt")
    return outputs


# ------------------------------------------------------------------------------------------------------------ its cost
def _matrices(case) -> tuple[int, int]:
    """Numbers of weights: of the layers' matrices, and of the head."""
    layers, width, heads, kv_heads, head_dim, ff, _, vocab, _ = SIZES[case["sizes"]]
    return layers * width * ((2 * heads + 2 * kv_heads) * head_dim + 3 * ff), vocab * width


def _steps(case) -> list[tuple[list[tuple[int, int]], int]]:
    """The steps of a pass: ((tokens, tokens in the cache before), ...) and the number of logit rows of each."""
    lengths = _lengths(case)
    if case["kind"] == "prefill":
        steps, done = [], {}
        for entries in _portions(range(len(lengths)), [range(n) for n in lengths]):
            steps.append(([(len(t), done.get(i, 0)) for i, t, _ in entries], sum(last for _, _, last in entries)))
            done.update({i: done.get(i, 0) + len(t) for i, t, _ in entries})
        return steps
    decoding = [(1, n + 1) for n in lengths]
    if case["kind"] == "decode":
        return [(decoding, len(lengths))]
    prompt, portion = case["prompt"], case["portion"]
    return [(decoding + [(min(portion, prompt - at), at)], len(lengths) + (at + portion >= prompt))
            for at in range(0, prompt, portion)]


def work(case) -> dict:
    if case["kind"] == "sample":
        return {"bytes": 4.0 * case["requests"] * case["vocab"], "flops": 0.0}
    layers, _, heads, kv_heads, head_dim, _, _, vocab, _ = SIZES[case["sizes"]]
    item = 2 if case["dtype"] == "bfloat16" else 4
    inner, head = _matrices(case)
    moved = flops = 0.0
    for entries, rows in _steps(case):
        tokens = sum(n for n, _ in entries)
        pairs = sum(n * before + n * (n + 1) / 2 for n, before in entries)
        flops += 2.0 * (tokens * inner + rows * head) + 4.0 * layers * heads * head_dim * pairs
        moved += item * (inner + (head if rows else 0)) + 4.0 * rows * vocab
        moved += 2.0 * item * layers * kv_heads * head_dim * sum(n + before for n, before in entries)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"          # whole numbers: the tokens drawn
    # Measured, one prompt whole against in portions and requests together against each alone: bfloat16 0.006 to 0.008 (0.5b),
    # 0.016 to 0.022 (7b, 14b), at most 0.12 in one logit.  float32 against 64 bits: 4e-6 (0.5b), 3e-5 (7b).
    if case["dtype"] == "bfloat16":
        return {"rel": 3e-2, "max": 0.4}
    return {"rel": 2e-5, "max": 8e-4} if case["sizes"] == "0.5b" else {"rel": 1e-4, "max": 4e-3}


# ------------------------------------------------------------------------------------------------------------ 64 bits
MOST_EXACT = 4e14        # multiplications and additions that 64-bit products get through in some seconds


def exact(case, seed):
    """The same logits from plain torch in float64 (the engine's weights are drawn in float32 by tensor name and rounded once to
    bfloat16, in both of its types)."""
    if case["kind"] == "sample":
        return None
    lengths = _lengths(case)
    mixed = case["kind"] == "mixed"
    vocab = SIZES[case["sizes"]][7]
    sequences = [_tokens(seed, f"prompt {i}", n, vocab) for i, n in enumerate(lengths)]
    wanted = [[n - 1] for n in lengths]
    steps = 1
    if case["kind"] != "prefill":
        steps = -(-case["prompt"] // case["portion"]) if mixed else 1
        for i, n in enumerate(lengths):
            coming = _tokens(seed, f"to come {i}", FOLLOWING, vocab)
            sequences[i] = sequences[i] + [coming[k % FOLLOWING] for k in range(steps + 1)]
            wanted[i] = [n + 1 + k for k in range(steps)]
    if mixed:
        sequences.append(_tokens(seed, "the prompt", case["prompt"], vocab))
        wanted.append([case["prompt"] - 1])
    if 2.0 * sum(map(len, sequences)) * _matrices(case)[0] > MOST_EXACT:
        return None
    rows = _logits(case, seed, sequences, wanted)
    if case["kind"] == "decode":
        return torch.cat(rows)
    if mixed:
        outputs = [torch.stack([r[k] for r in rows[:-1]]) for k in range(steps)]
        outputs[-1] = torch.cat([outputs[-1], rows[-1]])
        return outputs
    outputs, at = [], 0
    for entries in _portions(range(len(lengths)), [range(n) for n in lengths]):
        count = sum(last for _, _, last in entries)
        outputs.append(torch.cat(rows[at:at + count]) if count else torch.empty((0, vocab), dtype=torch.float64))
        at += count
    return outputs


def _logits(case, seed, sequences, wanted):
    layers, width, heads, kv_heads, head_dim, ff, eps, vocab, tied = SIZES[case["sizes"]]

    def weight(name, *shape, mean=0.0, std=0.02):
        gen = torch.Generator(device=DEVICE).manual_seed(_seed_of(seed, name))
        out = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32).mul_(std).add_(mean)
        return out.to(torch.bfloat16).double()

    def norm(h, name):
        return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + eps) * weight(name, width, mean=1.0, std=0.1)

    lengths = [len(s) for s in sequences]
    embedding = weight("model.embed_tokens.weight", vocab, width)
    h = embedding[torch.tensor([t for s in sequences for t in s], device=DEVICE)]
    if not tied:
        del embedding
    positions = torch.cat([torch.arange(n, device=DEVICE, dtype=torch.float64) for n in lengths])
    angles = positions[:, None] / 1e6 ** (torch.arange(0, head_dim, 2, device=DEVICE, dtype=torch.float64) / head_dim)
    cos, sin = angles.cos()[:, None], angles.sin()[:, None]

    def rotated(x):
        low, high = x.chunk(2, dim=-1)
        return torch.cat((low * cos - high * sin, high * cos + low * sin), -1)

    for layer in range(layers):
        at = functools.partial("model.layers.{}.{}".format, layer)
        x = norm(h, at("input_layernorm.weight"))
        q, k, v = (torch.addmm(weight(at(f"self_attn.{name}_proj.bias"), n * head_dim), x,
                               weight(at(f"self_attn.{name}_proj.weight"), n * head_dim, width).t()).view(-1, n, head_dim)
                   for name, n in (("q", heads), ("k", kv_heads), ("v", kv_heads)))
        q, k = rotated(q), rotated(k)
        mixed = torch.cat([_attention(*parts) for parts in zip(q.split(lengths), k.split(lengths), v.split(lengths))])
        h = h + mixed @ weight(at("self_attn.o_proj.weight"), width, heads * head_dim).t()
        x = norm(h, at("post_attention_layernorm.weight"))
        gate = weight(at("mlp.gate_proj.weight"), ff, width).t().contiguous()
        up = weight(at("mlp.up_proj.weight"), ff, width).t().contiguous()
        down = weight(at("mlp.down_proj.weight"), width, ff).t().contiguous()
        h = h + torch.cat([(torch.nn.functional.silu(rows @ gate) * (rows @ up)) @ down for rows in x.split(4096)])
    h = norm(h, "model.norm.weight")
    head = embedding if tied else weight("lm_head.weight", vocab, width)
    return [h[start:start + n][places] @ head.t()
            for start, n, places in zip([sum(lengths[:i]) for i in range(len(lengths))], lengths, wanted)]


def _attention(q, k, v):
    """Causal attention of one sequence: q [T, heads, D], k and v [T, kv heads, D] -> [T, heads * D]."""
    n, heads, dim = q.shape
    groups = heads // k.shape[1]
    out = torch.empty_like(q)
    for start in range(0, n, 1024):
        rows = slice(start, min(start + 1024, n))
        seen = rows.stop
        hidden = torch.arange(seen, device=q.device) > torch.arange(start, seen, device=q.device)[:, None]
        for head in range(heads):
            scores = (q[rows, head] @ k[:seen, head // groups].t()) / math.sqrt(dim)
            out[rows, head] = scores.masked_fill_(hidden, -math.inf).softmax(-1) @ v[:seen, head // groups]
    return out.reshape(n, heads * dim)
