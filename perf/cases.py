"""Performance cases of the decoder stage worker: passes as a serving program issues them
through ``hllm_amd.capi`` (decode batches, prompts prefilled in chunks, passes that mix both,
a whole model's greedy steps, the standalone sampler), over the range of sizes it meets.

A stage case is one stage (a contiguous layer range) of one of the model shapes the tests and
the benchmark use, with seeded synthetic weights:

* ``start`` / ``layers``: the owned layers. Layer 0 takes token IDs, other starts take F16
  N(0, 1) boundary rows; the model's last layer ends in the final norm and the LM head, other
  ends return F16 boundary rows.
* ``rows`` decode rows whose contexts spread log-uniformly over [low, high]. Each pass
  appends one token to every sequence, as a running request does; after ``WINDOW`` tokens the
  requests are renewed.
* ``tokens`` prompt tokens over ``prompts`` prompts of unequal lengths, allocated,
  prefilled in passes of at most ``chunk`` rows, and released within one run.

Outputs are boundary rows (F16), log-probabilities (the greedy token's and the five best),
or logits; ``exact`` computes them in 64 bits from the same seeds.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hllm_amd import capi, model, synthetic

# The head-dim-64 shape of the tests (no QK-norm, untied head) at a whole model's depth.
D64 = synthetic.ModelShape("d64-llama", 16, 2048, 8192, 32, 8, 64, 131072, eps=1e-5, theta=5e5,
                           qk_norm=False, tied=False)
SHAPES = {s.name: s for s in (synthetic.QWEN3_0_6B, synthetic.QWEN3_4B, synthetic.FALCON3_3B, D64)}
BLOCK = 64      # tokens per KV block (the default)
SERVE_STEPS = 8


def listed():
    return [
        # One interactive request on the first half of a small model: the smallest call, where
        # launches and host work count.
        dict(name="decode_1", kind="decode", model="qwen3-0.6b", start=0, layers=14,
             execution="f16", rows=1, low=100, high=100),
        # A handful of requests, head dimension 64: an odd small batch.
        dict(name="decode_7_d64", kind="decode", model="d64-llama", start=0, layers=12,
             execution="f16", rows=7, low=70, high=1100),
        # The benchmark's 64-row decode batch at its mix of contexts (mean about 480), on a
        # third of its layers as a pipeline stage.
        dict(name="decode_64", kind="decode", model="qwen3-4b", start=0, layers=12,
             execution="f16", rows=64, low=32, high=2048),
        # The last pipeline stage at 128 rows with contexts to 8192, LM head and
        # log-probabilities.
        dict(name="decode_128_tail", kind="decode", model="qwen3-4b", start=28, layers=8,
             execution="f16", rows=128, low=1, high=8192),
        # Few requests near the models' longest context: the KV cache is nearly all the work.
        dict(name="decode_3_long", kind="decode", model="qwen3-4b", start=0, layers=4,
             execution="f16", rows=3, low=12000, high=30000),
        # One short prompt on a small model: time to first token.
        dict(name="prefill_45", kind="prefill", model="qwen3-0.6b", start=0, layers=14,
             execution="f16", prompts=1, tokens=45, chunk=512),
        # One long prompt in 512-token chunks, as the continuous-batching loop feeds it.
        dict(name="prefill_2011", kind="prefill", model="qwen3-4b", start=0, layers=8,
             execution="f16", prompts=1, tokens=2011, chunk=512),
        # Several ragged prompts in one large pass, head dimension 256.
        dict(name="prefill_ragged_d256", kind="prefill", model="falcon3-3b", start=0, layers=6,
             execution="f16", prompts=5, tokens=1300, chunk=2048),
        # A continuous-batching step that carries a prompt's chunk beside the decode rows.
        dict(name="mixed_61_448", kind="mixed", model="qwen3-4b", start=0, layers=12,
             execution="f16", rows=61, low=32, high=2048, tokens=448),
        # F32 execution (the parity mode) with F16-resident weights, prompt and decode rows.
        dict(name="mixed_f32", kind="mixed", model="qwen3-0.6b", start=0, layers=6,
             execution="f32", rows=13, low=32, high=700, tokens=83),
        # The sampler on a caller's own logits: temperature, top-k, top-p and log-probabilities.
        dict(name="sample_16", kind="sample", rows=16, vocabulary=151936),
        # A whole model serving 64 requests: greedy steps that return tokens only, then one
        # that returns two requests' logits.
        dict(name="serve_64", kind="serve", model="qwen3-4b", start=0, layers=36,
             execution="f16", rows=64, low=32, high=1500),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "mixed", "mixed", "sample"])
    if kind == "sample":
        return dict(kind=kind, rows=_log_int(rng, 1, 32), vocabulary=_log_int(rng, 4096, 151936))
    name = rng.choice(sorted(SHAPES))
    execution = "f16"
    if name == "qwen3-0.6b" and rng.random() < 0.3:
        execution = "f32"
    layers = rng.randint(2, 4) if execution == "f32" else rng.randint(4, 10)
    final = kind == "decode" and rng.random() < 0.25
    start = SHAPES[name].layers - layers if final else rng.choice([0, SHAPES[name].layers - layers - 1])
    case = dict(kind=kind, model=name, start=start, layers=layers, execution=execution)
    if kind in ("decode", "mixed"):
        case["rows"] = _log_int(rng, 1, (16 if execution == "f32" else 64 if kind == "mixed" else 128))
        case["low"] = _log_int(rng, 1, 300)
        # At most about 116 000 cached tokens in all, and 30 000 in one sequence.
        most = 700 if execution == "f32" else 2048 if kind == "mixed" else \
            30000 if case["rows"] < 4 else 8192
        case["high"] = _log_int(rng, case["low"], most)
    if kind == "prefill":
        case["tokens"] = _log_int(rng, 16, 256 if execution == "f32" else 2048)
        case["prompts"] = rng.randint(1, min(8, case["tokens"] // 16))
        case["chunk"] = rng.choice([512, 2048])
    if kind == "mixed":
        case["tokens"] = _log_int(rng, 8, 128 if execution == "f32" else 512)
    return case


# ------------------------------------------------------------------ what a case means


def _contexts(case):
    """Each decode row's context at the first pass: log-uniform quantiles of [low, high]."""
    n, low, high = case["rows"], case["low"], case["high"]
    return [max(1, int(round(low * (high / low) ** ((i + 0.5) / n)))) for i in range(n)]


def _prompts(case):
    """The prompts' lengths: unequal shares of `tokens`."""
    n = case.get("prompts", 1)
    weights = [1 + (5 * i + 2) % 7 for i in range(n)]
    lengths = [max(1, case["tokens"] * w // sum(weights)) for w in weights]
    lengths[0] += case["tokens"] - sum(lengths)
    return lengths


def _window(case):
    return 256 if sum(_contexts(case)) < 4096 else 1024


def _shape(case):
    return SHAPES[case["model"]]


def _inputs(case, seed, index, count):
    """The input of `count` positions of sequence `index`: token IDs (numpy), or F16 boundary
    rows (a tensor on the GPU) for a stage that does not hold layer 0."""
    if case["start"] == 0:
        rng = np.random.default_rng([seed, index])
        return rng.integers(0, _shape(case).vocab, count).astype(np.uint64)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 4099 + index)
    return torch.randn(count, _shape(case).hidden, generator=g, device="cuda").half()


def _host(x):
    return x if isinstance(x, np.ndarray) else x.cpu().numpy().view(np.uint16)


def _feed(case, parts):
    """execute()'s input arguments for the concatenation of host inputs."""
    joined = parts[0] if len(parts) == 1 else np.concatenate(parts)
    return {"token_ids": joined} if case["start"] == 0 else {"boundary": joined}


def _sample_logits_inputs(case, seed):
    """Logits with a few likely tokens over a broad tail, as a trained model's are."""
    rng = np.random.default_rng(seed)
    logits = 2.0 * rng.standard_normal((case["rows"], case["vocabulary"]), dtype=np.float32)
    for r in range(case["rows"]):
        logits[r, rng.integers(0, case["vocabulary"], 40)] += rng.uniform(4.0, 12.0, 40).astype(np.float32)
    return logits


# ------------------------------------------------------------------ prepare and run


class _State:
    """A stage with its running requests."""

    def __init__(self, case, seed):
        self.case, self.seed = case, seed
        shape = _shape(case)
        c = case
        self.contexts = _contexts(c) if "rows" in c else []
        self.prompts = _prompts(c) if "tokens" in c else []
        self.window = _window(c) if self.contexts else 0
        element = 2 if c["execution"] == "f16" else 4
        held = [n + self.window + 1 for n in self.contexts] + self.prompts
        blocks = sum(-(-n // BLOCK) for n in held) + 8
        cfg = model.stage_config(
            shape, c["start"], c["start"] + c["layers"], first=c["start"] == 0,
            final=c["start"] + c["layers"] == shape.layers, execution=c["execution"],
            kv_cache_bytes=blocks * BLOCK * shape.kv_bytes_per_token(c["layers"], element),
            max_sequences=len(held) + 1, max_pass_rows=2048)
        self.final = bool(cfg.final_stage)
        self.stage = capi.Stage(cfg)
        model.synthesize(self.stage, shape, seed=seed)
        self.items, self.steps = [], 0
        if self.contexts:
            # The next tokens of every request (the sampled ones of an earlier pass, or given).
            self.feed = _feed(c, [_host(_inputs(c, seed, i, n + 1))[n:] for i, n in enumerate(self.contexts)])
            self.admit()
        if self.prompts:
            self.prompt_inputs = [_host(_inputs(c, seed, 1000 + i, n)) for i, n in enumerate(self.prompts)]
        if c["kind"] == "mixed":
            self.feed = _feed(c, [v for v in self.feed.values()] + self.prompt_inputs)

    def admit(self):
        """Renews the decode requests: their contexts are prefilled in passes of 2048 rows."""
        for item in self.items:
            self.stage.release(item.sequence)
        self.steps = 0
        sequences = [self.stage.allocate(n + self.window + 1) for n in self.contexts]
        whole = [_host(_inputs(self.case, self.seed, i, n + 1)) for i, n in enumerate(self.contexts)]
        for items, parts in _plan(sequences, self.contexts, whole, 2048, sample_last=False):
            self.stage.execute(items, **_feed(self.case, parts))
        logprobs = self.final and self.case["kind"] != "serve"
        self.items = [capi.item(s, 1, n, sample=self.final, logprobs=logprobs,
                                top_logprobs=5 if logprobs else 0)
                      for s, n in zip(sequences, self.contexts)]

    def advance(self):
        """One token more for every request."""
        self.steps += 1
        for item in self.items:
            item.first_position += 1


def _plan(sequences, lengths, inputs, chunk, sample_last):
    """Passes of at most `chunk` rows over the sequences' inputs: (items, input parts)."""
    items, parts, room = [], [], chunk
    for s, n, x in zip(sequences, lengths, inputs):
        at = 0
        while at < n:
            take = min(room, n - at)
            items.append(capi.item(s, take, at, sample=sample_last and at + take == n))
            parts.append(x[at:at + take])
            at, room = at + take, room - take
            if room == 0:
                yield items, parts
                items, parts, room = [], [], chunk
    if items:
        yield items, parts


def prepare(case, seed):
    if case["kind"] == "sample":
        options = [capi.item(0, 1, 0, temperature=0.7 + 0.02 * r, top_p=0.9, top_k=0 if r % 2 else 50,
                             seed=seed + r, generated_index=r, logprobs=True, top_logprobs=5)
                   for r in range(case["rows"])]
        return {"logits": _sample_logits_inputs(case, seed), "options": options}
    return _State(case, seed)


def run(state):
    if isinstance(state, dict):
        tokens, logprobs, _, top = capi.sample_logits(state["logits"], state["options"])
        return {"tokens": tokens.view(np.int64), "logprobs": logprobs, "top_logprobs": top}
    kind, stage = state.case["kind"], state.stage
    if kind == "prefill":
        sequences = [stage.allocate(n) for n in state.prompts]
        out = [stage.execute(items, **_feed(state.case, parts))["boundary"].view(np.float16)
               for items, parts in _plan(sequences, state.prompts, state.prompt_inputs, state.case["chunk"],
                                         sample_last=state.final)]
        for s in sequences:
            stage.release(s)
        return out
    if kind == "serve":
        if state.steps + SERVE_STEPS > state.window:
            state.admit()
        tokens = []
        for _ in range(SERVE_STEPS):
            tokens.append(stage.execute(state.items, **state.feed)["tokens"].view(np.int64))
            state.advance()
        # The last pass samples two requests and returns their logits; the others only extend
        # their caches.
        few = state.items[::len(state.items) // 2][:2]
        for item in state.items:
            item.flags = capi.ITEM_SAMPLE if any(item is f for f in few) else 0
        logits = stage.execute(state.items, **state.feed, want_logits=True)["logits"]
        for item in state.items:
            item.flags = capi.ITEM_SAMPLE
        state.advance()
        return {"tokens": tokens, "logits": logits}
    if state.steps == state.window:
        state.admit()
    if kind == "mixed":
        sequence = stage.allocate(state.prompts[0])
        items = state.items + [capi.item(sequence, state.prompts[0], 0, sample=False)]
        out = stage.execute(items, **state.feed)
        stage.release(sequence)
    else:
        out = stage.execute(state.items, **state.feed)
    state.advance()
    if state.final:
        return {"logprobs": out["logprobs"], "top_logprobs": out["top_logprobs"]}
    return out["boundary"].view(np.float16)


# ------------------------------------------------------------------ work and tolerance


def work(case):
    if case["kind"] == "sample":
        n = case["rows"] * case["vocabulary"]
        return {"bytes": n * 4 + case["rows"] * 64, "flops": n * 4}
    shape = _shape(case)
    layers, element = case["layers"], 2 if case["execution"] == "f16" else 4
    passes = SERVE_STEPS + 1 if case["kind"] == "serve" else 1
    per_layer = shape.layer_weight_bytes(1)
    kv = shape.kv_bytes_per_token(layers, element)
    contexts = _contexts(case) if "rows" in case else []
    prompts = _prompts(case) if "tokens" in case else []
    rows = len(contexts) + sum(prompts)
    attended = sum(n + 1 for n in contexts) + sum(n * (n + 1) // 2 for n in prompts)
    cached = sum(n + 1 for n in contexts) + sum(prompts)  # each cached token once per pass
    transport = rows * shape.hidden * 2
    total = per_layer * layers * 2 + cached * kv + rows * kv + transport
    flops = 2.0 * rows * per_layer * layers + 4.0 * attended * shape.heads * shape.head_dim * layers
    if case["start"] + layers == shape.layers:
        total += shape.vocab * shape.hidden * 2
        flops += 2.0 * len(contexts) * shape.vocab * shape.hidden
    else:
        total += transport
    return {"bytes": float(total * passes), "flops": float(flops * passes)}


def tolerance(case):
    if case["kind"] == "sample":
        return {"rel": 1e-11, "max": 1e-10, "differ": 0.0}
    if case["execution"] == "f32":
        # F32 stages differ from `exact` by the F16 rounding of the boundary (2.1e-4).
        return {"rel": 8e-4, "max": 4e-3}
    if case["kind"] == "serve":
        # 36 layers; near ties of the top two logits turn about 3 greedy tokens in 1000.
        return {"rel": 1.5e-2, "max": 1e-1, "differ": 0.01}
    if case["kind"] == "decode" and case["start"] + case["layers"] == _shape(case).layers:
        return {"rel": 5e-4, "max": 5e-3}  # log-probabilities: 1.1e-4 from `exact`
    # F16 stages of up to 12 layers are 0.7e-3 to 2e-3 from `exact`.
    return {"rel": 6e-3, "max": 4e-2}


# ------------------------------------------------------------------ 64-bit values


def _lsr(x, bits):
    return (x >> bits) & ((1 << (64 - bits)) - 1)


def _signed(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _elements(seed, tensor, index, mean, sigma):
    """Elements `index` (int64, on the GPU) of a synthetic F16 tensor, as F64: the definition
    in hllm_amd/synthetic.py."""
    total = torch.zeros_like(index)
    for j in range(3):
        z = (index * 3 + ((tensor << 40) + j + 1)) * _signed(0x9E3779B97F4A7C15) + _signed(seed)
        z = (z ^ _lsr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
        z = (z ^ _lsr(z, 27)) * _signed(0x94D049BB133111EB)
        z = z ^ _lsr(z, 31)
        for k in range(4):
            total += (z >> (16 * k)) & 0xFFFF
    n = (total + (6 - 6 * 65536)).float() / 65536
    value = n * torch.tensor(sigma, dtype=torch.float32, device="cuda")
    return (value + torch.tensor(mean, dtype=torch.float32, device="cuda")).half().double()


def _tensor(shape, seed, name):
    tensor, dims, mean, sigma = synthetic.tensor_spec(shape, name)
    n = math.prod(dims)
    parts = [_elements(seed, tensor, torch.arange(at, min(n, at + (1 << 24)), device="cuda"), mean, sigma)
             for at in range(0, n, 1 << 24)]
    return torch.cat(parts).reshape(dims)


def _norm(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _rope(x, position, theta):
    """Rotate-half RoPE of [n, heads, d] at `position` [n]."""
    d = x.shape[-1]
    rate = theta ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    angle = position.double()[:, None] * rate[None, :]
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend(q, k, v, last):
    """Causal attention of [n, heads, d] over [n, kv heads, d]; only row n - 1 where `last`."""
    n, heads, d = q.shape
    group = heads // k.shape[1]
    kt = k.permute(1, 2, 0).contiguous()              # [kv, d, n]
    vt = v.permute(1, 0, 2).contiguous()              # [kv, n, d]
    out = torch.zeros_like(q)
    step = max(1, (1 << 27) // (n * heads))
    for at in range(n - 1 if last else 0, n, step):
        to = min(n, at + step)
        block = q[at:to].reshape(to - at, k.shape[1], group, d).permute(1, 2, 0, 3)
        block = block.reshape(k.shape[1], group * (to - at), d).contiguous()
        score = torch.matmul(block, kt[:, :, :to].contiguous()) / math.sqrt(d)
        score = score.view(k.shape[1], group, to - at, to)
        beyond = torch.arange(to, device="cuda")[None, :] > torch.arange(at, to, device="cuda")[:, None]
        score = score.masked_fill(beyond, -math.inf).softmax(-1).view(k.shape[1], group * (to - at), to)
        got = torch.matmul(score, vt[:, :to].contiguous()).view(k.shape[1], group, to - at, d)
        out[at:to] = got.permute(2, 0, 1, 3).reshape(to - at, heads, d)
    return out


def _stage64(case, seed, lengths, inputs, only_last):
    """The stage's output rows in 64 bits, per sequence: every position, or the last one where
    only_last[i]."""
    shape = _shape(case)
    if case["start"] == 0:
        ids = torch.from_numpy(np.concatenate(inputs).astype(np.int64)).cuda()
        tensor, _, mean, sigma = synthetic.tensor_spec(shape, "model.embed_tokens.weight")
        column = torch.arange(shape.hidden, device="cuda")
        x = torch.cat([_elements(seed, tensor, part[:, None] * shape.hidden + column, mean, sigma)
                       for part in ids.split(4096)])
    else:
        x = torch.cat(inputs).double()
    position = torch.cat([torch.arange(n, device="cuda") for n in lengths])
    heads, kv, d = shape.heads, shape.kv_heads, shape.head_dim
    for layer in range(case["start"], case["start"] + case["layers"]):
        def weight(name):
            return _tensor(shape, seed, f"model.layers.{layer}.{name}.weight")
        qkv = torch.cat([weight(f"self_attn.{p}_proj") for p in "qkv"]).t().contiguous()
        y = torch.empty(x.shape[0], (heads + 2 * kv) * d, dtype=torch.float64, device="cuda")
        for at in range(0, x.shape[0], 8192):
            y[at:at + 8192] = _norm(x[at:at + 8192], shape.eps) @ qkv
        del qkv
        y = y.view(-1, heads + 2 * kv, d)
        out_t = weight("self_attn.o_proj").t().contiguous()
        at = 0
        for n, last in zip(lengths, only_last):
            q, k, v = y[at:at + n].split([heads, kv, kv], 1)
            if shape.qk_norm:
                q, k = _norm(q, shape.eps), _norm(k, shape.eps)
            p = position[at:at + n]
            last_layer = layer == case["start"] + case["layers"] - 1
            got = _attend(_rope(q, p, shape.theta), _rope(k, p, shape.theta), v, last and last_layer)
            x[at:at + n] += got.reshape(n, -1) @ out_t
            at += n
        del y, out_t
        gate, up, down = (weight(f"mlp.{p}_proj").t().contiguous() for p in ("gate", "up", "down"))
        for at in range(0, x.shape[0], 8192):
            z = _norm(x[at:at + 8192], shape.eps)
            x[at:at + 8192] += (torch.nn.functional.silu(z @ gate) * (z @ up)) @ down
        del gate, up, down
    rows, at = [], 0
    for n, last in zip(lengths, only_last):
        rows.append(x[at + n - 1:at + n] if last else x[at:at + n])
        at += n
    return rows


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        logits = torch.from_numpy(_sample_logits_inputs(case, seed)).double()
        return {"tokens": None, "logprobs": None, "top_logprobs": logits.log_softmax(-1).topk(5).values.numpy()}
    if kind == "serve":
        return None
    contexts = _contexts(case) if "rows" in case else []
    prompts = _prompts(case) if "tokens" in case else []
    lengths = [n + 1 for n in contexts] + prompts
    index = list(range(len(contexts))) + [1000 + i for i in range(len(prompts))]
    inputs = [_inputs(case, seed, i, n) for i, n in zip(index, lengths)]
    rows = _stage64(case, seed, lengths, inputs, [True] * len(contexts) + [False] * len(prompts))
    shape = _shape(case)
    if case["start"] + case["layers"] == shape.layers and kind == "decode":
        x = _norm(torch.cat(rows), shape.eps)
        name = "model.embed_tokens.weight" if shape.tied else "lm_head.weight"
        tensor, dims, mean, sigma = synthetic.tensor_spec(shape, name)
        column = torch.arange(shape.hidden, device="cuda")
        parts = []
        for part in torch.arange(dims[0], device="cuda").split(8192):
            w = _elements(seed, tensor, part[:, None] * shape.hidden + column, mean, sigma)
            parts.append(x @ w.t().contiguous())
        top = torch.cat(parts, 1).log_softmax(-1).topk(5).values.cpu().numpy()
        return {"logprobs": top[:, 0].copy(), "top_logprobs": top}
    out = torch.cat(rows).cpu().numpy()
    if kind == "prefill":
        return [out[at:at + case["chunk"]] for at in range(0, len(out), case["chunk"])]
    return out
