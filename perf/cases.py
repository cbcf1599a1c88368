"""The work a user has this package do on one GPU, as cases that can be timed and checked.

Every case is one call (or one fixed group of calls) of the public Python API on a model that the
program already holds: text generation, KV-cached decode, prompt prefill, scoring, gradients and
training steps, from the command line's small default model to the largest benchmark workload.
Shapes are the package's named workloads (``named_config``), the defaults of ``mesh-gpt train``,
``generate`` and ``mesh-gpt-bench``, and sizes between them.  ``exact`` restates the model in
64-bit torch.
"""
import math

import numpy as np
import torch

import grokking_abmod_amd as G

EPS = 1e-5
LEARNING_RATE, WEIGHT_DECAY, BETA1, BETA2, ADAM_EPS = 1e-3, 0.1, 0.9, 0.98, 1e-8

_MODELS = {
    # mesh-gpt train / generate without flags: the demo corpus has 28 characters
    "demo": dict(vocab=28, context=32, width=32, heads=4, layers=2, attention=4, ffn=6, butterfly=False),
    "tiny": dict(vocab=64, context=256, width=128, heads=4, layers=2, attention=7, ffn=7, butterfly=True),
    "symbolic": dict(vocab=99, context=4, width=128, heads=4, layers=2, attention=4, ffn=6, butterfly=False),
    "mid": dict(vocab=256, context=1024, width=512, heads=8, layers=6, attention=9, ffn=9, butterfly=True),
    "long": dict(vocab=256, context=8448, width=512, heads=8, layers=4, attention=9, ffn=9, butterfly=True),
    "high": dict(vocab=256, context=2048, width=1024, heads=16, layers=12, attention=10, ffn=10, butterfly=True),
}


def _case(call, model, batch, tokens, steps=0, temperature=0.0, last_only=True, answers=False, init="reference",
          **over):
    c = dict(call=call, **_MODELS[model])
    c.update(batch=batch, tokens=tokens, steps=steps, temperature=temperature, last_only=last_only, answers=answers,
             init=init)
    c.update(over)
    return c


def listed():
    cases = {
        # `mesh-gpt generate` as it comes: one prompt, 240 sampled characters; past 32 tokens the window slides and
        # every token recomputes it.  The smallest work, all latency.
        "demo_generate": _case("generate", "demo", 1, 17, steps=240, temperature=0.7),
        # An interactive completion on the small benchmark model: batch 1, 128 greedy tokens from the cache.
        "tiny_generate": _case("generate", "tiny", 1, 16, steps=128),
        # Serving in mid flight: 32 sequences, half a context long, decode on from their caches.
        "mid_decode": _case("decode", "mid", 32, 449, steps=48),
        # Few sequences over a very long context.
        "long_decode": _case("decode", "long", 8, 8192, steps=24, init="normal"),
        # The largest serving batch: 256 sequences of the largest model.
        "high_decode": _case("decode", "high", 256, 128, steps=8),
        # A batch of long documents read before generation.
        "long_prefill": _case("prefill", "long", 8, 8192),
        # Many ordinary prompts on the largest model.
        "high_prefill": _case("prefill", "high", 256, 128, init="normal"),
        # Scoring the complete equation table, as each evaluation of `mesh-gpt grok` does.
        "symbolic_logits": _case("logits", "symbolic", 9409, 4),
        # Scoring text: every position's logits for ragged windows of 1001 tokens.
        "mid_logits": _case("logits", "mid", 9, 1001, last_only=False, init="normal"),
        # One update of `mesh-gpt-bench` and `mesh-gpt grok`: 512 equations, the answers supervised.
        "symbolic_train": _case("train", "symbolic", 512, 4, answers=True),
        # One update of `mesh-gpt train` on the demo corpus: 8 windows of 32 characters.
        "demo_train": _case("train", "demo", 8, 32),
        # The gradient of a text batch on the mid-sized model.
        "mid_gradient": _case("gradient", "mid", 8, 512),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    call = rng.choice(["generate", "decode", "prefill", "logits", "train", "gradient"])
    init = rng.choice(["reference", "normal"])
    if call == "generate":
        if rng.random() < 0.5:  # small models, the window sliding for the later tokens
            c = _case(call, "demo", _spread(rng, 1, 4), rng.randint(1, 30), steps=_spread(rng, 24, 160))
            c.update(width=rng.choice([32, 64, 128]), context=rng.randint(24, 64), layers=rng.randint(1, 3))
        else:
            c = _case(call, "tiny", _spread(rng, 1, 16), rng.randint(5, 100), steps=_spread(rng, 24, 150))
            c.update(butterfly=rng.random() < 0.7)
        c["temperature"] = rng.choice([0.0, 0.7]) if c["batch"] == 1 else 0.0
    elif call == "decode":
        model = rng.choice(["mid", "long", "high"])
        batch = _spread(rng, 1, {"mid": 48, "long": 8, "high": 128}[model])
        tokens = _spread(rng, 40, {"mid": 900, "long": 6000, "high": 300}[model])
        c = _case(call, model, batch, tokens, steps=rng.randint(4, 24))
        c.update(context=tokens + c["steps"] + rng.randint(0, 60), layers=rng.randint(2, c["layers"]))
    elif call == "prefill":
        model = rng.choice(["tiny", "mid", "long", "high"])
        tokens = _spread(rng, 20, {"tiny": 250, "mid": 1000, "long": 7000, "high": 1500}[model])
        c = _case(call, model, max(1, min(_spread(rng, 1, 256), 30000 // tokens)), tokens)
        c.update(context=tokens + rng.randint(1, 60), layers=rng.randint(2, c["layers"]))
    elif call == "logits":
        model = rng.choice(["symbolic", "demo", "tiny", "mid"])
        tokens = rng.randint(2, 4) if model == "symbolic" else _spread(rng, 9, _MODELS[model]["context"])
        rows = _spread(rng, 500, 30000 if model != "mid" else 9000)
        c = _case(call, model, max(1, rows // tokens), tokens, last_only=rng.random() < 0.5)
    else:
        model = rng.choice(["symbolic", "demo", "tiny", "mid"])
        tokens = rng.randint(3, 4) if model == "symbolic" else _spread(rng, 8, min(512, _MODELS[model]["context"]))
        rows = _spread(rng, 200, 4000 if model != "mid" else 3500)
        c = _case(call, model, max(1, rows // tokens), tokens, answers=model == "symbolic")
        if model in ("tiny", "mid"):
            c.update(width=rng.choice([64, 128, 256] if model == "tiny" else [256, 512, 1024]), layers=rng.randint(1, 3))
    c["init"] = "reference" if call in ("train", "gradient") else init
    return c


# ---- inputs, from the seed alone


def _parameters(case, seed):
    """The package's seeded initialisation in distribution (edges 0.7 +- 0.1 and +- 0.2, each stack's last layer at
    0.3 of that), or N(0, 0.5^2) edges; flat, in parameter order."""
    rng = np.random.default_rng([seed, 1])
    W, A, F = case["width"], case["attention"], case["ffn"]
    stacks = [A] + [A, A, A, A, F] * case["layers"]
    parts = []
    for depth in stacks:
        if case["init"] == "normal":
            w = 0.5 * rng.standard_normal((depth, W, 2))
        else:
            w = rng.random((depth, W, 2))
            w[..., 0] = 0.6 + 0.2 * w[..., 0]
            w[..., 1] = 0.4 * (w[..., 1] - 0.5)
            w[-1] *= 0.3
        parts.append(w.reshape(-1))
    return np.concatenate(parts).astype(np.float32)


def _tokens(case, seed):
    """(inputs, targets), batch x tokens each.  Equations are (a, operator, b, equals) with the answer supervised;
    other batches are uniform tokens with every next token supervised."""
    rng = np.random.default_rng([seed, 2])
    B, S, V = case["batch"], case["tokens"], case["vocab"]
    stream = rng.integers(0, V, (B, S + 1), dtype=np.uint32)
    inputs, targets = stream[:, :-1].copy(), stream[:, 1:].copy()
    if case["answers"]:
        inputs[:, 1] = V - 2
        inputs[:, -1] = V - 1
        targets[:, :-1] = G.IGNORE_TARGET
    return inputs, targets


def prepare(case, seed):
    config = G.GptConfig(vocab_size=case["vocab"], context=case["context"], width=case["width"], heads=case["heads"],
                         layers=case["layers"], attention_mesh_depth=case["attention"], ffn_mesh_depth=case["ffn"],
                         connectivity=int(case["butterfly"]), long_context=int(case["context"] > 4096))
    serving = case["call"] in ("generate", "decode", "prefill")
    model = G.MeshGpt(0, config, 7, max_batch=case["batch"] if serving else 1)
    model.set_parameters(_parameters(case, seed))
    inputs, targets = _tokens(case, seed)
    state = dict(case=case, seed=int(seed), model=model, inputs=inputs, targets=targets)
    if case["call"] == "train":
        state["options"] = G.AdamW(learning_rate=LEARNING_RATE, weight_decay=WEIGHT_DECAY, beta1=BETA1, beta2=BETA2,
                                   epsilon=ADAM_EPS)
    if case["call"] == "decode":
        model.prefill(inputs, case["temperature"], state["seed"], reserve=case["tokens"] + case["steps"] + 1)
    return state


def run(state):
    case, model = state["case"], state["model"]
    call, batch, tokens = case["call"], case["batch"], case["tokens"]
    if call == "generate":
        out = model.generate_tokens(state["inputs"], case["steps"], case["temperature"], state["seed"])
        return {"tokens": out, "logits": model.last_logits(batch)}
    if call == "prefill":
        model.prefill(state["inputs"], case["temperature"], state["seed"])
        return {"tokens": model.read_tokens(batch), "logits": model.last_logits(batch)}
    if call == "decode":
        model.rewind()
        model.decode(case["steps"])
        return {"tokens": model.read_tokens(batch), "logits": model.last_logits(batch)}
    if call == "logits":
        return {"logits": model.logits(state["inputs"], tokens, case["last_only"])}
    if call == "gradient":
        loss, gradient = model.loss_and_gradient(state["inputs"], state["targets"], tokens)
        return {"loss": loss, "gradient": gradient}
    loss = model.train_batch(state["inputs"], state["targets"], tokens, state["options"])
    return {"loss": loss, "parameters": model.parameters()}


# ---- what a pass cannot do without


def work(case):
    """Weights, tokens and outputs once, and for each decode step the cached keys and values it attends over; a mesh
    layer is two multiply-adds a channel.  A prefill whose only output is each sequence's last row needs the last
    block's keys and values of every row, and the rest of that block for the last rows alone."""
    W, L, V, A, F = (case[k] for k in ("width", "layers", "vocab", "attention", "ffn"))
    B, S, steps = case["batch"], case["tokens"], case["steps"]
    weights = 8 * W * (A + L * (4 * A + F))

    def forward(rows, first, last_only):
        """Operations of one pass over `rows` new positions of each sequence after `first` cached ones."""
        pairs = rows * first + rows * (rows + 1) // 2
        flops = (L - 1) * B * (4 * W * (4 * A + F) * rows + 4 * W * pairs)
        if last_only:
            return flops + B * (4 * W * (2 * A * rows + 2 * A + F) + 4 * W * (first + rows) + 2 * W * V)
        return flops + B * (4 * W * (4 * A + F) * rows + 4 * W * pairs + 2 * W * V * rows)

    call = case["call"]
    if call == "generate":
        flops = traffic = 0
        length = S
        cached = 0
        for _ in range(steps):
            window = min(length, case["context"])
            first = cached if length <= case["context"] else 0
            flops += forward(window - first, first, True)
            traffic += weights + 4 * V * W + 8 * L * B * W * window
            cached = window
            length += 1
        return {"bytes": traffic, "flops": flops}
    if call == "decode":
        flops = sum(forward(1, S + i, True) for i in range(steps))
        traffic = sum(weights + 4 * V * W + 8 * L * B * W * (S + i + 1) for i in range(steps))
        return {"bytes": traffic, "flops": flops}
    if call == "prefill":
        return {"bytes": weights + 4 * B * S + 8 * L * B * W * S + 4 * B * V, "flops": forward(S, 0, True)}
    if call == "logits":
        rows = 1 if case["last_only"] else S
        return {"bytes": weights + 4 * B * S + 4 * B * V * rows, "flops": forward(S, 0, case["last_only"])}
    # forward and backward: per mesh layer two multiply-adds forward and four backward; per attention pair and channel
    # two and four; three products of the head
    pairs = S * (S + 1) // 2
    flops = B * (L * (12 * W * (4 * A + F) * S + 12 * W * pairs) + 6 * W * V * S) + 12 * V * W * A
    state = weights // 4 * (24 if call == "train" else 8)
    return {"bytes": state + 8 * B * S, "flops": flops}


def tolerance(case):
    """32-bit sums in another order, through the whole model: against 64 bits the logits are 1e-7 to 2e-6 off (N(0,
    0.5) weights the most) and gradients 1e-7, and this is about four times the most.  A generated token differs only
    where two are tied within rounding.  An AdamW update of a fresh model is the gradient's sign times the learning
    rate, so a gradient that is itself rounding moves its parameter by up to twice that."""
    if case["call"] in ("generate", "decode", "prefill"):
        return {"rel": 1e-5, "max": 4e-4, "differ": 0.01}
    if case["call"] == "train":
        return {"rel": 1e-4, "max": 1e-2}
    return {"rel": 1e-5, "max": 4e-4}


# ---- the model in 64 bits


class _Exact:
    """The forward pass in float64 torch: mesh stacks, RMSNorm, QK-Norm, slice RoPE, causal attention, exclusive
    self-attention and the tied head."""

    def __init__(self, case, parameters):
        self.c = case
        dev = parameters.device
        W, A, F = case["width"], case["attention"], case["ffn"]
        self.flat = parameters
        depths = [A] + [A, A, A, A, F] * case["layers"]
        self.stacks, at = [], 0
        for depth in depths:
            n = depth * W * 2
            self.stacks.append(parameters[at:at + n].view(depth, W, 2))
            at += n
        self.E = self.mesh(self._codes().to(dev), self.stacks[0])

    def _codes(self):
        V, W = self.c["vocab"], self.c["width"]
        bits = (V - 1).bit_length()
        masks = [1 << b for b in range(bits)] + [m for m in range(1, 1 << bits) if m & (m - 1)]
        code = np.empty((V, W))
        token = np.arange(V)
        for channel in range(W):
            word = token & masks[channel % len(masks)]
            odd = np.zeros(V, dtype=np.int64)
            for b in range(bits):
                odd ^= (word >> b) & 1
            code[:, channel] = np.where(odd == 0, -1.0, 1.0)
        return torch.from_numpy(code)

    def mesh(self, x, stack):
        W, depth = self.c["width"], stack.shape[0]
        levels = W.bit_length() - 1
        for layer in range(depth):
            stride = (1 << (layer % levels)) if self.c["butterfly"] else 1
            x = x * stack[layer, :, 0] + torch.roll(x, -stride, -1) * stack[layer, :, 1]
            if layer + 1 < depth:
                x = torch.where(x >= 0, x, torch.expm1(torch.clamp(x, max=0.0)))
        return x

    @staticmethod
    def norm(x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)

    def heads(self, x):
        B, S, W = x.shape
        H = self.c["heads"]
        return x.view(B, S, H, W // H).transpose(1, 2).contiguous()

    def rope(self, x, first):
        half = x.shape[-1] // 2
        pos = torch.arange(first, first + x.shape[2], dtype=torch.float64, device=x.device)
        rate = 10000.0 ** (torch.arange(half, dtype=torch.float64, device=x.device) / half)
        angle = pos[:, None] / rate
        cos, sin = torch.cos(angle), torch.sin(angle)
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def attend(self, q, k, v, first):
        """Rows of q sit at positions first, first + 1, ...; k and v hold every position from 0."""
        B, H, S, hd = q.shape
        T = k.shape[2]
        kt = k.transpose(-1, -2).contiguous()
        step = max(1, min(S, (1 << 28) // (B * H * T)))
        out = []
        at = torch.arange(T, device=q.device)
        for i in range(0, S, step):
            rows = q[:, :, i:i + step].contiguous()
            score = torch.matmul(rows, kt) / math.sqrt(hd)
            past = at[None, :] > (torch.arange(i, i + rows.shape[2], device=q.device) + first)[:, None]
            score = score.masked_fill(past, -math.inf)
            out.append(torch.matmul(torch.softmax(score, -1), v))
        return torch.cat(out, 2)

    def forward(self, tokens, cache=None, first=0):
        """Final normalised rows of tokens (batch x rows); with `cache` (a list of each block's k and v) the rows
        follow the cached ones and are added to them."""
        x = self.E[tokens]
        for b in range(self.c["layers"]):
            wq, wk, wv, wp, wf = self.stacks[1 + 5 * b:6 + 5 * b]
            n = self.norm(x)
            q, k, v = (self.heads(self.mesh(n, w)) for w in (wq, wk, wv))
            q, k = self.rope(self.norm(q), first), self.rope(self.norm(k), first)
            own = v
            if cache is not None:
                if len(cache) > b:
                    k, v = torch.cat([cache[b][0], k], 2), torch.cat([cache[b][1], v], 2)
                    cache[b] = (k, v)
                else:
                    cache.append((k, v))
            y = self.attend(q, k, v, first)
            u = own / torch.clamp(own.norm(dim=-1, keepdim=True), min=1e-12)
            y = y - (y * u).sum(-1, keepdim=True) * u
            x = x + self.mesh(y.transpose(1, 2).reshape(x.shape), wp)
            x = x + self.mesh(self.norm(x), wf)
        return self.norm(x)

    def logits(self, rows):
        return torch.matmul(rows, self.E.t().contiguous())


def _unit(state):
    mask = (1 << 64) - 1
    state = (state + 0x9E3779B97F4A7C15) & mask
    z = state
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
    z ^= z >> 31
    return state, np.float32((z >> 40) / 16777216.0)


def _choose(logits, temperature, states):
    """The next token of each row of float64 logits: the first maximum, or one draw from the softmax by a scan in
    32 bits."""
    rows = logits.to(torch.float32).cpu().numpy()
    if temperature == 0.0:
        return rows.argmax(-1)
    chosen = []
    for i, row in enumerate(rows):
        p = np.exp((row - row.max()) / np.float32(temperature)).astype(np.float32)
        states[i], u = _unit(states[i])
        left = u * np.cumsum(p, dtype=np.float32)[-1]
        token = len(p) - 1
        for t, value in enumerate(p):
            left = np.float32(left - value)
            if left < 0:
                token = t
                break
        chosen.append(token)
    return np.array(chosen)


def _exact_generate(model, case, inputs, seed, steps):
    """The sequences after `steps` new tokens, and the logits that chose the last of them."""
    device = model.flat.device
    tokens = torch.from_numpy(inputs.astype(np.int64)).to(device)
    states = [int(seed) + b for b in range(len(inputs))]
    cache, done, logits = [], 0, None
    for _ in range(steps):
        length = tokens.shape[1]
        if length <= case["context"]:
            rows = model.forward(tokens[:, done:], cache, done)
            done = length
        else:
            rows = model.forward(tokens[:, length - case["context"]:])
        logits = model.logits(rows[:, -1])
        new = torch.from_numpy(_choose(logits, case["temperature"], states)).to(device)
        tokens = torch.cat([tokens, new[:, None]], 1)
    return {"tokens": None, "logits": logits}


def exact(case, seed):
    device = "cuda"
    inputs, targets = _tokens(case, seed)
    flat = torch.from_numpy(_parameters(case, seed).astype(np.float64)).to(device)
    call, B, S = case["call"], case["batch"], case["tokens"]
    if call in ("train", "gradient"):
        flat.requires_grad_(True)
        model = _Exact(case, flat)
        logits = model.logits(model.forward(torch.from_numpy(inputs.astype(np.int64)).to(device))).view(B * S, -1)
        wanted = targets.reshape(-1).astype(np.int64)
        keep = torch.from_numpy(np.flatnonzero(wanted != G.IGNORE_TARGET)).to(device)
        wanted = torch.from_numpy(wanted).to(device)[keep]
        loss = torch.nn.functional.cross_entropy(logits[keep], wanted)
        loss.backward()
        if call == "gradient":
            return {"loss": float(loss.detach()), "gradient": flat.grad}
        w = flat.detach()
        step = flat.grad / (flat.grad.abs() + ADAM_EPS)  # the first step's corrected moments are g and g^2
        return {"loss": float(loss.detach()), "parameters": w - LEARNING_RATE * (step + WEIGHT_DECAY * w)}
    with torch.no_grad():
        model = _Exact(case, flat)
        if call == "logits":
            rows = model.forward(torch.from_numpy(inputs.astype(np.int64)).to(device))
            return {"logits": model.logits(rows[:, -1] if case["last_only"] else rows).view(-1, case["vocab"])}
        steps = {"generate": case["steps"], "prefill": 1, "decode": case["steps"] + 1}[call]
        return _exact_generate(model, case, inputs, seed, steps)
