"""The work a serving program gives the KDA operators, as measurable cases.

Every case is one call of a public wrapper (``sgl_glm53_ascend_ops.ops``) on
inputs that are already on the GPU, as an attention layer makes it: one decode
step, one speculative-verify step, one prefill of a request or of a batch.
Sizes are those of this repository's measured configurations, latency rows and
tests, and generic ones between them. A pass returns the output tensor and the
state pool (which the call updates in place), plus the per-step checkpoints
where the call writes them.

A case's plain values:

* ``op``: ``"recurrent"`` (``kda_varlen_recurrent`` / its prepared-gate form),
  ``"chunk"`` (``kda_varlen_chunk`` / its prepared-gate form) or ``"heads4"``
  (``prepared_recurrent``: fp32 inputs with a multiplicative decay, four heads
  a call);
* ``gates``: ``"raw"`` (bf16 ``a``, ``b``; in-kernel norms), ``"log"`` (fp32
  log decay and beta) or ``"decay"`` (``heads4``);
* ``requests`` of ``low`` to ``high`` tokens each, the lengths drawn with
  ``lens_seed`` (part of the case: every seed of the inputs has them alike);
* ``heads``, ``dim`` (K = V), ``slots`` of the state pool, ``fp32`` (q, k, v in
  fp32 instead of bf16), ``index64`` (int64 metadata), ``prefill``,
  ``checkpoints`` (per-step states written), ``track`` (a prefix of each
  request tracked into a slot of its own), ``harsh`` (faster log decays),
  ``zero`` (requests start from a zero state).
"""

import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "01-glm53-ascend_amd"))

from sgl_glm53_ascend_ops.ops import (  # noqa: E402
    kda_prepared_varlen_chunk,
    kda_prepared_varlen_recurrent,
    kda_varlen_chunk,
    kda_varlen_recurrent,
    prepared_recurrent,
)

DEV = "cuda"
LOWER_BOUND = -5.0


def _case(op, gates, heads, requests, low, high, **more):
    case = dict(op=op, gates=gates, heads=heads, requests=requests, low=low, high=high, lens_seed=0, dim=128,
                slots=requests + 1, fp32=False, index64=False, prefill=False, checkpoints=False, track=False,
                harsh=False, zero=False)
    case.update(more)
    if case["track"]:
        case["slots"] = max(case["slots"], 2 * requests + 1)
    return case


def listed():
    return [
        # One request's next token on a 16-head shard: the smallest call, where latency counts.
        dict(_case("recurrent", "raw", 16, 1, 1, 1), name="decode_1"),
        # A small serving batch (an odd count) on a 32-head shard, with the int64 metadata that index
        # arithmetic in torch gives.
        dict(_case("recurrent", "raw", 32, 37, 1, 1, index64=True), name="decode_37"),
        # The headline decode step: 256 sequences, 32 heads, a permuted half of a 512-slot pool.
        dict(_case("recurrent", "log", 32, 256, 1, 1, slots=512), name="decode_256"),
        # Speculative verify: four draft tokens per request, every step's state kept.
        dict(_case("recurrent", "raw", 32, 16, 4, 4, checkpoints=True), name="verify_16x4"),
        # Multi-step decode of a large batch from a 2048-slot pool.
        dict(_case("recurrent", "log", 16, 1024, 4, 4, slots=2048, harsh=True), name="steps_1024x4"),
        # The fp32 reference configuration: two short sequences, K = V = 64.
        dict(_case("recurrent", "log", 4, 2, 37, 63, dim=64, fp32=True, zero=True), name="fp32_2x64"),
        # Short prompts prefilled together (below the chunked form's 128 tokens a request).
        dict(_case("recurrent", "raw", 32, 16, 20, 120, prefill=True, lens_seed=1), name="prefill_short_16"),
        # One prompt of the reference's latency rows on an 8-head shard, with its prefix tracked.
        dict(_case("recurrent", "raw", 8, 1, 1024, 1024, prefill=True, track=True), name="prefill_1k_h8"),
        # A long prompt on few heads.
        dict(_case("chunk", "raw", 4, 1, 16384, 16384, prefill=True), name="prefill_16k_h4"),
        # The headline chunked prefill: 8192 tokens, 32 heads, zero initial state.
        dict(_case("chunk", "log", 32, 1, 8192, 8192, zero=True, slots=3), name="prefill_8k_h32"),
        # A varlen prefill batch: 16 sequences of 1 to 4096 tokens from a 64-slot pool.
        dict(_case("chunk", "log", 32, 16, 1, 4096, slots=64, lens_seed=4), name="prefill_16_varlen"),
        # Long context with a harsh decay.
        dict(_case("chunk", "log", 16, 1, 65536, 65536, zero=True, harsh=True, slots=3), name="prefill_64k_h16"),
    ]


def _log(rng, low, high):
    """A whole number between the two, spread over its logarithm."""
    return max(low, min(high, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "short", "prompt", "batch", "batch", "heads4"])
    more = dict(lens_seed=rng.randrange(1 << 20), index64=rng.random() < 0.3)
    heads = rng.choice([4, 8, 16, 32, 64])
    if kind == "decode":  # one token each, up to the headline step's states
        n = _log(rng, 1, 8192 // heads if heads > 16 else 512)
        return _case("recurrent", rng.choice(["raw", "log"]), heads, n, 1, 1, slots=n + 1 + rng.randrange(n + 1), **more)
    if kind == "verify":  # two to eight tokens each, the steps' states kept or not
        n = _log(rng, 1, 4096 // heads)
        steps = rng.randint(2, 8)
        return _case("recurrent", rng.choice(["raw", "log"]), heads, n, steps, steps,
                     checkpoints=n * heads <= 1024 and rng.random() < 0.6, **more)
    if kind == "short":  # prompts below 128 tokens
        n = _log(rng, 1, 1024 // heads)
        low = rng.randint(1, 60)
        return _case("recurrent", "raw", heads, n, low, rng.randint(low, 127), prefill=True, track=rng.random() < 0.3, **more)
    if kind == "prompt":  # one prompt, up to the headline prefill's tokens x heads
        t = _log(rng, 129, 8192 * 32 // heads if heads > 8 else 32768)
        op, gates = rng.choice([("recurrent", "raw"), ("chunk", "raw"), ("chunk", "log")])
        return _case(op, gates, heads, 1, t, t, prefill=True, harsh=gates == "log" and rng.random() < 0.3,
                     track=rng.random() < 0.3, **more)
    if kind == "batch":  # several prompts at once
        n = rng.randint(2, 64)
        high = _log(rng, 64, min(4096, 32768 * 32 // (heads * n)))
        return _case("chunk", rng.choice(["raw", "log"]), heads, n, rng.randint(1, high), high, prefill=True,
                     track=rng.random() < 0.3, **more)
    n = _log(rng, 1, 64)  # heads4: decode or a few steps of four heads, fp32
    steps = rng.randint(1, 4)
    return _case("heads4", "decay", 4, n, steps, steps, fp32=rng.random() < 0.5, **more)


def _lengths(case):
    rng = random.Random(case["lens_seed"])
    return [rng.randint(case["low"], case["high"]) for _ in range(case["requests"])]


def _tracked(case):
    """Tracked length of each request: anywhere from 0 to its end, chunk boundaries among them."""
    rng = random.Random(case["lens_seed"] + 1)
    return [rng.choice([rng.randint(0, n), n // 64 * 64, n]) for n in _lengths(case)]


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    lens = _lengths(case)
    T, N, H, D = sum(lens), case["requests"], case["heads"], case["dim"]
    index = torch.int64 if case["index64"] else torch.int32
    dtype = torch.float32 if case["fp32"] else torch.bfloat16

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=DEV)

    def unit(x):
        return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)

    # the pool [slots, H, K, V] with K contiguous; slot 0 is the padding row, the requests sit on
    # shuffled slots, tracked prefixes on slots of their own
    pool = (randn(case["slots"], H, D, D) * 0.05).transpose(-1, -2)
    order = (torch.randperm(case["slots"] - 1, generator=gen, device=DEV) + 1).to(index)
    indices = order[:N].contiguous()
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).to(index)
    state = dict(case=case, pool=pool, indices=indices, cu=cu, scale=D ** -0.5)
    if case["zero"]:
        pool[indices.long()] = 0.0
    if case["gates"] == "raw":  # a layer's bf16 projections and its gate parameters
        for name in ("q", "k", "v", "a"):
            state[name] = (randn(1, T, H, D) * 0.2).bfloat16()
        state["b"] = randn(1, T, H).bfloat16()
        state["A_log"] = randn(H) * 0.1
        state["dt_bias"] = randn(H * D) * 0.1
    else:  # prepared gates: normalized q and k, log decay, beta
        qk = torch.float32 if case["gates"] == "decay" else dtype
        state["q"], state["k"] = unit(randn(1, T, H, D)).to(qk), unit(randn(1, T, H, D)).to(qk)
        state["v"] = randn(1, T, H, D).to(dtype)
        x = randn(1, T, H, D)
        state["g"] = torch.nn.functional.logsigmoid(x * 2 - 2 if case["harsh"] else x)
        state["beta"] = torch.sigmoid(randn(1, T, H))
    if case["gates"] == "decay":  # the scale is folded into q, the caller owns the output
        state["q"] = state["q"] * state["scale"]
        state["g"] = state["g"].exp()
        state["out"] = torch.zeros_like(state["v"])
    if case["checkpoints"]:
        state["steps"] = torch.zeros(N, case["high"], H, D, D, device=DEV).transpose(-1, -2)
    if case["track"]:
        state["track"] = dict(track_state_indices=order[N:2 * N].contiguous(),
                              track_state_lens=torch.tensor(_tracked(case), device=DEV).to(index))
    return state


def run(state):
    case, pool = state["case"], state["pool"]
    if case["gates"] == "decay":
        prepared_recurrent(state["q"], state["k"], state["v"], state["g"], state["beta"], state["out"], pool,
                           state["indices"], state["cu"])
        return {"out": state["out"], "state": pool}
    more = dict(initial_state_source=pool, initial_state_indices=state["indices"], cu_seqlens=state["cu"],
                scale=state["scale"], **state.get("track", {}))
    if case["checkpoints"]:
        more["intermediate_state"] = state["steps"]
    if case["gates"] == "raw":
        call = kda_varlen_chunk if case["op"] == "chunk" else kda_varlen_recurrent
        out = call(A_log=state["A_log"], a=state["a"], dt_bias=state["dt_bias"], q=state["q"], k=state["k"],
                   v=state["v"], b=state["b"], lower_bound=LOWER_BOUND, prefill=case["prefill"], **more)
    else:
        call = kda_prepared_varlen_chunk if case["op"] == "chunk" else kda_prepared_varlen_recurrent
        out = call(state["q"], state["k"], state["v"], state["g"], state["beta"], **more)
    result = {"out": out, "state": pool}
    if case["checkpoints"]:
        result["steps"] = state["steps"]
    return result


def work(case):
    lens = _lengths(case)
    T, N, H, D = sum(lens), case["requests"], case["heads"], case["dim"]
    x = 4 if case["fp32"] else 2
    qk = 4 if case["gates"] == "decay" else x
    token = 2 * D * qk + 2 * D * x  # q, k; v, out
    token += 2 * D + 2 if case["gates"] == "raw" else 4 * D + 4  # a, b; g, beta
    states = N * (1 if case["checkpoints"] else 2)  # read; written back unless the steps are kept
    states += T if case["checkpoints"] else 0
    states += sum(1 for n in _tracked(case)) if case["track"] else 0
    size = T * H * token + states * H * D * D * 4 + (8 if case["index64"] else 4) * (2 * N + 1)
    size += H * (D + 1) * 4 if case["gates"] == "raw" else 0
    # the recurrence: decay, prediction, update and readout of every state element; the chunked form's
    # products over 64-token chunks (every [64, 64] and [64, 128] tile dense) where prompts are long
    chunked = case["op"] == "chunk" or (case["prefill"] and T >= 128 * N)
    flops = T * H * (2 * (5 * 64 * D + 3 * D * D) if chunked else 7 * D * D)
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # Measured against exact(): bf16 outputs carry their own rounding (1.7e-3 in the 2-norm), as any
    # correct implementation's do; fp32 results of the token loop sit near 1e-7, and the prepared fp32
    # cases return nothing else.
    if case["fp32"]:
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 7e-3, "max": 0.1}


def exact(case, seed):
    """The recurrence in 64 bits, token by token, over all requests at once."""
    state = prepare(case, seed)
    lens = _lengths(case)
    N, H, D = case["requests"], case["heads"], case["dim"]
    f = torch.float64
    pool = state["pool"].to(f)
    steps = state["steps"].to(f) if case["checkpoints"] else None
    out = torch.zeros(state["v"].shape, dtype=f, device=DEV)
    S = pool[state["indices"].long()].contiguous()  # [N, H, K, V]
    starts = torch.tensor([sum(lens[:n]) for n in range(N)], device=DEV)
    size = torch.tensor(lens, device=DEV)
    track = {}
    if case["track"]:
        for n, (slot, r) in enumerate(zip(state["track"]["track_state_indices"].tolist(), _tracked(case))):
            track.setdefault(r, []).append((n, slot))

    def tokens(name, rows):
        return state[name][0, rows].to(f)

    def unit(x):
        return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)

    def save(t):
        for n, slot in track.get(t, ()):
            pool[slot] = S[n]

    def block(t0, t1):
        """Tokens t0 .. t1 of every request, [N, t, H, ...], those past a request's end without effect."""
        t = torch.arange(t0, t1, device=DEV)
        live = t[None, :] < size[:, None]
        rows = starts[:, None] + torch.minimum(t[None, :], size[:, None] - 1)
        q, k, v = tokens("q", rows), tokens("k", rows), tokens("v", rows)
        if case["gates"] == "raw":
            q, k = unit(q) * state["scale"], unit(k)
            x = tokens("a", rows) + state["dt_bias"].to(f).view(H, D)
            g = LOWER_BOUND * torch.sigmoid(state["A_log"].to(f).exp()[:, None] * x)
            beta = torch.sigmoid(tokens("b", rows))
        else:
            g, beta = tokens("g", rows), tokens("beta", rows)
            if case["gates"] == "decay":
                g = g.log()
            else:
                q = q * state["scale"]
        mask = live[:, :, None]
        return rows, live, q, k, v, torch.where(mask[..., None], g, 0.0).exp(), torch.where(mask, beta, 0.0)

    longest, width = max(lens), max(1, min(512, (1 << 26) // (N * H * D)))
    save(0)
    for t0 in range(0, longest, width):
        t1 = min(longest, t0 + width)
        rows, live, q, k, v, dec, beta = block(t0, t1)
        o = torch.empty_like(v)
        q, k, dec, v, beta = q[..., None], k[..., None], dec[..., None], v[..., None, :], beta[..., None, None]
        for i in range(t1 - t0):
            S.mul_(dec[:, i])
            d = (v[:, i] - (S * k[:, i]).sum(-2, keepdim=True)) * beta[:, i]
            S.addcmul_(k[:, i], d)
            o[:, i] = (S * q[:, i]).sum(-2)
            if steps is not None:
                steps[:, t0 + i] = S
            if track:
                save(t0 + i + 1)
        out[0, rows[live]] = o[live]
    if case["checkpoints"]:
        return {"out": out, "state": pool, "steps": steps}
    pool[state["indices"].long()] = S
    return {"out": out, "state": pool}
