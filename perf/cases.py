"""What this library's speed is judged on: the calls a reinforcement-learning program makes into
it, from one decoded token to a training step's logit gradient, and the tensor products, sorts and
softmaxes around them.

Each case is a dict of plain values with an "op":

  sample      nt_hip_rl_sample: the masked inverse-CDF draw and its log-probability per row, as a
              serving loop calls the C entry, with buffers that it keeps between steps.
  gumbel      nt_hip_rl_sample_gumbel: the reference's own sampler (one u64 of the caller's ChaCha
              stream per logit), from the same loop.
  score       nt_hip_rl_score: log-probabilities of given tokens, with the entropy and, beside a
              reference model, its log-probabilities and the exact KL.
  ppo         one PPO update's work on the logits through the host mirror (noetic_rl): the scoring
              pass with its statistics, the clipped loss, and the gradient of loss + KL - entropy.
  readout     the decode step from the hidden states (noetic_rl.readout_sample_logp): the head's
              product and the draw in one call, the weight packed once.
  matmul      noetic_ops.matmul at the default f32 precision, or at MatmulPrecision.HALF.
  sort        noetic_ops.sort_desc along the last axis (what top-k and top-p draws are made of).
  softmax     noetic_ops.log_softmax over the last axis, the reference's op sequence.

Sizes are the benchmark configurations' own (vocabularies of 32000, 50304, 128256 and 151936), the
reference's matmul shapes, and generic ones around them.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "noetic-tensor_amd"))

import noetic_ops as ops  # noqa: E402
import noetic_rl as nr  # noqa: E402

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16, "u8": torch.uint8, "i32": torch.int32,
          "f64": torch.float64}
_CODE = {"f32": nr.NT_F32, "bf16": nr.NT_BF16, "f16": nr.NT_F16}
_ESIZE = {"f32": 4, "bf16": 2, "f16": 2}
# mask: none; u8 keep-masks of grammar-like runs (30% kept) or of independent bytes (90% kept), a
# row each; the runs as the reference's additive f32 0/-inf mask, a row each ("f32") or one row that
# every position shares ("f32_shared")
_MASK_BYTES = {"none": 0, "runs": 1, "bernoulli": 1, "f32": 4, "f32_shared": 0}
_PPO = {"clip": 0.2, "kl": 0.05, "entropy": -0.01}


def listed():
    return [
        # one sequence decoded alone: the latency of a single row
        {"name": "sample_one", "op": "sample", "rows": 1, "vocab": 32000, "dtype": "f32", "mask": "none", "tau": 0.8,
         "entropy": False},
        # constrained decode of 256 sequences under a grammar: the headline configuration
        {"name": "sample_grammar", "op": "sample", "rows": 256, "vocab": 128256, "dtype": "bf16", "mask": "runs",
         "tau": 0.7, "entropy": False},
        # the same decode through the reference's own Gumbel-max sampler
        {"name": "gumbel_grammar", "op": "gumbel", "rows": 256, "vocab": 128256, "dtype": "bf16", "mask": "runs",
         "tau": 0.7},
        # an unconstrained decode step of 64 sequences, Gumbel-max
        {"name": "gumbel_decode", "op": "gumbel", "rows": 64, "vocab": 32000, "dtype": "f32", "mask": "none",
         "tau": 0.8},
        # log-probabilities of one decode step's tokens for a serving batch: few rows, a large
        # vocabulary, one additive mask for all
        {"name": "score_decode", "op": "score", "rows": 64, "vocab": 128256, "dtype": "bf16", "mask": "f32_shared",
         "tau": 0.7, "ref": False},
        # rollout scoring at a large vocabulary in f32, a random keep-mask, no temperature
        {"name": "score_rollout", "op": "score", "rows": 4096, "vocab": 151936, "dtype": "f32", "mask": "bernoulli",
         "tau": 1.0, "ref": False},
        # a PPO update: forward with reference KL and entropy, loss, gradient on the bf16 logits
        {"name": "ppo_step", "op": "ppo", "seeds": 4, "batch": 8, "tokens": 256, "vocab": 50304, "dtype": "bf16",
         "mask": "none", "tau": 1.0},
        # the decode step from the hidden states at the headline's rows and vocabulary
        {"name": "readout_decode", "op": "readout", "rows": 256, "dim": 4096, "vocab": 128256, "mask": "runs",
         "tau": 0.7},
        # a projection at the default precision (the reference's f32 arithmetic to the bit)
        {"name": "matmul_f32", "op": "matmul", "m": 2048, "k": 2048, "n": 2048, "precision": "f32", "tb": False},
        # a large projection at half precision
        {"name": "matmul_half", "op": "matmul", "m": 4096, "k": 4096, "n": 4096, "precision": "half", "tb": False},
        # the descending order of a batch's vocabulary rows for a top-p draw
        {"name": "sort_vocab", "op": "sort", "rows": 64, "vocab": 128256},
        # full log-probabilities of a batch of positions, kept as a tensor
        {"name": "softmax_rows", "op": "softmax", "rows": 256, "vocab": 50304},
    ]


def _size(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, lo=1000, hi=152000):
    """A vocabulary: one of the configurations', one padded to 8 or 64, or any whole number."""
    v = rng.choice([32000, 50304, 128256, 151936]) if rng.random() < 0.3 else _size(rng, lo, hi)
    pad = rng.choice([1, 8, 64])
    return min(max(v, lo), hi) // pad * pad


def draw(rng):
    op = rng.choice(["sample", "sample", "gumbel", "score", "ppo", "readout", "matmul", "matmul", "sort", "softmax"])
    V = _vocab(rng)
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    tau = rng.choice([0.6, 0.7, 0.8, 1.0])
    if op in ("sample", "gumbel"):
        rows = _size(rng, 1, 256)
        if op == "sample" and rng.random() < 0.2:
            tau = 0.0  # greedy
        c = {"op": op, "rows": rows, "vocab": V, "dtype": dtype, "tau": tau,
             "mask": rng.choice(["none", "none", "runs", "bernoulli", "f32", "f32_shared"])}
        if op == "sample":
            c["entropy"] = rng.random() < 0.3
        return c
    if op == "score":
        rows = _size(rng, 1, min(16384, 400_000_000 // V))
        return {"op": op, "rows": rows, "vocab": V, "dtype": dtype, "tau": tau, "ref": rng.random() < 0.5,
                "mask": rng.choice(["none", "bernoulli", "f32_shared"])}
    if op == "ppo":
        seeds, batch = rng.choice([1, 2, 4]), rng.choice([1, 4, 7, 8])
        tokens = _size(rng, 1, max(1, min(1024, 300_000_000 // (V * seeds * batch))))
        return {"op": op, "seeds": seeds, "batch": batch, "tokens": tokens, "vocab": V, "dtype": dtype, "tau": tau,
                "mask": rng.choice(["none", "none", "f32_shared"])}
    if op == "readout":
        return {"op": op, "rows": _size(rng, 1, 256), "dim": 16 * _size(rng, 16, 256), "vocab": min(V, 128256),
                "tau": tau, "mask": rng.choice(["none", "runs"])}
    if op == "matmul":
        half = rng.random() < 0.5
        m, k, n = (_size(rng, 64, 4096 if half else 2048) for _ in range(3))
        if rng.random() < 0.5:
            m, k, n = (v // 64 * 64 for v in (m, k, n))
        return {"op": op, "m": m, "k": k, "n": n, "precision": "half" if half else "f32", "tb": rng.random() < 0.4}
    if op == "sort":
        return {"op": op, "rows": _size(rng, 1, 64), "vocab": _vocab(rng, 100, 128256)}
    return {"op": "softmax", "rows": _size(rng, 8, 256), "vocab": _vocab(rng, 100, 50304)}


# ------------------------------------------------------------------------------------- inputs

class _Held:
    """A torch allocation as the buffer behind a noetic_rl.Tensor."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


def _given(t, dtype):
    """A contiguous torch tensor as the library's device tensor, in place."""
    return nr.Tensor(tuple(t.shape), dtype, _Held(t))


class _Export:
    def __init__(self, t):
        self.owner = t
        kind = {"f32": "<f4", "bf16": "<i2", "f16": "<f2", "i32": "<i4", "u8": "|u1"}[t.dtype]
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": kind, "data": (t.ptr, False), "version": 2}


def _taken(t):
    """The library's device tensor as a torch tensor over the same memory (kept alive by it)."""
    x = torch.as_tensor(_Export(t), device="cuda")
    return x.view(torch.bfloat16) if t.dtype == "bf16" else x


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(shape, dtype, g, std):
    t = torch.empty(shape, dtype=_TORCH[dtype], device="cuda")
    return t.normal_(0.0, std, generator=g)


def _keep_runs(rows, V, g):
    """Contiguous kept runs (mean 96) between excluded gaps (mean 224), at least one token kept."""
    pairs = int(V / 320 * 2) + 64
    u = torch.rand((rows, pairs, 2), device="cuda", generator=g)
    mean = torch.tensor([224.0, 96.0], device="cuda")
    length = (-torch.log1p(-u) * mean).floor().long() + 1
    edge = length.reshape(rows, -1).cumsum(1) - torch.randint(0, 320, (rows, 1), device="cuda", generator=g)
    flips = torch.zeros((rows, V + 1), dtype=torch.int32, device="cuda")
    flips.scatter_add_(1, edge.clamp(0, V), torch.ones_like(edge, dtype=torch.int32))
    keep = (flips[:, :V].cumsum(1) % 2 == 1)
    return _at_least_one(keep, g)


def _at_least_one(keep, g):
    one = torch.randint(0, keep.shape[1], (keep.shape[0], 1), device="cuda", generator=g)
    return keep.scatter_(1, one, True)


def _mask(case, rows, g, tokens=None):
    """(mask tensor or None, the boolean it keeps) for `rows` logits rows; `tokens` stay allowed."""
    kind, V = case["mask"], case["vocab"]
    if kind == "none":
        return None, None
    shared = kind == "f32_shared"
    n = 1 if shared else rows
    keep = (_keep_runs(n, V, g) if kind in ("runs", "f32", "f32_shared")
            else _at_least_one(torch.rand((n, V), device="cuda", generator=g) < 0.9, g))
    if tokens is not None:
        keep[0 if shared else torch.arange(rows, device="cuda"), tokens.reshape(-1).long()] = True
    if kind in ("f32", "f32_shared"):
        return torch.where(keep, 0.0, -math.inf).contiguous(), keep
    return keep.to(torch.uint8), keep


def _logit_rows(case, rows, g):
    """What the sampler, the scorer and the losses are given: logits of a language model's spread."""
    return _normal((rows, case["vocab"]), case["dtype"], g, 2.0 if case["op"] in ("sample", "gumbel") else 1.5)


def _clear_uniforms(x, case, g):
    """One uniform per row, each moved to the middle of its token's step of the row's CDF (of its most
    probable token's where that step is under 4e-6): where a uniform meets an edge, the last bit of a
    sum decides the token, and no comparison says anything."""
    u = torch.rand(x["logits"].shape[0], dtype=torch.float64, device="cuda", generator=g)
    for s in _chunks(u.shape[0], case["vocab"]):
        p = torch.softmax(_tempered64(x, case, s), 1)
        cdf = p.cumsum(1)
        at = torch.searchsorted(cdf, u[s, None] * cdf[:, -1:], right=True).clamp(max=cdf.shape[1] - 1)
        at = torch.where(p.gather(1, at) < 4e-6, p.argmax(1, keepdim=True), at)
        below = torch.where(at > 0, cdf.gather(1, (at - 1).clamp(min=0)), 0.0)
        u[s] = (0.5 * (below + cdf.gather(1, at)) / cdf[:, -1:])[:, 0]
    return u


def _tokens(rows, V, g):
    return torch.randint(0, V, (rows,), device="cuda", generator=g, dtype=torch.int32)


def _reference(policy, g):
    """A frozen reference model's logits: the policy's plus N(0, 0.1^2)."""
    ref = torch.empty_like(policy).normal_(0.0, 0.1, generator=g)
    return ref.add_(policy)


def _inputs(case, seed):
    """Every input as torch tensors, a function of the case and the seed alone."""
    g, op = _generator(seed), case["op"]
    if op in ("sample", "gumbel"):
        rows = case["rows"]
        x = {"logits": _logit_rows(case, rows, g)}
        x["mask"], x["keep"] = _mask(case, rows, g)
        x["uniforms"] = _clear_uniforms(x, case, g) if op == "sample" else None
    elif op in ("score", "ppo"):
        rows = case["rows"] if op == "score" else case["seeds"] * case["batch"] * case["tokens"]
        x = {"logits": _logit_rows(case, rows, g), "tokens": _tokens(rows, case["vocab"], g)}
        x["ref"] = _reference(x["logits"], g) if op == "ppo" or case["ref"] else None
        x["mask"], x["keep"] = _mask(case, rows, g, x["tokens"])
        if op == "ppo":
            x["advantages"] = torch.randn((case["seeds"], case["batch"]), device="cuda", generator=g)
            now = torch.cat([_log_softmax64(x, case, s)[0].gather(1, x["tokens"][s].long()[:, None])[:, 0]
                             for s in _chunks(rows, case["vocab"])])
            # the policy has moved since the rollout; a ratio at the clip's edge, where rounding decides
            # whether the token has a gradient, is put back to 1
            moved = 0.1 * torch.randn(rows, device="cuda", generator=g, dtype=torch.float64)
            edge = torch.tensor([1.0 - _PPO["clip"], 1.0 + _PPO["clip"]], device="cuda", dtype=torch.float64).log()
            moved[(moved[:, None] - edge).abs().amin(1) < 1e-3] = 0.0
            x["old_logp"] = (now - moved).float().reshape(case["seeds"], case["batch"], case["tokens"])
    elif op == "readout":
        rows, d, V = case["rows"], case["dim"], case["vocab"]
        x = {"hidden": _normal((rows, d), "bf16", g, 1.0), "weight": _normal((d, V), "bf16", g, 2.0 / math.sqrt(d))}
        x["mask"], x["keep"] = _mask(case, rows, g)
        x["uniforms"] = _clear_uniforms(dict(x, logits=x["hidden"].double() @ x["weight"].double()), case, g)
    elif op == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        x = {"a": _normal((m, k), "f32", g, 1.0), "b": _normal((n, k) if case["tb"] else (k, n), "f32", g, 1.0)}
    else:
        x = {"logits": _normal((case["rows"], case["vocab"]), "f32", g, 2.0)}
    return x


# ------------------------------------------------------------------------------------- cases

def _ptr(t):
    return None if t is None else t.data_ptr()


def _mask_args(case, x):
    """(mask_kind, mask pointer, mask_ld) of the C entries."""
    if x["mask"] is None:
        return nr.NT_MASK_NONE, None, 0
    kind = nr.NT_MASK_U8 if x["mask"].dtype == torch.uint8 else nr.NT_MASK_F32
    return kind, x["mask"].data_ptr(), 0 if case["mask"] == "f32_shared" else case["vocab"]


def prepare(case, seed):
    nr.claim(0)
    x, op = _inputs(case, seed), case["op"]
    x.pop("keep", None)
    s = {"case": case, "x": x}
    row = lambda kind: torch.empty(case["rows"], dtype=_TORCH[kind], device="cuda")  # noqa: E731
    if op in ("sample", "gumbel", "score"):
        rows, V, every_row = case["rows"], case["vocab"], nr.NtMaskRows(0, 0, 0, 0)
        mk, mptr, mld = _mask_args(case, x)
        head = (_CODE[case["dtype"]], mk, rows, V, V, mptr, mld, case["tau"])
        s["status"] = row("u8")
    if op == "sample":
        out = {"ids": row("i32"), "logp": row("f32")}
        if case["entropy"]:
            out["entropy"] = row("f32")
        s["out"] = out
        s["args"] = nr.NtRlSampleArgs(_ptr(x["logits"]), *head, _ptr(x["uniforms"]), _ptr(out["ids"]),
                                      _ptr(out["logp"]), _ptr(out.get("entropy")), _ptr(s["status"]), every_row)
        s["entry"] = nr.lib().nt_hip_rl_sample
    elif op == "gumbel":
        stream = nr.Rng(seed, "sampling")
        block, word = stream.word_pos()
        s["out"] = {"ids": row("i32")}
        s["args"] = nr.NtRlGumbelArgs(_ptr(x["logits"]), *head, stream.key(), block, word, 0, _ptr(s["out"]["ids"]),
                                      _ptr(s["status"]), every_row)
        s["entry"] = nr.lib().nt_hip_rl_sample_gumbel
    elif op == "score":
        out = {"logp": row("f32"), "entropy": row("f32")}
        if case["ref"]:
            out.update(ref_logp=row("f32"), kl=row("f32"))
        s["out"] = out
        s["args"] = nr.NtRlScoreArgs(_ptr(x["logits"]), _ptr(x["ref"]), *head, _ptr(x["tokens"]), _ptr(out["logp"]),
                                     _ptr(out.get("ref_logp")), _ptr(out.get("kl")), _ptr(out["entropy"]),
                                     _ptr(s["status"]), None, None, None, None, every_row)
        s["entry"] = nr.lib().nt_hip_rl_score
    elif op == "ppo":
        shape = (case["seeds"], case["batch"], case["tokens"])
        give = lambda t: _given(t.reshape(shape + (case["vocab"],)), case["dtype"])  # noqa: E731
        mask = None if x["mask"] is None else _given(x["mask"].reshape(1, 1, 1, case["vocab"]), "f32")
        s["policy"] = nr.Tempered(give(x["logits"]), case["tau"], mask)
        s["reference"] = nr.Tempered(give(x["ref"]), case["tau"], mask)
        s["tokens"] = _given(x["tokens"].reshape(shape), "i32")
        s["old"], s["advantages"] = _given(x["old_logp"], "f32"), _given(x["advantages"], "f32")
    elif op == "readout":
        s["weight"] = nr.PackedReadout(_given(x.pop("weight"), "bf16"))
        s["hidden"] = _given(x["hidden"], "bf16")
        s["mask"] = None if x["mask"] is None else _given(x["mask"], "u8")
        s["uniforms"] = _given(x["uniforms"], "f64")
    elif op == "matmul":
        s["a"], s["b"] = _given(x["a"], "f32"), _given(x["b"], "f32")
        s["al"], s["bl"] = ops.Layout.contiguous(s["a"].shape), ops.Layout.contiguous(s["b"].shape)
        if case["tb"]:
            s["bl"] = s["bl"].swapped(0, 1)
    else:
        s["rows"] = _given(x["logits"], "f32")
    nr.sync()
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op in ("sample", "gumbel", "score"):
        nr._check(s["entry"](C.byref(s["args"])), op)
        return s["out"]
    if op == "ppo":
        return _ppo_step(s)
    if op == "readout":
        with nr.matmul_precision_scope(nr.MatmulPrecision.HALF):
            ids, logp = nr.readout_sample_logp(s["hidden"], s["weight"], case["tau"], s["mask"], None,
                                               uniforms=s["uniforms"])
        return {"ids": _taken(ids), "logp": _taken(logp)}
    if op == "matmul":
        y, _ = ops.matmul(s["a"], s["al"], s["b"], s["bl"], nr.MatmulPrecision(case["precision"]))
        return _taken(y)
    if op == "sort":
        values, positions = ops.sort_desc(s["rows"], (case["rows"], case["vocab"], 1))
        return {"values": _taken(values), "positions": _taken(positions)}
    return _taken(ops.log_softmax(ops.DTensor(s["rows"]), 1).storage)


def _ppo_step(s):
    """loss = clipped_policy_loss + 0.05 KL - 0.01 H, each the mean over a seed's tokens; returns the
    loss per seed, the scoring pass's outputs and the gradient on the policy's logits."""
    shape, mean = s["tokens"].shape, nr.TokenReduction.TOKEN_MEAN
    clip = nr.Clip.symmetric(_PPO["clip"])
    logp, ref_logp, kl, entropy, stats = nr.score_with_stats(s["policy"], s["reference"], s["tokens"])
    loss = nr.clipped_policy_loss(logp, s["old"], s["advantages"], None, clip, mean)
    g_logp = nr.clipped_policy_loss_backward(logp, s["old"], s["advantages"], None, clip, mean)
    g_kl = nr.reduce_tokens_backward(None, shape, mean, scale=_PPO["kl"])
    g_entropy = nr.reduce_tokens_backward(None, shape, mean, scale=_PPO["entropy"])
    grad = nr.score_grad(s["policy"], s["reference"], s["tokens"], stats, kl=kl, entropy=entropy, g_logp=g_logp,
                         g_kl=g_kl, g_entropy=g_entropy)
    return {"loss": _taken(loss), "logp": _taken(logp), "ref_logp": _taken(ref_logp), "kl": _taken(kl),
            "entropy": _taken(entropy), "grad": _taken(grad)}


def work(case):
    """Each input read once and each output written once; a keep-mask's excluded logits count too.
    The Gumbel sampler's draws are generated, not read."""
    op, e = case["op"], _ESIZE.get(case.get("dtype"), 4)
    if op in ("sample", "gumbel", "score"):
        rows, V = case["rows"], case["vocab"]
        b = rows * V * (e + _MASK_BYTES[case["mask"]]) + (4 * V if case["mask"] == "f32_shared" else 0)
        if op == "score":
            return {"bytes": b + (rows * V * e if case["ref"] else 0) + rows * (21 if case["ref"] else 13), "flops": 0}
        return {"bytes": b + rows * (17 if op == "sample" else 5), "flops": 0}
    if op == "ppo":  # both logits once for the forward, once for the gradient, the gradient written
        rows = case["seeds"] * case["batch"] * case["tokens"]
        return {"bytes": rows * case["vocab"] * e * 5 + rows * 24, "flops": 0}
    if op == "readout":
        rows, d, V = case["rows"], case["dim"], case["vocab"]
        mask = rows * V if case["mask"] == "runs" else 0
        return {"bytes": 2 * d * V + 2 * rows * d + mask + 17 * rows, "flops": 2 * rows * d * V}
    if op == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    n = case["rows"] * case["vocab"]
    return {"bytes": 12 * n if op == "sort" else 8 * n, "flops": 0}


def tolerance(case):
    """Two correct orders of the same sums, measured over these ranges: log-probabilities and entropies
    within 5e-7 (rel) and 3e-6 (max), an exact KL of 0.005 nats, a difference of two logarithms, within
    1e-5 and 5e-5; about four times that here."""
    op = case["op"]
    if op in ("gumbel", "sort"):
        return "exact"  # token ids; values in their order
    if op == "sample":
        return {"rel": 2e-6, "max": 1e-5, "differ": 0.005}
    if op == "readout":  # the logits' own f32 sums over the hidden dimension
        return {"rel": 4e-6, "max": 4e-5, "differ": 0.005}
    if op == "ppo" and case["dtype"] != "f32":  # the gradient comes in the logits' 16-bit type
        return {"rel": 4e-4, "max": 1e-2}
    if op == "ppo" or case.get("ref"):
        return {"rel": 4e-5, "max": 2e-4}
    if op == "matmul":  # f32 sums; the operands of a half product are rounded alike everywhere
        return {"rel": 2e-6, "max": 2e-5}
    return {"rel": 2e-6, "max": 2e-5}


# ------------------------------------------------------------------------------------- 64 bits

def _chunks(rows, V):
    step = max(1, 100_000_000 // V)
    return [slice(i, min(rows, i + step)) for i in range(0, rows, step)]


def _tempered64(x, case, s, name="logits"):
    z = x[name][s].double()
    if case["tau"] not in (0.0, 1.0):
        z /= case["tau"]
    if x.get("keep") is not None:
        z.masked_fill_(~(x["keep"] if x["keep"].shape[0] == 1 else x["keep"][s]), -math.inf)
    return z


def _log_softmax64(x, case, s):
    out = [torch.log_softmax(_tempered64(x, case, s), 1)]
    if x.get("ref") is not None:
        out.append(torch.log_softmax(_tempered64(x, case, s, "ref"), 1))
    return out


def _drawn64(z, u, greedy):
    """The inverse-CDF draw's log-probability (the maximum's if greedy) and the row's entropy."""
    lp = torch.log_softmax(z, 1)
    if greedy:
        return lp.max(1)[0], _entropy64(lp)
    cdf = lp.exp().cumsum(1)
    at = torch.searchsorted(cdf, u[:, None] * cdf[:, -1:], right=True).clamp(max=z.shape[1] - 1)
    return lp.gather(1, at)[:, 0], _entropy64(lp)


def _entropy64(lp):
    return -torch.where(lp == -math.inf, 0.0, lp.exp() * lp).sum(1)


def _kl64(lp, lr):
    return torch.where(lp == -math.inf, 0.0, lp.exp() * (lp - lr)).sum(1)


def _scored64(x, case):
    cols = {"logp": [], "ref_logp": [], "kl": [], "entropy": []}
    for s in _chunks(x["logits"].shape[0], case["vocab"]):
        at = x["tokens"][s].long()[:, None]
        lp, *lr = _log_softmax64(x, case, s)
        cols["logp"].append(lp.gather(1, at)[:, 0])
        cols["entropy"].append(_entropy64(lp))
        if lr:
            cols["ref_logp"].append(lr[0].gather(1, at)[:, 0])
            cols["kl"].append(_kl64(lp, lr[0]))
    return {k: torch.cat(v) for k, v in cols.items() if v}


def _ppo64(x, case):
    S, B, T = case["seeds"], case["batch"], case["tokens"]
    out = _scored64(x, case)
    adv = x["advantages"].double()[:, :, None].expand(S, B, T)
    ratio = (out["logp"].reshape(S, B, T) - x["old_logp"].double()).exp()
    lo, hi = 1.0 - _PPO["clip"], 1.0 + _PPO["clip"]
    plain, clipped = -ratio * adv, -ratio.clamp(lo, hi) * adv
    per = torch.maximum(plain, clipped)
    inside = (plain >= clipped) | ((ratio >= lo) & (ratio <= hi))
    share = 1.0 / (B * T)
    g_logp = (torch.where(inside, -ratio * adv, 0.0) * share).reshape(-1)
    grad = torch.empty(x["logits"].shape, dtype=torch.float64, device="cuda")
    for s in _chunks(grad.shape[0], case["vocab"]):
        lp, lr = _log_softmax64(x, case, s)
        p = lp.exp()
        lp, lr = lp.masked_fill(p == 0, 0.0), lr.masked_fill(p == 0, 0.0)
        at = x["tokens"][s].long()[:, None]
        g = -g_logp[s][:, None] * p
        g += _PPO["kl"] * share * p * (lp - lr - out["kl"][s][:, None])
        g -= _PPO["entropy"] * share * p * (lp + out["entropy"][s][:, None])
        g.scatter_add_(1, at, g_logp[s][:, None])
        grad[s] = g / case["tau"]
    out = {k: v.reshape(S, B, T) for k, v in out.items()}
    return dict(out, loss=per.mean((1, 2)), grad=grad.reshape(S, B, T, -1))


def exact(case, seed):
    """run()'s outputs in 64 bits from torch alone; None in the place of tokens and positions."""
    op = case["op"]
    if op == "gumbel":
        return None
    x = _inputs(case, seed)
    if op == "sample":
        got = [_drawn64(_tempered64(x, case, s), x["uniforms"][s], case["tau"] == 0.0)
               for s in _chunks(case["rows"], case["vocab"])]
        logp, entropy = (torch.cat(v) for v in zip(*got))
        return {"ids": None, "logp": logp, **({"entropy": entropy} if case["entropy"] else {})}
    if op == "score":
        return _scored64(x, case)
    if op == "ppo":
        return _ppo64(x, case)
    if op == "readout":
        z = dict(x, logits=x["hidden"].double() @ x["weight"].double())
        return {"ids": None, "logp": _drawn64(_tempered64(z, case, slice(None)), x["uniforms"], False)[0]}
    if op == "matmul":
        a, b = x["a"], x["b"].t() if case["tb"] else x["b"]
        if case["precision"] == "half":  # the product of the operands rounded to bf16
            a, b = a.bfloat16(), b.bfloat16()
        return a.double() @ b.double().contiguous()
    if op == "sort":
        return {"values": torch.sort(x["logits"].double(), dim=1, descending=True)[0], "positions": None}
    return torch.log_softmax(x["logits"].double(), 1)
