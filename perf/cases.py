"""Performance cases of the stick-breaking attention operators.

A case is one call that a model makes once per layer: the forward alone (prefill, evaluation) or the
forward and the backward (a training step) of `sb_attn` / `sb_attn_varlen`, or of their fused forms that
return `o + rem * v`.  Its fields:

  op, fused        which public operator
  backward         forward + backward through autograd, or the forward under no_grad
  grad_rem         the loss also reaches `rem`, the second output (two-output operators only)
  dtype            element type of q, k, v and of the incoming gradient
  heads, head_dim
  layout           "heads": stored [.., heads, tokens, head_dim]; "tokens": stored token-major, as a
                   projection leaves them, and handed over as a head-major view
  attend_current   a token may attend to itself
  batch, tokens    fixed length: `batch` sequences of `tokens` tokens.  Packed documents: batch is 1,
                   `tokens` tokens in all
  min_len, max_len, spread, first_len, doc_seed
                   packed documents: lengths drawn from [min_len, max_len], evenly ("even") or evenly over
                   the logarithm ("log"), behind one document of first_len tokens (0: none); the last one is
                   cut to fill
  zero_start, cu64 packed documents: cu_seqlens with a leading zero; as int64
"""
import math
import os
import random
import sys

import torch

_PACKAGE = os.path.abspath("stickbreaking-attention_amd")   # of the tree that is the working folder
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from stickbreaking_attention import sb_attn, sb_attn_fused, sb_attn_varlen, sb_attn_varlen_fused  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _case(name, op, heads, head_dim, tokens, **more):
    c = dict(name=name, op=op, fused=False, backward=True, grad_rem=False, dtype="bf16", heads=heads, head_dim=head_dim,
             layout="heads", attend_current=False, batch=1, tokens=tokens, min_len=0, max_len=0, spread="even",
             first_len=0, doc_seed=0, zero_start=False, cu64=False)
    assert set(more) <= set(c), more
    c.update(more)
    return c


def listed():
    return [
        # The smallest training step: one short sequence, a handful of workgroups; launches and host work count.
        _case("attn 1x4x512 d64", "attn", 4, 64, 512),
        # Prefill / evaluation of a few short prompts of very unequal lengths (one token up to a few hundred).
        _case("varlen prefill 596 d128", "varlen", 4, 128, 596, backward=False, spread="log", min_len=1, max_len=331,
              doc_seed=2024),
        # A small packed micro-batch in half precision, odd lengths, through the fused operator.
        _case("varlen f16 fused 3001 d64", "varlen", 12, 64, 3001, fused=True, dtype="f16", attend_current=True,
              spread="log", min_len=40, max_len=1500, doc_seed=7, zero_start=True, cu64=True),
        # The fixed-length operator on an ordinary batch; the loss reaches both outputs, as `o + rem * v` outside does.
        _case("attn 4x16x2048 d64", "attn", 16, 64, 2048, batch=4, grad_rem=True),
        # Packed pretraining documents, the repository's headline workload: 16 K tokens of 512 ... 4096.
        _case("varlen 16k h32 d128", "varlen", 32, 128, 16384, min_len=512, max_len=4096, doc_seed=1340),
        # Many short documents: next to no arithmetic per byte, tile edges everywhere.
        _case("varlen 16k short docs d64", "varlen", 32, 64, 16384, spread="log", min_len=16, max_len=256, doc_seed=1341,
              zero_start=True),
        # Long-context evaluation: one document of 32 K tokens among long ones, forward alone.
        _case("varlen 64k fwd d128", "varlen", 32, 128, 65536, backward=False, spread="log", min_len=1024,
              max_len=16384, first_len=32768, doc_seed=1342),
        # Four full-length sequences of 4096 tokens, 12 heads, token-major storage (what a projection
        # writes), through the fused operator: the upstream benchmark's shape.
        _case("varlen 4x4096 h12 d128 fused", "varlen", 12, 128, 16384, fused=True, layout="tokens", min_len=4096,
              max_len=4096),
        # Wide heads.
        _case("varlen 16k h16 d256", "varlen", 16, 256, 16384, min_len=512, max_len=4096, doc_seed=1340),
        # A head_dim between the kernels' own, an odd token count, ragged documents.
        _case("varlen 7001 h16 d96", "varlen", 16, 96, 7001, layout="tokens", grad_rem=True, spread="log", min_len=100,
              max_len=3000, doc_seed=96),
        # float32 callers (computed on 16-bit matrix cores), fixed length that is no multiple of a tile.
        _case("attn f32 2x8x1500 d64", "attn", 8, 64, 1500, batch=2, dtype="f32"),
        # Narrow heads, forward alone.
        _case("attn fwd 4x16x2048 d32", "attn", 16, 32, 2048, batch=4, backward=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    c = _case("", "varlen" if rng.random() < 0.65 else "attn", _log_int(rng, 2, 32),
              rng.choice((32, 64, 64, 80, 96, 128, 128, 128, 160, 256)), 0)
    del c["name"]
    c["dtype"] = rng.choice(("bf16", "bf16", "bf16", "bf16", "f16", "f32"))
    c["backward"] = rng.random() < 0.7
    c["fused"] = rng.random() < 0.35
    c["grad_rem"] = c["backward"] and not c["fused"] and rng.random() < 0.5
    c["layout"] = rng.choice(("heads", "tokens"))
    c["attend_current"] = rng.random() < 0.25
    if c["op"] == "attn":
        c["batch"] = _log_int(rng, 1, 8)
        c["tokens"] = _log_int(rng, 64, 8192)
    else:
        c["tokens"] = _log_int(rng, 256, 65536)
        c["min_len"] = _log_int(rng, 1, max(1, c["tokens"] // 4))
        c["max_len"] = _log_int(rng, max(16, c["min_len"]), c["tokens"])
        c["spread"] = rng.choice(("even", "log"))
        c["doc_seed"] = rng.randrange(1 << 20)
        c["zero_start"] = rng.random() < 0.5
        c["cu64"] = rng.random() < 0.3
    while _cost(c) > 0.3 * _cost(_largest()):
        c["tokens"] = c["tokens"] // 2 + 1
        c["max_len"] = min(c["max_len"], c["tokens"])
        c["min_len"] = min(c["min_len"], c["max_len"])
    return c


def _largest():
    return next(c for c in listed() if c["first_len"])


def _cost(c):
    """Grows about as the time of a large case does: score pairs times the width of the head, narrow heads and the
    backward being dearer than their arithmetic."""
    return _pairs(c) * (c["head_dim"] + 64) * (5 if c["backward"] else 1)


def _lengths(c):
    """Lengths of the documents (of the batch entries) in order."""
    if c["op"] == "attn":
        return [c["tokens"]] * c["batch"]
    rng = random.Random(c["doc_seed"])
    lo, hi, left, out = c["min_len"], c["max_len"], c["tokens"], []
    while left > 0:
        if c["first_len"] and not out:
            n = c["first_len"]
        elif c["spread"] == "log":
            n = _log_int(rng, lo, hi)
        else:
            n = rng.randint(lo, hi)
        out.append(min(n, left))
        left -= out[-1]
    return out


def _pairs(c):
    return c["heads"] * sum(n * n for n in _lengths(c)) / 2.0


def prepare(case, seed):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(seed)
    H, T, d, B = case["heads"], case["tokens"], case["head_dim"], case["batch"]
    fixed, dtype = case["op"] == "attn", _DTYPES[case["dtype"]]

    def values(*tail):
        """A head-major tensor of N(0, 1) values in the case's storage order."""
        if case["layout"] == "tokens":
            shape = ((B, T, H) if fixed else (T, H)) + tail
            t = torch.randn(shape, generator=gen, device=dev).to(dtype)
            return t.transpose(1, 2) if fixed else t.transpose(0, 1)
        shape = ((B, H, T) if fixed else (H, T)) + tail
        return torch.randn(shape, generator=gen, device=dev).to(dtype)

    s = {"case": case, "q": values(d), "k": values(d), "v": values(d)}
    if case["backward"]:
        for n in "qkv":
            s[n].requires_grad_()
        s["do"] = values(d)
        if case["grad_rem"]:
            s["drem"] = values()
    if not fixed:
        lengths = _lengths(case)
        ends, at = [0] if case["zero_start"] else [], 0
        for n in lengths:
            at += n
            ends.append(at)
        s["cu"] = torch.tensor(ends, dtype=torch.int64 if case["cu64"] else torch.int32, device=dev)
        s["longest"] = max(lengths)
    return s


def _forward(s):
    c = s["case"]
    if c["op"] == "attn":
        return (sb_attn_fused if c["fused"] else sb_attn)(s["q"], s["k"], s["v"], attend_current=c["attend_current"])
    return (sb_attn_varlen_fused if c["fused"] else sb_attn_varlen)(
        s["q"], s["k"], s["v"], s["cu"], s["longest"], zero_start=c["zero_start"], attend_current=c["attend_current"])


def run(state):
    c = state["case"]
    if not c["backward"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    inputs = (state["q"], state["k"], state["v"])
    if c["fused"]:
        return (out,) + torch.autograd.grad(out, inputs, state["do"])
    o, rem = out
    if c["grad_rem"]:
        return (o, rem) + torch.autograd.grad((o, rem), inputs, (state["do"], state["drem"]))
    return (o, rem) + torch.autograd.grad(o, inputs, state["do"])


def work(case):
    """Bytes: q, k, v (and the incoming gradients) read once, o and rem (and dq, dk, dv) written once.  Operations: two
    matrix products forward and five backward per causal pair."""
    size = {"bf16": 2, "f16": 2, "f32": 4}[case["dtype"]]
    rows = case["heads"] * case["batch"] * case["tokens"]
    mats = 4 + (4 if case["backward"] else 0)
    per_row = (0 if case["fused"] else 1) + (1 if case["grad_rem"] else 0)
    return {"bytes": rows * size * (mats * case["head_dim"] + per_row),
            "flops": (14.0 if case["backward"] else 4.0) * case["head_dim"] * _pairs(case)}


def tolerance(case):
    # 16-bit matrix operands and outputs, sums in fp32; float32 callers are computed with bf16 operands
    return {"rel": 2e-3 if case["dtype"] == "f16" else 1e-2}
