"""The attention calls this package is measured on.

A case is one call of the public API as a program makes it: a training step of
one attention layer (forward and backward), an inference forward (prefill), or
a decoding step. ``listed()`` gives fixed cases, ``draw(rng)`` one more of the
same kinds and ranges; ``prepare`` / ``run`` / ``exact`` make its inputs, run
it and compute it in 64 bits with plain PyTorch.

Case fields:
  kind    "train": O and the gradients of q, k, v; "forward": O without autograd
  B, Hq, Hkv, Nq, Nkv, D   batch, query and key/value heads, lengths, head size
  causal, dtype            mask; "float16" or "bfloat16"
  layout  how the program holds the tensors:
          "heads"  contiguous [B, H, N, D]
          "tokens" the projections' [B, N, H, D], passed as transposed views
          "cache"  decoding against a key/value cache allocated for ``cache``
                   tokens ([B, Hkv, cache, D]) and filled up to Nkv
  spread  factor on the iid N(0, 1) inputs
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parent.parent / "triton-flash-attention_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from triton_flash_attention import scaled_dot_product_attention  # noqa: E402

# The benchmark's causal B2 H32 N8192 D128 shape without its mask is the
# largest listed case; a drawn one has at most its multiply-adds and elements.
_MOST_PAIRS_D = 2 * 32 * 8192 * 8192 * 128
_MOST_ELEMENTS = 2 * 32 * 8192 * 128


def _case(kind, B, Hq, Hkv, Nq, Nkv, D, causal, dtype, layout="heads", cache=0, spread=1.0,
          **name):
    return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, Nq=Nq, Nkv=Nkv, D=D, causal=causal, dtype=dtype,
                layout=layout, cache=cache, spread=spread, **name)


def listed():
    return [
        # The smallest call: one short ragged sequence, few heads, inference
        # (the benchmark's first configuration). Launch latency counts.
        _case("forward", 1, 4, 4, 257, 257, 64, False, "float16", name="small_forward"),
        # Short training sequences, the first row of the README's sweep.
        _case("train", 4, 16, 16, 512, 512, 64, True, "float16", name="short_train"),
        # The headline: causal training at N 4096.
        _case("train", 4, 16, 16, 4096, 4096, 64, True, "float16", name="train_d64"),
        # Grouped heads and a ragged length just past a tile.
        _case("train", 2, 16, 4, 2049, 2049, 64, True, "float16", name="train_gqa_ragged"),
        # The largest: bidirectional training at N 8192, head size 128.
        _case("train", 2, 32, 32, 8192, 8192, 128, False, "float16", spread=0.5,
              name="train_d128_long"),
        # One long causal sequence with small grouped heads.
        _case("train", 1, 8, 2, 16381, 16381, 32, True, "float16", name="train_d32_long"),
        # A decoder layer's training step as a model runs it: bf16, grouped
        # heads, the projections' [B, N, H, D] tensors passed as views.
        _case("train", 2, 32, 8, 2048, 2048, 128, True, "bfloat16", layout="tokens",
              name="train_decoder_layer"),
        # An encoder layer's training step: bidirectional, a head size between
        # the kernels' widths, an odd length, projection views.
        _case("train", 4, 16, 16, 1025, 1025, 80, False, "bfloat16", layout="tokens",
              name="train_encoder_d80"),
        # Cross-attention training: few queries read many keys.
        _case("train", 2, 16, 16, 64, 16384, 64, False, "float16", name="train_cross"),
        # Prefill of one prompt of odd length: inference, projection views.
        _case("forward", 1, 32, 8, 3001, 3001, 128, True, "bfloat16", layout="tokens",
              name="prefill"),
        # Decoding, one new token per sequence against full keys and values.
        _case("forward", 8, 32, 8, 1, 8192, 128, False, "float16", name="decode_batch"),
        # Decoding against a partly filled cache, a small batch.
        _case("forward", 2, 32, 8, 1, 3001, 128, False, "bfloat16", layout="cache", cache=8192,
              name="decode_cache"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _odd(rng, n):
    """A length as programs have it: a multiple of 64, or any."""
    return max(64, n // 64 * 64) if rng.random() < 0.4 and n >= 64 else n


def draw(rng):
    while True:
        kind = rng.choice(["train", "train", "train", "cross", "prefill", "decode", "decode"])
        dtype = rng.choice(["float16", "bfloat16"])
        D = rng.choice([32, 64, 64, 64, 128, 128, 128, 80, 96, 40])
        Hkv = rng.choice([2, 4, 8, 16])
        group = rng.choice([1, 1, 2, 4, 8])
        Hq = min(32, Hkv * group)
        B = _log_int(rng, 1, 8)
        spread = rng.choice([0.5, 1.0])
        causal, layout, cache = rng.random() < 0.6, rng.choice(["heads", "tokens"]), 0
        if kind == "decode":
            Nq, Nkv = rng.choice([1, 1, 1, 2, 4, 16]), _odd(rng, _log_int(rng, 256, 32768))
            B, causal = _log_int(rng, 1, 32), False
            layout = rng.choice(["heads", "cache"])
            if layout == "cache":
                cache = -(-Nkv * rng.choice([1, 2, 4]) // 1024) * 1024
        elif kind == "cross":
            Nq, Nkv, causal = _odd(rng, _log_int(rng, 16, 1024)), _odd(rng, _log_int(rng, 64, 16384)), False
        else:
            Nq = Nkv = _odd(rng, _log_int(rng, 64, 16384))
        if (B * Hq * Nq * Nkv * D <= _MOST_PAIRS_D and B * Hq * Nq * D <= _MOST_ELEMENTS
                and B * Hkv * max(Nkv, cache) * D <= _MOST_ELEMENTS):
            return _case("train" if kind in ("train", "cross") else "forward", B, Hq, Hkv, Nq, Nkv,
                         D, causal, dtype, layout=layout, cache=cache, spread=spread)


def _shapes(case):
    B, D = case["B"], case["D"]
    nkv = case["cache"] or case["Nkv"]
    q, kv = (B, case["Hq"], case["Nq"], D), (B, case["Hkv"], nkv, D)
    if case["layout"] == "tokens":
        q, kv = ((s[0], s[2], s[1], s[3]) for s in (q, kv))
    return q, kv


def _tensors(case, seed):
    """q, k, v and (training) dO as the program holds them."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q, kv = _shapes(case)
    shapes = [q, kv, kv] + ([q] if case["kind"] == "train" else [])
    dtype = getattr(torch, case["dtype"])
    return [(torch.randn(s, generator=gen, device="cuda") * case["spread"]).to(dtype) for s in shapes]


def _heads(case, t):
    """The [B, H, N, D] tensor (a view in the other layouts) the API is given."""
    if case["layout"] == "tokens":
        return t.transpose(1, 2)
    return t


def prepare(case, seed):
    tensors = _tensors(case, seed)
    if case["kind"] == "train":
        for t in tensors[:3]:
            t.requires_grad_()
    return {"case": case, "tensors": tensors}


def run(state):
    case, (q, k, v, *rest) = state["case"], state["tensors"]
    kwargs = dict(is_causal=case["causal"], enable_gqa=case["Hq"] != case["Hkv"], backend="triton")
    if case["kind"] == "forward":
        with torch.no_grad():
            q, k, v = (_heads(case, t) for t in (q, k, v))
            if case["layout"] == "cache":
                k, v = k[:, :, :case["Nkv"]], v[:, :, :case["Nkv"]]
            return {"o": scaled_dot_product_attention(q, k, v, **kwargs)}
    out = scaled_dot_product_attention(*(_heads(case, t) for t in (q, k, v)), **kwargs)
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), _heads(case, rest[0]))
    return {"o": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def _pairs(case):
    """Query-key pairs under the (top-left) causal mask of one head."""
    nq, nk = case["Nq"], case["Nkv"]
    if not case["causal"]:
        return nq * nk
    n = min(nq, nk)
    return n * (n + 1) // 2 + (nq - n) * nk


def work(case):
    q = case["B"] * case["Hq"] * case["Nq"] * case["D"]
    kv = case["B"] * case["Hkv"] * case["Nkv"] * case["D"]
    matmul = 2 * case["B"] * case["Hq"] * _pairs(case) * case["D"]
    if case["kind"] == "forward":  # q, k, v read; O written; Q K^T and P V
        return {"bytes": 2 * (2 * q + 2 * kv), "flops": 2 * matmul}
    # also dO read, dQ, dK, dV written; the backward's S, dP, dV, dK and dQ
    return {"bytes": 2 * (4 * q + 4 * kv), "flops": 7 * matmul}


def tolerance(case):
    # Rounding to 16 bits of the outputs and of the probabilities: about 3e-4
    # (fp16) and 2.5e-3 (bf16) against 64 bits, measured; four times that.
    if case["dtype"] == "float16":
        return {"rel": 2e-3, "max": 3e-2}
    return {"rel": 1.2e-2, "max": 2e-1}


def exact(case, seed):
    q, k, v, *rest = (_heads(case, t) for t in _tensors(case, seed))
    k, v = k[:, :, :case["Nkv"]], v[:, :, :case["Nkv"]]
    group, scale = case["Hq"] // case["Hkv"], case["D"] ** -0.5
    nq, nk = case["Nq"], case["Nkv"]
    train = case["kind"] == "train"
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    dq = torch.empty_like(o) if train else None
    dk = torch.zeros(k.shape, dtype=torch.float64, device=q.device) if train else None
    dv = torch.zeros_like(dk) if train else None
    # One head at a time, in blocks of queries.
    block = max(1, min(nq, (1 << 27) // nk))
    cols = torch.arange(nk, device=q.device)
    for b in range(case["B"]):
        for h in range(case["Hq"]):
            kd, vd = k[b, h // group].double(), v[b, h // group].double()
            for i in range(0, nq, block):
                qd = q[b, h, i:i + block].double()
                s = (qd @ kd.t()).mul_(scale)
                if case["causal"]:
                    rows = torch.arange(i, i + qd.shape[0], device=q.device)
                    s.masked_fill_(cols[None, :] > rows[:, None], -math.inf)
                p = torch.softmax(s, dim=-1)
                ob = p @ vd
                o[b, h, i:i + block] = ob
                if train:
                    g = rest[0][b, h, i:i + block].double()
                    dv[b, h // group] += p.t() @ g
                    ds = (g @ vd.t()).sub_((g * ob).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                    dq[b, h, i:i + block] = ds @ kd
                    dk[b, h // group] += ds.t() @ qd
    if not train:
        return {"o": o}
    grads = (_heads(case, t) for t in (dq, dk, dv))  # laid out as the leaves
    return dict(zip(("o", "dq", "dk", "dv"), (o, *grads)))
