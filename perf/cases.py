"""Performance cases of the DSA forward and its stages on one GPU.

Each case calls one public entry point the way a program does: the whole
forward (dsa_attention), the lightning indexer (lightning_indexer), the
per-row select (topk_threshold) and the precomputed-threshold attention.
Every call is a forward pass over whole sequences: the library has no
backward and no single-token entry point.  Inputs are N(0,1) with indexer
weights N(0,1)/sqrt(HI), the distributions the repository's benchmark and
tests use.

  listed()            the fixed cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs on the GPU
  run(state)          one pass, returning its outputs
  work(case)          compulsory bytes and arithmetic of one pass
  tolerance(case)     how far another correct implementation may differ
  exact(case, seed)   the result in float64 from plain torch
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dsa-cpu-topk_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import dsa_attention as D  # noqa: E402
import lightning_indexer as LI  # noqa: E402
import topk_threshold as TK  # noqa: E402

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}


def _forward(name, B, T, k, HI, DI, HQ, DH, dtype, entry):
    return {"name": name, "kind": "forward", "entry": entry, "B": B, "T": T, "k": k, "HI": HI,
            "DI": DI, "HQ": HQ, "DH": DH, "dtype": dtype}


def listed():
    return [
        # The smallest call: one short sequence, where launch latency counts.
        _forward("forward_short", 1, 128, 8, 4, 32, 4, 32, "fp32", "fused"),
        # The benchmark's headline forward, a batch of short sequences.
        _forward("forward_batch", 16, 512, 32, 4, 32, 4, 32, "fp32", "fused"),
        # Sequences at the one-kernel forward's length limit, 16-bit, the head
        # sizes of the long-row configuration.
        _forward("forward_2k_bf16", 4, 2048, 128, 8, 64, 8, 64, "bf16", "fused"),
        # Long rows in fp32: scores spill to HBM, three stages.
        _forward("forward_4k_fp32", 4, 4096, 256, 8, 64, 8, 64, "fp32", "split"),
        # The largest call: one long sequence at DeepSeek-V3.2-like sizes.
        _forward("forward_16k_bf16", 1, 16384, 2048, 64, 128, 16, 128, "bf16", "split"),
        # A prompt of no particular length (odd T, k not a power of two), fp16.
        _forward("forward_ragged_fp16", 2, 3001, 300, 16, 128, 16, 128, "fp16", "any"),
        # The indexer alone, the full square with its -inf upper triangle, as
        # callers who rank or inspect scores take it; odd length.
        {"name": "indexer_fp32", "kind": "indexer", "B": 4, "T": 2047, "HI": 8, "DI": 64,
         "dtype": "fp32"},
        # The indexer from hidden states: projections and scores in one call.
        {"name": "indexer_hidden_bf16", "kind": "hidden", "B": 1, "T": 4096, "D": 2048, "HI": 64,
         "DI": 128, "dtype": "bf16"},
        # The indexer on e4m3 activations with their quantisation scales.
        {"name": "indexer_fp8", "kind": "fp8", "B": 1, "T": 8192, "HI": 64, "DI": 128},
        # The select alone on plain score rows (the top-K extension's table).
        {"name": "topk_rows", "kind": "topk", "rows": 64 * 2048, "n": 2048, "k": 128},
        # The selection as a boolean mask of causal scores.
        {"name": "topk_mask", "kind": "mask", "B": 2, "T": 4096, "k": 256},
        # The attention alone with a threshold made elsewhere (the offload path).
        {"name": "attention_1k_fp32", "kind": "attention", "B": 8, "T": 1024, "k": 64, "HQ": 8,
         "DH": 64, "dtype": "fp32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pow2(rng, lo, hi):
    return 1 << rng.randint(lo.bit_length() - 1, hi.bit_length() - 1)


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "indexer", "hidden", "fp8", "topk", "mask",
                       "attention", "attention"])
    dtype = rng.choice(["fp32", "bf16", "fp16"])
    if kind == "topk":
        n = _log(rng, 64, 32768)
        rows = max(1, min(_log(rng, 64, 131072), (1 << 28) // n))
        return {"kind": kind, "rows": rows, "n": n, "k": max(1, min(n, _log(rng, 8, max(9, n // 4))))}
    if kind == "mask":
        T = _log(rng, 128, 8192)
        return {"kind": kind, "B": max(1, min(rng.randint(1, 8), (1 << 27) // (T * T))), "T": T,
                "k": max(1, min(T, _log(rng, 8, max(9, T // 4))))}
    if kind in ("indexer", "hidden", "fp8"):
        HI, DI = _pow2(rng, 4, 64), rng.choice([64, 128] if kind == "fp8" else [32, 64, 128])
        T = _log(rng, 128, 8192 if kind == "fp8" or dtype != "fp32" else 4096)
        per = T * T * HI * DI
        B = max(1, min(rng.randint(1, 8), int(1.2e11 if dtype == "fp32" and kind != "fp8" else 1e12) // per))
        c = {"kind": kind, "B": B, "T": T, "HI": HI, "DI": DI}
        if kind != "fp8":
            c["dtype"] = dtype
        if kind == "hidden":
            c["D"] = rng.choice([512, 1024, 2048])
        return c
    HQ, DH = _pow2(rng, 4, 16), rng.choice([32, 64, 128])
    T = _log(rng, 64, 4096 if dtype == "fp32" else 8192)
    k = max(1, min(T, _log(rng, 8, max(9, T // 8))))
    if kind == "attention":
        T = 1 << max(6, min(12, T.bit_length()))  # this entry point takes powers of two
        per = T * T * HQ * DH
        return {"kind": kind, "B": max(1, min(rng.randint(1, 16), int(2e11) // per)), "T": T,
                "k": min(k, T), "HQ": HQ, "DH": DH, "dtype": dtype}
    HI, DI = _pow2(rng, 4, 32), rng.choice([32, 64, 128])
    per = T * T * (HI * DI + 2 * HQ * DH)
    B = max(1, min(rng.randint(1, 32), int(1.5e11 if dtype == "fp32" else 1e12) // per))
    return {"kind": "forward", "entry": "any", "B": B, "T": T, "k": k, "HI": HI, "DI": DI, "HQ": HQ,
            "DH": DH, "dtype": dtype}


# ---------------------------------------------------------------------------
def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * scale).to(dtype)


def _causal(T):
    return torch.ones(T, T, device="cuda", dtype=torch.bool).tril()


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    c, kind = case, case["kind"]
    if kind == "topk":
        return dict(case=c, scores=_randn(g, c["rows"], c["n"]))
    B, T = c["B"], c["T"]
    if kind == "mask":
        return dict(case=c, scores=_randn(g, B, T, T).masked_fill_(~_causal(T), float("-inf")))
    if kind == "fp8":
        HI, DI = c["HI"], c["DI"]
        q, k = _randn(g, B, T, HI, DI), _randn(g, B, T, DI)
        qs, ks = q.abs().amax(-1) / 448.0, k.abs().amax(-1) / 448.0
        return dict(case=c, q=(q / qs.unsqueeze(-1)).to(torch.float8_e4m3fn),
                    k=(k / ks.unsqueeze(-1)).to(torch.float8_e4m3fn),
                    w=_randn(g, B, T, HI, scale=HI ** -0.5), qs=qs, ks=ks)
    dt = DTYPES[c["dtype"]]
    if kind == "attention":
        scores = _randn(g, B, T, T).masked_fill_(~_causal(T), float("-inf"))
        thr = torch.cat([s.topk(c["k"], dim=-1).values[..., -1:] for s in scores.split(1)])
        sh = (B, T, c["HQ"], c["DH"])
        return dict(case=c, scores=scores, thr=thr,
                    att=tuple(_randn(g, *sh, dtype=dt) for _ in range(3)))
    HI, DI = c["HI"], c["DI"]
    if kind == "hidden":
        Dm = c["D"]
        return dict(case=c, h=_randn(g, B, T, Dm, dtype=dt),
                    W=tuple(_randn(g, Dm, n, scale=Dm ** -0.5 * s, dtype=dt)
                            for n, s in ((HI * DI, 1.0), (DI, 1.0), (HI, HI ** -0.5))))
    idx = (_randn(g, B, T, HI, DI, dtype=dt), _randn(g, B, T, DI, dtype=dt),
           _randn(g, B, T, HI, scale=HI ** -0.5, dtype=dt))
    if kind == "indexer":
        return dict(case=c, idx=idx)
    sh = (B, T, c["HQ"], c["DH"])
    return dict(case=c, idx=idx, att=tuple(_randn(g, *sh, dtype=dt) for _ in range(3)))


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "forward":
        fn = {"fused": D.dsa_attention_triton, "split": D.dsa_attention_split_triton,
              "any": D.dsa_forward_hip}[c["entry"]]
        return fn(*state["idx"], *state["att"], c["k"])
    if kind == "indexer":
        return LI.indexer_scores_triton(*state["idx"])
    if kind == "hidden":
        return LI.indexer_triton(state["h"], *state["W"], c["HI"], c["DI"])
    if kind == "fp8":
        return LI.indexer_scores_hip(state["q"], state["k"], state["w"], q_scale=state["qs"],
                                     k_scale=state["ks"])
    if kind == "topk":
        return TK.topk_threshold(state["scores"], c["k"])
    if kind == "mask":
        return LI.topk_mask(state["scores"], c["k"])
    return D.sparse_attention_with_threshold_triton(state["scores"], state["thr"], *state["att"])


def _selected(T, k):
    k = min(k, T)
    return k * (k + 1) // 2 + (T - k) * k


def work(case):
    c, kind = case, case["kind"]
    if kind == "topk":
        return {"bytes": 4.0 * c["rows"] * (c["n"] + 1), "flops": 1.0 * c["rows"] * c["n"]}
    B, T = c["B"], c["T"]
    pairs = B * T * (T + 1) // 2
    if kind == "mask":
        return {"bytes": 5.0 * B * T * T, "flops": 1.0 * B * T * T}
    es = BYTES[c["dtype"]] if "dtype" in c else 1
    if kind == "attention":
        e = B * T * c["HQ"] * c["DH"]
        return {"bytes": 4.0 * pairs + 4.0 * B * T + 3.0 * es * e + 4.0 * e,
                "flops": 4.0 * B * _selected(T, c["k"]) * c["HQ"] * c["DH"]}
    HI, DI = c["HI"], c["DI"]
    fl = pairs * HI * (2.0 * DI + 2)
    if kind == "hidden":
        n = HI * DI + DI + HI
        return {"bytes": es * (B * T * c["D"] + c["D"] * n) + 4.0 * B * T * T,
                "flops": fl + 2.0 * B * T * c["D"] * n}
    if kind == "fp8":
        return {"bytes": B * T * (HI * DI + DI + 8.0 * HI + 4) + 4.0 * B * T * T, "flops": fl}
    idx_bytes = es * B * T * (HI * DI + DI + HI)
    if kind == "indexer":
        return {"bytes": idx_bytes + 4.0 * B * T * T, "flops": fl}
    e = B * T * c["HQ"] * c["DH"]
    return {"bytes": idx_bytes + 3.0 * es * e + 4.0 * e,
            "flops": fl + 4.0 * B * _selected(T, c["k"]) * c["HQ"] * c["DH"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("topk", "mask"):
        return "exact"
    if kind == "forward":
        # A score rounded differently can move a row's k-th largest across a
        # near-tie, and that row then swaps one of its k keys: up to a few
        # rows in 10^4, each off by about 1.4/sqrt(k) of its norm.
        return {"rel": 5e-3 if case["dtype"] == "fp32" else 1e-2, "max": 0.99}
    if kind == "fp8":
        # the fp8 instruction's sum of 128 products keeps 13-14 bits
        return {"rel": 1e-4, "max": 4e-3}
    if kind == "hidden" and case["dtype"] != "fp32":
        return {"rel": 1e-2, "max": 0.2}  # q, k and w are rounded to 16 bits between the steps
    if kind == "attention" and case["dtype"] != "fp32":
        return {"rel": 1e-2, "max": 0.2}  # probabilities in 16 bits on some paths
    return {"rel": 1e-5, "max": 2e-4}


def _rows_in(T, B, HI):
    """Query rows per chunk so that a float64 [B, HI, rows, T] block is at most 1 GiB."""
    return max(1, min(T, (1 << 27) // (B * HI * T)))


def _indexer64(q, k, w):
    """q [B,T,HI,DI], k [B,T,DI], w [B,T,HI] -> causal scores, float64."""
    q, k, w = q.double(), k.double(), w.double()
    B, T, HI, DI = q.shape
    kt = k.transpose(1, 2).contiguous()
    out = torch.empty(B, T, T, device=q.device, dtype=torch.float64)
    step = _rows_in(T, 1, HI)
    for b in range(B):
        for t in range(0, T, step):
            n = min(step, T - t)
            dots = (q[b, t:t + n].reshape(n * HI, DI) @ kt[b]).view(n, HI, T).clamp_(min=0)
            out[b, t:t + n] = (w[b, t:t + n].unsqueeze(-1) * dots).sum(1)
    return out.masked_fill_(~_causal(T), float("-inf"))


def _attention64(scores, thr, Q, K, V):
    B, T, HQ, DH = Q.shape
    out = torch.empty(B, T, HQ, DH, device=Q.device, dtype=torch.float64)
    drop = ~((scores >= thr) & _causal(T))
    for b in range(B):
        for h in range(HQ):
            lg = (Q[b, :, h].double() @ K[b, :, h].double().t().contiguous()) / math.sqrt(DH)
            out[b, :, h] = torch.softmax(lg.masked_fill_(drop[b], float("-inf")), -1) @ V[b, :, h].double()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "mask":
        return None  # no computed numbers
    s = prepare(case, seed)
    if kind == "topk":
        return torch.cat([x.topk(case["k"], dim=-1).values[..., -1:].double()
                          for x in s["scores"].split(8192)])
    if kind == "attention":
        return _attention64(s["scores"], s["thr"], *s["att"])
    if kind == "indexer":
        return _indexer64(*s["idx"])
    if kind == "fp8":
        return _indexer64(s["q"].double() * s["qs"].double().unsqueeze(-1),
                          s["k"].double() * s["ks"].double().unsqueeze(-1), s["w"])
    if kind == "hidden":
        h = s["h"].double()
        q, k, w = (h @ W.double() for W in s["W"])
        return _indexer64(q.view(*q.shape[:2], case["HI"], case["DI"]), k, w)
    if case["T"] > 1024:
        # Over long rows some row's k-th and next score nearly always lie
        # closer than fp32 resolves, and which key that row takes has no
        # right answer: the stages' own cases carry the comparison.
        return None
    scores = _indexer64(*s["idx"])
    thr = scores.topk(min(case["k"], case["T"]), dim=-1).values[..., -1:]
    return _attention64(scores, thr, *s["att"])
