"""GPU: the dense MFMA attention with fp32 probabilities (kernel="dense") --
tile edges, both block forms, non-finite and wide-range operands -- against
the float64 oracle and the per-query gathers."""
from __future__ import annotations

import math

import pytest
import torch

import _dsa_lib as L
from dsa_attention import sparse_attention_hip
from helpers import say
from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu

F32, BF, HF = torch.float32, torch.bfloat16, torch.float16


def case(T, HQ, D, k, dtype, B=1, seed=0):
    _, _, _, Q, K, V = O.make_inputs(B, T, 1, 1, HQ, D, D, dtype=dtype, seed0=seed)
    g = torch.Generator().manual_seed(seed + 5)
    s = torch.randn(B, T, T, generator=g)
    s = torch.where(torch.rand(B, T, T, generator=g) < 0.1, 0.0, s)
    masked = s.masked_fill(~torch.ones(T, T, dtype=torch.bool).tril(), -math.inf)
    return s, O.topk_threshold(masked, min(k, T)), Q, K, V


def bound(Q, K, V, T):
    """Elementwise bound on the difference of two fp32 evaluations: rel_bound
    of the largest |V|, which bounds the pieces' share (2^-32 of it) too."""
    return rel_bound(Q, K, T) * float(V.double().abs().max())


def rel_bound(Q, K, T):
    """Bound on what fp32 evaluation changes, relative to sum p |V| / sum p: a
    logit is off by at most 16 * 2^-24 |q||k| scale (products to 2^-22, sums)
    and exp2's argument by 2^-24 of its size (<= 64), a probability by that
    relative to itself, numerator and normaliser both; the sums over the
    keys add (T/32 + 8) * 2^-24."""
    D = Q.shape[-1]
    lg = float(Q.double().norm(dim=-1).max() * K.double().norm(dim=-1).max()) / math.sqrt(D)
    return (2 * (16 * lg + 64) + T / 32 + 8) * 2.0 ** -24


@pytest.mark.parametrize("dtype", [F32, BF, HF])
@pytest.mark.parametrize("T,HQ,D,k", [(1, 1, 64, 1), (31, 2, 128, 5), (63, 4, 64, 9), (64, 1, 128, 8),
                                      (65, 8, 64, 64), (127, 2, 64, 20), (128, 2, 128, 30),
                                      (129, 4, 64, 129), (200, 1, 128, 16), (257, 2, 64, 3),
                                      (333, 16, 128, 40), (333, 32, 64, 70)])
def test_dense_edges(dev, T, HQ, D, k, dtype):
    """Remainders of the key and query tiles, one to several tiles, every key
    selected, rows that no wave's tile holds; two key groups per block."""
    say(f"dense T={T} HQ={HQ} D={D} k={k} {dtype}")
    s, thr, Q, K, V = case(T, HQ, D, k, dtype, B=2, seed=T)
    out = sparse_attention_hip(*(x.to(dev) for x in (s, thr, Q, K, V)), kernel="dense").cpu()
    want = O.sparse_attn_threshold(s, thr, Q, K, V)
    err = float((out.double() - want).abs().max())
    assert err <= bound(Q, K, V, T), err


@pytest.mark.parametrize("dtype,HQ,D", [(F32, 16, 64), (F32, 8, 128), (BF, 16, 64), (HF, 8, 128)])
def test_dense_many_blocks(dev, dtype, HQ, D):
    """More than two blocks per compute unit: one key group per block.  All
    rows against the gathers, which the oracle tests cover."""
    T, k = 2200, 150
    B = 2 * 256 * 128 // (HQ * T) + 1
    say(f"dense many blocks B={B} T={T} HQ={HQ} D={D} {dtype}")
    g = torch.Generator(device=dev).manual_seed(3)
    s = torch.randn(B, T, T, generator=g, device=dev)
    tril = torch.ones(T, T, dtype=torch.bool, device=dev).tril()
    thr = s.masked_fill(~tril, -math.inf).topk(k, dim=-1).values[..., -1:].contiguous()
    Q, K, V = (torch.randn(B, T, HQ, D, generator=g, device=dev).to(dtype) for _ in range(3))
    a = sparse_attention_hip(s, thr, Q, K, V, kernel="dense")
    b = sparse_attention_hip(s, thr, Q, K, V, kernel="gather")
    torch.cuda.synchronize()
    assert float((a - b).abs().max()) <= 2 * bound(Q, K, V, T)


@pytest.mark.parametrize("dtype,D", [(F32, 64), (F32, 128), (BF, 64), (HF, 128)])
def test_dense_nonfinite(dev, dtype, D):
    """inf and NaN in Q, K and V, selected and not, and rows that select
    nothing: what the gathers give, NaN for NaN."""
    T, HQ, k = 400, 2, 12
    s, thr, Q, K, V = case(T, HQ, D, k, dtype, B=2, seed=9)
    thr[0, 7], thr[0, 300] = math.nan, math.inf
    for x, at, v in ((K, (0, 70, 0, 3), math.inf), (K, (0, 71, 1, 0), -math.inf),
                     (K, (0, 90, 0, 5), math.nan), (V, (0, 150, 1, 2), math.inf),
                     (V, (0, 151, 0, 9), math.nan), (Q, (0, 200, 0, 1), math.inf),
                     (Q, (0, 201, 1, 1), math.nan)):
        x[at] = v
    args = tuple(x.to(dev) for x in (s, thr, Q, K, V))
    a = sparse_attention_hip(*args, kernel="dense").cpu()
    b = sparse_attention_hip(*args, kernel="gather").cpu()
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    assert torch.equal(torch.isinf(a), torch.isinf(b))
    fin = torch.isfinite(b)
    clean = [torch.nan_to_num(x.float(), 0, 0, 0) for x in (Q, K, V)]
    assert float((a - b)[fin].abs().max()) <= 2 * bound(*clean, T)
    assert bool(torch.isfinite(a[1]).all())


def _own_norm(out, s, thr, Q, K, V, T):
    """Every element within rel_bound of its own sum p |V| / sum p, plus the
    2^-19 of its row's largest output that the 16-bit pieces may cost."""
    want = O.sparse_attn_threshold(s, thr, Q, K, V)
    cap = O.sparse_attn_threshold(s, thr, Q, K, V.abs())
    lim = rel_bound(Q, K, T) * cap + 2.0 ** -19 * want.abs().amax(dim=-1, keepdim=True)
    worst = float(((out.double() - want).abs() / lim.clamp(min=1e-300)).max())
    assert worst <= 1.0, worst


@pytest.mark.parametrize("dtype,HQ,D", [(F32, 16, 64), (F32, 8, 128), (BF, 16, 64), (BF, 16, 128),
                                        (HF, 16, 64), (HF, 16, 128)])
@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("gap", [6.0, 10.0, 13.0, 16.0, 30.0])
def test_dense_sink(dev, dtype, HQ, D, groups, gap):
    """A key that every query selects at a logit far above the rest, with V = 0:
    the output is what the small probabilities carry, and has their relative
    accuracy, not the large one's; one and two key groups per block."""
    T, k, sink = 300, 90, 70
    B = 2 if groups == 2 else 2 * 256 // (HQ * ((T + 127) // 128)) + 1
    say(f"dense sink B={B} HQ={HQ} D={D} {dtype} gap={gap}")
    s, _, Q, K, V = case(T, HQ, D, k, F32, B=B, seed=int(gap))
    Q[..., 0], K[..., 0] = 4.0, 0.0
    K[:, sink] = 0.0
    K[:, sink, :, 0] = gap * math.sqrt(D) / 4.0
    V[:, sink] = 0.0
    s[:, :, sink] = 9.0
    masked = s.masked_fill(~torch.ones(T, T, dtype=torch.bool).tril(), -math.inf)
    thr = O.topk_threshold(masked, k)
    Q, K, V = (x.to(dtype) for x in (Q, K, V))
    out = sparse_attention_hip(*(x.to(dev) for x in (s, thr, Q, K, V)), kernel="dense").cpu()
    _own_norm(out, s, thr, Q, K, V, T)


@pytest.mark.parametrize("dtype,HQ,D", [(F32, 16, 64), (F32, 8, 128), (BF, 16, 64), (HF, 16, 128)])
@pytest.mark.parametrize("groups", [1, 2])
def test_dense_large_logits(dev, dtype, HQ, D, groups):
    """Logits of N(0, 64^2): the running max moves often, probabilities span
    all of fp32, and two key groups merge across that."""
    T, k = 300, 120
    B = 2 if groups == 2 else 2 * 256 // (HQ * ((T + 127) // 128)) + 1
    say(f"dense large logits B={B} HQ={HQ} D={D} {dtype}")
    s, thr, Q, K, V = case(T, HQ, D, k, F32, B=B, seed=3)
    Q, K, V = (Q * 8).to(dtype), (K * 8).to(dtype), V.to(dtype)
    out = sparse_attention_hip(*(x.to(dev) for x in (s, thr, Q, K, V)), kernel="dense").cpu()
    _own_norm(out, s, thr, Q, K, V, T)


@pytest.mark.parametrize("dtype,D", [(F32, 64), (F32, 128), (HF, 64), (HF, 128)])
def test_dense_does_ordinary_rows_itself(dev, dtype, D):
    """N(0, 1) operands leave no tile to the gathers: every 128-query tile's
    output differs from theirs in rounding."""
    T, HQ, k = 1024, 4, 200
    args = tuple(x.to(dev) for x in case(T, HQ, D, k, dtype, seed=4))
    a, b = (sparse_attention_hip(*args, kernel=n).view(T // 128, -1) for n in ("dense", "gather"))
    assert bool((a != b).any(dim=1).all())


@pytest.mark.parametrize("dtype,HQ,D", [(F32, 4, 64), (F32, 16, 128), (HF, 16, 64), (HF, 4, 128),
                                        (BF, 4, 64), (BF, 16, 128)])
@pytest.mark.parametrize("B", [1, 40])
def test_dense_gathers_single_rows(dev, dtype, HQ, D, B):
    """A row the pieces cannot carry is gathered by itself, all its heads: it
    equals the gathers bit for bit, and its neighbours keep the dense sums."""
    T, k = 300, 150
    say(f"dense single rows B={B} HQ={HQ} D={D} {dtype}")
    s, thr, Q, K, V = case(T, HQ, D, k, dtype, B=B, seed=9)
    b, rows = B - 1, [64, 95, 96, 127, 128, 191, 255, 256, T - 1]
    if dtype is F32:
        Q[b, rows, HQ - 1] *= 2.0 ** 62  # beyond the scales
    elif dtype is HF:  # only keys of V = 0 selected
        V[b, 7] = 0.0
        s[b, rows], thr[b, rows] = -9.0, 0.0
        s[b, rows, 7] = 9.0
    else:
        Q[b, rows, HQ - 1] = math.nan
    args = tuple(x.to(dev) for x in (s, thr, Q, K, V))
    d, g = (sparse_attention_hip(*args, kernel=n)[b].cpu() for n in ("dense", "gather"))
    assert torch.equal(torch.nan_to_num(d[rows], nan=7e7), torch.nan_to_num(g[rows], nan=7e7))
    others = [t for t in range(64, T) if t not in rows]
    assert bool((d != g)[others].flatten(1).any(dim=1).all())


@pytest.mark.parametrize("span", [4, 9, 30, 70])
def test_dense_fp32_ranges(dev, span):
    """fp32 operands of very different magnitude: V tiles on neighbouring and on
    far-apart scales (beyond 2^-60 gathered), Q and K rows scaled against each
    other, rows of zeros, and rows beyond the scales."""
    T, HQ, D, k = 300, 2, 64, 25
    s, thr, Q, K, V = case(T, HQ, D, k, F32, seed=span)
    say(f"dense ranges span={span}")
    V = V.clone()
    V[:, 100:200] *= 2.0 ** -span
    V[:, 10] = 0.0
    K = K.clone()
    K[:, 130:140] *= 2.0 ** -span
    K[:, 20] = 0.0
    Q = Q * 2.0 ** min(span, 40)
    K = K * 2.0 ** -min(span, 40)
    Q[:, 33] = 0.0
    out = sparse_attention_hip(*(x.to(dev) for x in (s, thr, Q, K, V)), kernel="dense").cpu()
    want = O.sparse_attn_threshold(s, thr, Q, K, V)
    # rows that selected keys of 100..199 only would need the bound of those
    assert float((out.double() - want).abs().max()) <= bound(Q, K, V, T)


def test_dense_arguments(dev):
    x = torch.zeros(1, 64, 2, 32, device=dev)
    s, t = torch.zeros(1, 64, 64, device=dev), torch.zeros(1, 64, 1, device=dev)
    with pytest.raises(L.DSAUnsupported):
        sparse_attention_hip(s, t, x, x, x, kernel="dense")


@pytest.mark.parametrize("B,T,k,HQ,D,dtype", [(8, 1024, 64, 8, 64, F32), (2, 2048, 256, 16, 128, HF),
                                                (2, 3001, 300, 16, 128, HF), (4, 4096, 256, 8, 64, F32)])
def test_split_forward_takes_it(dev, B, T, k, HQ, D, dtype):
    """The split forward at shapes the rule gives to the dense kernel equals
    its stages run apart."""
    from dsa_attention import dsa_split_hip
    from lightning_indexer import indexer_scores_hip
    from topk_threshold import topk_threshold

    assert L.lib().dsa_sparse_attn_pick(L.dtype_code(dtype), B, T, HQ, D, D, k) == 1
    ins = tuple(x.to(dev) for x in O.make_inputs(B, T, 4, 32, HQ, D, D, dtype=dtype))
    sc = indexer_scores_hip(*ins[:3], write_upper=False)
    thr = topk_threshold(sc, k, causal=True)
    want = sparse_attention_hip(sc, thr, *ins[3:], kernel="dense")
    assert torch.equal(dsa_split_hip(*ins, k), want)


@pytest.mark.parametrize("B,T,k,HI,DI,HQ,D,dtype,split", [
    (4, 512, 32, 64, 128, 4, 128, BF, 1), (2, 1024, 64, 8, 64, 8, 64, F32, 1),
    (3, 950, 40, 16, 128, 4, 64, BF, 1), (2, 1500, 16, 4, 32, 4, 32, F32, 0),
    (16, 512, 32, 4, 32, 4, 32, F32, 0), (2, 100, 9, 8, 128, 4, 32, BF, 0)])
def test_forward_picks_split_or_fused(dev, B, T, k, HI, DI, HQ, D, dtype, split):
    """Either side of the forward's rule gives the same attention: the other
    form's output up to fp32 rounding, rows whose selection differs by a
    near-tie apart (at most a handful)."""
    import dsa_attention as DA

    ins = tuple(x.to(dev) for x in O.make_inputs(B, T, HI, DI, HQ, D, D, dtype=dtype, seed0=T))
    assert DA._split_is_faster(*ins, k) == bool(split)
    got = DA.dsa_forward_hip(*ins, k)
    assert torch.equal(got, (DA.dsa_split_hip if split else DA.dsa_fused_hip)(*ins, k))
    other = (DA.dsa_fused_hip if split else DA.dsa_split_hip)(*ins, k)
    off = (got - other).abs().amax(dim=(-1, -2)) > 2 * bound(*(x.cpu() for x in ins[3:]), T)
    assert int(off.sum()) <= max(2, B * T // 1000)


@pytest.mark.parametrize("B,T,k,HQ,D,dtype", [(2, 2048, 256, 16, 128, HF), (1, 4200, 300, 4, 64, BF)])
def test_forward_without_its_workspace(dev, monkeypatch, B, T, k, HQ, D, dtype):
    """Where the split forward's workspace and the dense kernel's cannot be
    had, the stages run apart on the kernels that need none; a dense kernel
    asked for by name raises."""
    from dsa_attention import dsa_split_hip, selection_mask, sparse_attention_from_mask
    from lightning_indexer import indexer_scores_hip
    from topk_threshold import topk_threshold

    ins = tuple(x.to(dev) for x in O.make_inputs(B, T, 4, 32, HQ, D, D, dtype=dtype))
    sc = indexer_scores_hip(*ins[:3], write_upper=False)
    thr = topk_threshold(sc, k, causal=True)
    if L.lib().dsa_sparse_attn_uses_mask(L.dtype_code(dtype), T, HQ, D, D):
        want = sparse_attention_from_mask(selection_mask(sc, thr), *ins[3:])
    else:
        want = sparse_attention_hip(sc, thr, *ins[3:], kernel="gather")
    empty = torch.empty

    def no_workspace(*a, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no workspace")
        return empty(*a, **kw)

    monkeypatch.setattr(torch, "empty", no_workspace)
    assert torch.equal(dsa_split_hip(*ins, k), want)
    with pytest.raises(torch.OutOfMemoryError):
        sparse_attention_hip(sc, thr, *ins[3:], kernel="dense")


def test_forced_staged_refuses_what_it_refused(dev):
    """A staged kernel asked for by name stays refused for other shapes,
    whatever top_k says of the dense kernel."""
    x = torch.zeros(1, 3072, 4, 64, device=dev, dtype=BF)
    s, t = torch.zeros(1, 3072, 3072, device=dev), torch.zeros(1, 3072, 1, device=dev)
    with pytest.raises(L.DSAUnsupported):
        sparse_attention_hip(s, t, x, x, x, kernel="staged", top_k=3072)
