"""The attention calls this framework is timed on, through its public entry points.

A case is one attention layer of a model, forward only or forward and backward. Its keys:

  path     "layer"  a transformers model's layer in a prompt (prefill) pass: ``triton_gqa_attention``, inputs
                    as the (B, H, N, D) views of (B, N, H, D) projections, position ids and, with ``real``
                    below 1, the padding mask a model hands over
           "infer"  ``attention_flash_gqa`` (no autograd, no LSE)
           "train"  ``flash_attn_gqa_train`` and the gradients of q, k and v
  B, Hq, Hkv, N, D, causal, window, dtype, softcap   the layer
  docs     > 0: packed documents per row (segment tables, built once per batch as a training loop does)
  real     share of real tokens in the shortest row of a right-padded batch (1: nothing is padded)

Work and bytes count attended (query, key) pairs exactly: causal, window and document bounds included.
"""
from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch

import gemma_triton_flash_attn_amd as gfa
from gemma_triton_flash_attn_amd import segments
from gemma_triton_flash_attn_amd.hf_integration import triton_gqa_attention

_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}
_MAX_FLOPS = 3.07e13  # the largest listed case has 3.08e13


def _case(path, B, Hq, Hkv, N, D, causal=True, window=0, dtype="bf16", softcap=0.0, docs=0, real=1.0, **kw):
    return dict(kw, path=path, B=B, Hq=Hq, Hkv=Hkv, N=N, D=D, causal=causal, window=window, dtype=dtype,
                softcap=softcap, docs=docs, real=real)


def listed():
    return [
        # Gemma-4-E2B (8 query heads, 1 KV head), a short chat prompt: a sliding layer. The smallest call; a model
        # makes 28 of them per prompt, and launches and host work count.
        _case("layer", 1, 8, 1, 333, 256, window=512, name="e2b_sliding_short_prompt"),
        # The same model's global layer on a prompt of about a thousand tokens.
        _case("layer", 1, 8, 1, 1024, 512, name="e2b_global_1k_prompt"),
        # A small serving batch of prompts of unequal length, right-padded, through the same global layer.
        _case("layer", 4, 8, 1, 1500, 512, real=0.4, name="e2b_global_padded_batch"),
        # Long-context prefill (bench.py's end-to-end model at N=16384): its sliding layer.
        _case("layer", 1, 8, 1, 16384, 256, window=512, name="e2b_sliding_16k_prefill"),
        # A larger model's global layer, 8k prompt, the plain inference entry point.
        _case("infer", 1, 32, 4, 8192, 512, name="global_8k_prefill"),
        # Training, global layer, 16k: the headline benchmark and the largest case.
        _case("train", 1, 32, 4, 16384, 512, name="global_16k_train"),
        # Training at an ordinary fine-tuning length, global layer of the 16-head model, two rows, fp16.
        _case("train", 2, 16, 2, 2048, 512, dtype="fp16", name="global_2k_train_fp16"),
        # Training, sliding layer of the 16-head model (16:8, window 1024), 16k.
        _case("train", 1, 16, 8, 16384, 256, window=1024, name="sliding_16k_train"),
        # The same layer on packed documents of unequal length.
        _case("train", 1, 16, 8, 8192, 256, window=1024, docs=7, name="sliding_packed_train"),
        # A Llama-shaped layer (head dim 128, 32:8) at a common training length.
        _case("train", 1, 32, 8, 4096, 128, name="d128_4k_train"),
        # Head dim 64, as many KV heads as query heads, no causal mask (an encoder), ragged length, fp16.
        _case("train", 2, 16, 16, 2001, 64, causal=False, dtype="fp16", name="d64_encoder_train_fp16"),
        # A Gemma-2-shaped layer: logits soft-capped at 50, head dim 256, fine-tuning length.
        _case("train", 1, 8, 4, 2048, 256, softcap=50.0, name="softcap_2k_train"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more layer of the same families: the heads, head dims, masks and options above, sequence lengths over
    their range (odd ones among them), batches of 1 to 4."""
    family = rng.choice(["sliding", "sliding", "global", "global", "padded", "packed", "d128", "d64", "softcap"])
    train = rng.random() < 0.5
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    n = _log_int(rng, 96, 16384)
    if rng.random() < 0.4:
        n = max(64, n // 64 * 64)
    b = rng.choice([1, 1, 2, 4])
    if family == "sliding":
        hq, hkv, w = rng.choice([(8, 1, 512), (16, 8, 1024), (32, 16, 1024)])
        c = _case("train" if train else rng.choice(["layer", "infer"]), b, hq, hkv, n, 256, window=w, dtype=dtype)
    elif family == "global":
        hq, hkv = rng.choice([(8, 1), (16, 2), (32, 4)])
        c = _case("train" if train else rng.choice(["layer", "infer"]), b, hq, hkv, n, 512, dtype=dtype)
    elif family == "padded":
        d, w = rng.choice([(512, 0), (256, 512)])
        c = _case("layer", rng.choice([2, 3, 4]), 8, 1, n, d, window=w, dtype=dtype, real=rng.choice([0.3, 0.5, 0.8]))
    elif family == "packed":
        d, hq, hkv, w = rng.choice([(256, 16, 8, 1024), (512, 16, 2, 0)])
        n = max(n, 512)
        c = _case("train", 1, hq, hkv, n, d, window=w, dtype=dtype, docs=rng.randint(2, 12))
    elif family == "d128":
        hq, hkv = rng.choice([(32, 8), (16, 4), (16, 16)])
        c = _case("train" if train else "layer", b, hq, hkv, n, 128, window=rng.choice([0, 0, 1024]), dtype=dtype)
    elif family == "d64":
        hq, hkv = rng.choice([(16, 16), (32, 32), (32, 8)])
        c = _case("train" if train else "infer", b, hq, hkv, n, 64, causal=rng.random() < 0.5, dtype=dtype)
    else:
        hq, hkv, w = rng.choice([(8, 4, 0), (8, 4, 4096), (16, 8, 4096)])
        c = _case("train" if train else "layer", b, hq, hkv, n, 256, window=w, softcap=50.0, dtype=dtype)
    while work(c)["flops"] > _MAX_FLOPS:
        c["N"] = c["N"] * 3 // 4
    return c


def _bounds(case):
    """Per batch row, its runs of tokens that attend to each other: [(first, end), ...] (padding in none)."""
    B, N = case["B"], case["N"]
    rng = random.Random(1000 * N + 10 * case["docs"] + B)
    if case["docs"]:
        cuts = [sorted(rng.sample(range(1, N), case["docs"] - 1)) for _ in range(B)]
        return [list(zip([0] + c, c + [N])) for c in cuts]
    if case["real"] < 1.0:
        least = max(1, int(case["real"] * N))
        rows = [N, least] + [rng.randint(least, N) for _ in range(B)]
        return [[(0, n)] for n in rows[:B]]
    return [[(0, N)] for _ in range(B)]


def _pairs(case):
    """Attended (query, key) pairs of one query head, over the batch."""
    w = case["window"] if case["causal"] else 0
    total = 0
    for row in _bounds(case):
        for a, e in row:
            n = e - a
            if not case["causal"]:
                total += n * n
            elif 0 < w < n:
                total += w * (w + 1) // 2 + w * (n - w)
            else:
                total += n * (n + 1) // 2
    return total


def work(case):
    """Each input read once and each output written once; two matrix products per pair forward, five more backward."""
    B, Hq, Hkv, N, D = (case[x] for x in ("B", "Hq", "Hkv", "N", "D"))
    q_bytes, kv_bytes = 2 * B * Hq * N * D, 2 * B * Hkv * N * D
    if case["path"] == "train":
        # in: q, k, v, dO; out: O, dq, dk, dv
        return {"bytes": 4 * q_bytes + 4 * kv_bytes, "flops": 14 * D * Hq * _pairs(case)}
    return {"bytes": 2 * q_bytes + 2 * kv_bytes, "flops": 4 * D * Hq * _pairs(case)}


def _scale(case):
    return 1.0 / math.sqrt(case["D"])


def _inputs(case, seed, dev):
    """q, k, v, dO as (B, H, N, D), standard normal (as after Gemma's q/k norms). The layers' inputs are views of
    (B, N, H, D) storage, the layout of a model's projections."""
    B, Hq, Hkv, N, D = (case[x] for x in ("B", "Hq", "Hkv", "N", "D"))
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = _DTYPE[case["dtype"]]

    def one(heads):
        if case["path"] == "layer":
            return torch.randn(B, N, heads, D, generator=g, device=dev).to(dt).transpose(1, 2)
        return torch.randn(B, heads, N, D, generator=g, device=dev).to(dt)

    return one(Hq), one(Hkv), one(Hkv), one(Hq)


def prepare(case, seed):
    dev = torch.device("cuda")
    q, k, v, do = _inputs(case, seed, dev)
    st = dict(case=case, q=q, k=k, v=v)
    if case["path"] == "train":
        for x in (q, k, v):
            x.requires_grad_(True)
        st["do"] = do
        st["segments"] = None
        if case["docs"]:
            cu = [0] + [e for _, e in _bounds(case)[0]]
            st["segments"] = segments.from_cu_seqlens(torch.tensor(cu, device=dev), case["N"])
    elif case["path"] == "layer":
        # what transformers hands to an attention function: the module, position ids, and the
        # (B, N) padding mask where rows are padded
        st["module"] = SimpleNamespace(is_causal=case["causal"], head_dim=case["D"])
        st["position_ids"] = torch.arange(case["N"], device=dev)[None]
        st["mask"] = None
        if case["real"] < 1.0:
            n = torch.tensor([row[0][1] for row in _bounds(case)], device=dev)
            st["mask"] = torch.arange(case["N"], device=dev)[None] < n[:, None]
    return st


def run(state):
    c = state["case"]
    cap = c["softcap"] or None
    if c["path"] == "train":
        q, k, v = state["q"], state["k"], state["v"]
        o = gfa.flash_attn_gqa_train(q, k, v, c["causal"], c["window"], scale=_scale(c), segments=state["segments"],
                                     softcap=cap)
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["do"])
        return o.detach(), dq, dk, dv
    with torch.no_grad():
        if c["path"] == "infer":
            return gfa.attention_flash_gqa(state["q"], state["k"], state["v"], c["causal"], c["window"],
                                           scale=_scale(c), softcap=cap)
        out, _ = triton_gqa_attention(state["module"], state["q"], state["k"], state["v"], state["mask"],
                                      scaling=_scale(c), softcap=cap, sliding_window=c["window"] or None,
                                      position_ids=state["position_ids"])
        return out


def tolerance(case):
    """Four times the relative error against the 64-bit result (bf16 up to 2.6e-3, fp16 up to 3.3e-4, for every
    output): inputs, P, dS and outputs are rounded to the 16-bit type, sums are 32-bit."""
    return {"rel": 1.1e-2 if case["dtype"] == "bf16" else 1.4e-3}


def exact(case, seed):
    """The same outputs in 64 bits, from plain torch: per head, in blocks of query rows."""
    dev = torch.device("cuda")
    q, k, v, do = _inputs(case, seed, dev)
    B, Hq, Hkv, N, D = (case[x] for x in ("B", "Hq", "Hkv", "N", "D"))
    train, causal, cap = case["path"] == "train", case["causal"], case["softcap"]
    window = case["window"] if causal else 0
    scale = _scale(case)
    out = torch.zeros(B, Hq, N, D, dtype=torch.float64, device=dev)
    dq = torch.zeros_like(out) if train else None
    dk = torch.zeros(B, Hkv, N, D, dtype=torch.float64, device=dev) if train else None
    dv = torch.zeros_like(dk) if train else None
    for b, row in enumerate(_bounds(case)):
        for first, end in row:
            for head in range(Hq):
                kh = head // (Hq // Hkv)
                kd, vd = k[b, kh].double(), v[b, kh].double()
                for r0 in range(first, end, 1024):
                    r1 = min(r0 + 1024, end)
                    k0 = max(first, r0 - window + 1) if window > 0 else first
                    k1 = r1 if causal else end
                    qb, kb, vb = q[b, head, r0:r1].double(), kd[k0:k1], vd[k0:k1]
                    s = (qb @ kb.t()) * scale
                    if cap > 0:
                        t = torch.tanh(s / cap)
                        s = cap * t
                    if causal:
                        gap = torch.arange(r0, r1, device=dev)[:, None] - torch.arange(k0, k1, device=dev)[None]
                        hidden = gap < 0
                        if window > 0:
                            hidden |= gap >= window
                        s = s.masked_fill(hidden, float("-inf"))
                    p = torch.softmax(s, dim=1)
                    o = p @ vb
                    out[b, head, r0:r1] = o
                    if train:
                        dob = do[b, head, r0:r1].double()
                        dv[b, kh, k0:k1] += p.t() @ dob
                        ds = p * (dob @ vb.t() - (dob * o).sum(1, keepdim=True))
                        if cap > 0:
                            ds = ds * (1 - t * t)
                        dq[b, head, r0:r1] = scale * (ds @ kb)
                        dk[b, kh, k0:k1] += scale * (ds.t() @ qb)
    if train:
        return out, dq, dk, dv
    return out.transpose(1, 2) if case["path"] == "layer" else out
