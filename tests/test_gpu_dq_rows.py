"""dQ from the dS store on both sides of the rule that picks its kernel (use_rows_kernel in gfa_api.hip:
bwd_dq_rows_kernel up to 256 row blocks, 512 under full causal masking; bwd_dq_ds_kernel past it),
against the recomputing dQ kernel, at the edges of the 32-key tiles, key groups and layouts.

Both round dS to the 16-bit type before dS K, from fp32 values that differ in the last bits, so a
rounding may fall to the neighbouring value: at most one unit roundoff of dS in every term, 2^-8
(bf16) or 2^-11 (fp16) of the result's norm. Where dP - delta cancels (a row that sees one key: dQ is
zero) what is left is the fp32 error of those sums, 2^-22 of |dO| |V| ~ D per key, times scale |K| ~
D^-0.5 per element. Padding rows are exactly zero.
"""
from __future__ import annotations

import pytest
import torch

from conftest import exact64, make_inputs, recomputing

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
CASES = [
    # B, Hq, Hkv, N, D, causal, window, feature
    *((1, 4, 2, n, d, True, 0, "plain") for d in (512, 256) for n in (1, 31, 32, 33, 65, 129, 160, 257)),
    *((1, 4, 1, n, d, False, 0, "plain") for d in (512, 256) for n in (33, 96, 130)),
    *((2, 4, 2, n, 256, True, 50, "plain") for n in (64, 100, 300)),
    (1, 4, 2, 200, 512, True, 70, "plain"),
    (2, 4, 2, 200, 512, True, 0, "segments"),
    (2, 4, 2, 333, 256, True, 64, "segments"),
    (2, 4, 2, 130, 256, False, 0, "segments"),
    (1, 4, 2, 161, 256, True, 0, "softcap"),
    (1, 4, 2, 97, 512, False, 0, "dropout"),
    (4, 32, 4, 97, 512, True, 0, "plain"),      # 512 row blocks, causal: the last small grid
    (4, 32, 4, 129, 512, True, 0, "plain"),     # 640
    (4, 32, 16, 65, 256, False, 0, "plain"),    # 384, not causal: past the line
    (4, 32, 16, 129, 256, True, 40, "segments"),
    (4, 32, 16, 150, 256, True, 0, "softcap"),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window,feature", CASES)
def test_matches_recomputing(B, Hq, Hkv, N, D, causal, window, feature, dtype, device):
    import gemma_triton_flash_attn_amd as gfa
    from gemma_triton_flash_attn_amd.attention import _backward, _forward, backward_workspace

    print(f"case B={B} {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype} {feature}", flush=True)
    q, k, v, do = make_inputs(B, Hq, Hkv, N, D, dtype, device, seed=N + D, layout="bnhd" if N % 2 else "bhnd")
    kw = {"plain": {}, "softcap": {"softcap": 10.0}, "dropout": {"dropout_p": 0.2, "dropout_seed": 7},
          "segments": {}}[feature]
    if feature == "segments":  # a packed row (with a one-token document), then padded and empty rows
        rows = [gfa.segments.from_cu_seqlens([0, 1, N // 3, N // 2 + 1, N], N, device=device)]
        rows += [gfa.segments.from_lengths([n], N, device=device) for n in (N // 2, 0, N)[:B - 1]]
        kw["segments"] = tuple(torch.cat([r[i] for r in rows]) for i in (0, 1))
    window = 0 if window >= N else window
    assert backward_workspace(B, Hq, Hkv, N, D, causal, window, dtype, segments="segments" in kw)[1]
    sc = D ** -0.5
    o, lse = _forward(q, k, v, causal, window, sc, True, **kw)
    got = _backward(q, k, v, o, lse, do, causal, window, sc, **kw)[0]
    with recomputing():
        want = _backward(q, k, v, o, lse, do, causal, window, sc, **kw)[0]
    diff, norm = float((got.double() - want.double()).norm()), float(want.double().norm())
    floor = 2.0 ** -22 * D ** 0.5 * got.numel() ** 0.5
    assert torch.isfinite(got).all() and diff <= U[dtype] * norm + floor, (diff, norm)
    if feature == "segments":
        pad = (kw["segments"][0] == kw["segments"][1])[:, None, :, None].expand_as(got)
        assert bool((got[pad] == 0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window,feature",
                         [c for c in CASES if c[7] in ("plain", "segments") and c[3] > 32])
def test_matches_exact(B, Hq, Hkv, N, D, causal, window, feature, dtype, device):
    """dQ against 64 bits. Its operands P, dS and O are rounded to the 16-bit type (delta = rowsum(dO O) from
    the rounded O) and so is dQ, each rounding within u / 2 of its value; independent, they give an error of
    about u / 2 of the norm, and 2 u covers it with room for the first rows, whose few keys add
    nothing up."""
    import gemma_triton_flash_attn_amd as gfa
    from gemma_triton_flash_attn_amd.attention import _backward, _forward

    print(f"case B={B} {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype} {feature}", flush=True)
    q, k, v, do = make_inputs(B, Hq, Hkv, N, D, dtype, device, seed=N + D)
    segs = None
    if feature == "segments":
        rows = [gfa.segments.from_cu_seqlens([0, 1, N // 3, N // 2 + 1, N], N, device=device)]
        rows += [gfa.segments.from_lengths([n], N, device=device) for n in (N // 2, 0, N)[:B - 1]]
        segs = tuple(torch.cat([r[i] for r in rows]) for i in (0, 1))
    window = 0 if window >= N else window
    o, lse = _forward(q, k, v, causal, window, D ** -0.5, True, segments=segs)
    got = _backward(q, k, v, o, lse, do, causal, window, D ** -0.5, segments=segs)[0]
    want = exact64(q, k, v, causal, window, segs, do)[1]
    assert float((got.double() - want).norm()) <= 2 * U[dtype] * float(want.norm())
