"""Split dK/dV grids whose key blocks get different split counts (plan_dkv in gfa_plan.h; a block with one
split writes its rows directly) against the unsplit grid (q_splits = 1), on grids small enough to be
split: every form of the kernel, ragged and odd sizes, more than 64 key blocks (the block search's
second batch), windows, segment tables, soft-capping and dropout.

P, dS and their products are the same; only the fp32 sums are taken in another order (1e-5 of the
largest gradient covers their difference) before the one rounding to 16 bits, which can then fall
to the neighbouring value: one unit in the last place, 2^-7 (bf16) or 2^-10 (fp16) of the value.
"""
from __future__ import annotations

import pytest
import torch

from conftest import exact64, make_inputs

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}
CASES = [
    # B, Hq, Hkv, N, D, causal, window, dtype, feature
    (1, 16, 8, 800, 256, True, 0, torch.bfloat16, "plain"),
    (1, 8, 4, 1709, 256, True, 0, torch.bfloat16, "softcap"),
    (1, 8, 4, 1051, 256, True, 300, torch.float16, "dropout"),
    (1, 32, 16, 700, 256, True, 300, torch.bfloat16, "plain"),
    (1, 8, 1, 5000, 256, True, 512, torch.bfloat16, "plain"),
    (1, 16, 8, 333, 256, False, 0, torch.float16, "segments"),
    (2, 16, 2, 700, 512, True, 0, torch.float16, "plain"),
    (1, 16, 2, 1300, 512, True, 0, torch.bfloat16, "segments"),
    (1, 8, 1, 97, 512, True, 0, torch.bfloat16, "softcap"),
    (1, 4, 1, 65, 512, False, 0, torch.float16, "dropout"),
    (1, 32, 8, 1000, 128, True, 0, torch.bfloat16, "plain"),
    (1, 4, 4, 33, 128, True, 0, torch.float16, "plain"),
    (1, 2, 1, 9000, 64, True, 0, torch.bfloat16, "plain"),
    (1, 16, 16, 1001, 64, True, 0, torch.float16, "segments"),
    (3, 6, 2, 129, 64, False, 0, torch.bfloat16, "dropout"),
]


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window,dtype,feature", CASES)
def test_matches_unsplit(B, Hq, Hkv, N, D, causal, window, dtype, feature, device):
    import gemma_triton_flash_attn_amd as gfa
    from gemma_triton_flash_attn_amd import _lib
    from gemma_triton_flash_attn_amd.attention import _backward, _forward

    print(f"case B={B} {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype} {feature}", flush=True)
    assert _lib.bwd_workspace_size(B, Hq, Hkv, N, D, causal, window) > 0, "the case should be split"
    q, k, v, do = make_inputs(B, Hq, Hkv, N, D, dtype, device, seed=N + D)
    kw = {"plain": {}, "softcap": {"softcap": 10.0}, "dropout": {"dropout_p": 0.2, "dropout_seed": 99},
          "segments": {}}[feature]
    if feature == "segments":
        cuts = [0, 1, N // 3, N // 2 + 1, N]
        kw["segments"] = gfa.segments.from_cu_seqlens(cuts, N, device=device)
    sc = D ** -0.5
    o, lse = _forward(q, k, v, causal, window, sc, True, **kw)
    got = _backward(q, k, v, o, lse, do, causal, window, sc, **kw)
    for _ in range(2):  # the same splits, the same order: run to run equal
        again = _backward(q, k, v, o, lse, do, causal, window, sc, **kw)
        assert all(torch.equal(a, b) for a, b in zip(got[:3], again[:3]))
    for splits in (1, 2, 4):
        ref = _backward(q, k, v, o, lse, do, causal, window, sc, q_splits=splits, **kw)
        assert torch.equal(got[0], ref[0])  # dQ does not depend on the splits
        for name, a, b in zip(("dK", "dV"), got[1:3], ref[1:3]):
            a, b = a.float(), b.float()
            bound = ULP[dtype] * b.abs() + 1e-5 * b.abs().max()
            assert bool(((a - b).abs() <= bound).all()), (name, splits, float((a - b).abs().max()))


def test_more_planes_than_a_grid_dimension(device):
    """An explicit split of more (tensor, batch, KV head) planes than a launch grid's second dimension
    holds (65535): the reduction walks them."""
    from gemma_triton_flash_attn_amd.attention import _backward, _forward

    B, N, D, dtype = 33000, 33, 128, torch.bfloat16
    g = torch.Generator(device=device).manual_seed(1)
    q, k, v, do = (torch.randn(B, 1, N, D, generator=g, device=device).to(dtype) for _ in range(4))
    o, lse = _forward(q, k, v, True, 0, D ** -0.5, True)
    got, ref = (_backward(q, k, v, o, lse, do, True, 0, D ** -0.5, q_splits=n) for n in (2, 1))
    for a, b in zip(got[1:3], ref[1:3]):
        a, b = a.float(), b.float()
        assert bool(((a - b).abs() <= ULP[dtype] * b.abs() + 1e-5 * b.abs().max()).all())


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window,dtype,feature",
                         [c for c in CASES if c[8] in ("plain", "segments") and c[3] <= 5000])
def test_matches_exact(B, Hq, Hkv, N, D, causal, window, dtype, feature, device):
    """dK and dV against 64 bits, in every block of 64 keys. P, dS, O and the results are rounded to the
    16-bit type, each within half a unit in the last place (u / 2, u = ULP / 2): independent, they
    give about u / 2 of a block's norm, and ULP = 2 u covers it."""
    import gemma_triton_flash_attn_amd as gfa
    from gemma_triton_flash_attn_amd.attention import _backward, _forward

    print(f"case B={B} {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype} {feature}", flush=True)
    q, k, v, do = make_inputs(B, Hq, Hkv, N, D, dtype, device, seed=N + D)
    segs = None
    if feature == "segments":
        segs = gfa.segments.from_cu_seqlens([0, 1, N // 3, N // 2 + 1, N], N, device=device)
    o, lse = _forward(q, k, v, causal, window, D ** -0.5, True, segments=segs)
    got = _backward(q, k, v, o, lse, do, causal, window, D ** -0.5, segments=segs)
    want = exact64(q, k, v, causal, window, segs, do)

    def blocks(t):
        return torch.nn.functional.pad(t, (0, 0, 0, -N % 64)).view(B, Hkv, -1, 64 * D).norm(dim=-1)

    for name, a, b in (("dK", got[1], want[2]), ("dV", got[2], want[3])):
        assert bool((blocks(a.double() - b) <= ULP[dtype] * blocks(b)).all()), name
