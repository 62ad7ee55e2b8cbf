"""The small-grid forward (gfa_fwd_rows.hip), which the library takes for short prompts, against the
general one (fwd_kernel, which an explicit ``block_kv`` always runs) and against the oracle.

Sizes sit at the edges of its tiles (32, 64 and 128 keys per wave at head dims 256 and 512, 128, 64;
32-row blocks; two or four key groups) and of the rule that selects it (256 to 1024 row blocks).

Both forwards round P to the 16-bit type before P V (unit roundoff u = 2^-8 in bf16, 2^-11 in fp16,
relative to P, against their own reference max) and O at the end, so with A = softmax |V| they
differ by at most 2 u (A + |O|), plus fp32 sums (1e-4 covers them, and fp16's subnormal P).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_inputs
from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}
GENERAL_BKV = {512: 32, 256: 32, 128: 64, 64: 64}
SEED = 0x5EED_77


def _np(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def _tables(B, N, device):
    """Row 0 packed (a one-token document among them), the others right-padded, the last all padding."""
    import gemma_triton_flash_attn_amd as gfa

    cuts = sorted({1, N // 3 + 1, N // 2 + 1})
    rows = [gfa.segments.from_cu_seqlens([0] + [c for c in cuts if c < N] + [N], N, device=device)]
    rows += [gfa.segments.from_lengths([n], N, device=device) for n in ([N // 2, 0][:B - 1])]
    return torch.cat([r[0] for r in rows]), torch.cat([r[1] for r in rows])


def _compare(B, Hq, Hkv, N, D, causal, window, dtype, device, feature="plain", layout="bhnd", oracle=True):
    from gemma_triton_flash_attn_amd.attention import _forward

    print(f"case B={B} {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype} {feature} {layout}", flush=True)
    q, k, v = make_inputs(B, Hq, Hkv, N, D, dtype, device, seed=N + D, with_do=False, layout=layout)
    kw, okw = {}, {}
    if feature == "segments":
        kw["segments"] = _tables(B, N, device)
        okw["segments"] = tuple(t.cpu().numpy() for t in kw["segments"])
    elif feature == "softcap":
        kw["softcap"] = okw["softcap"] = 5.0
    elif feature == "dropout":
        kw.update(dropout_p=0.2, dropout_seed=SEED)
        okw["dropout"] = (0.2, SEED)
    w = 0 if window >= N else window
    sc = D ** -0.5
    o, lse = _forward(q, k, v, causal, w, sc, True, **kw)
    og, lg = _forward(q, k, v, causal, w, sc, True, block_kv=GENERAL_BKV[D], **kw)
    torch.cuda.synchronize()
    fin = torch.isfinite(lg[..., :N])
    assert torch.equal(fin, torch.isfinite(lse[..., :N]))
    assert float((lse[..., :N] - lg[..., :N])[fin].abs().max()) <= 1e-4
    if not oracle:
        # the bound with A <= max |V|
        bound = 2 * U[dtype] * (float(v.float().abs().max()) + og.float().abs()) + 1e-4
        assert bool(((o.float() - og.float()).abs() <= bound).all())
        return
    a_ref, _ = orc.forward(_np(q), _np(k), np.abs(_np(v)), causal, w, **okw)
    o_ref, _ = orc.forward(_np(q), _np(k), _np(v), causal, w, **okw)
    bound = 2 * U[dtype] * (a_ref + np.abs(o_ref)) + 1e-4
    assert bool((np.abs(_np(o) - _np(og)) <= bound).all()), np.abs(_np(o) - _np(og)).max()
    assert bool((np.abs(_np(o) - o_ref) <= bound).all()), np.abs(_np(o) - o_ref).max()


SIZES = {512: (1, 31, 33, 64, 65, 130, 200), 256: (1, 32, 33, 127, 129, 160, 257), 128: (63, 65, 129, 255, 257, 300),
         64: (129, 130, 255, 257, 383, 513)}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal,window", [(True, 0), (True, 37), (False, 0)])
@pytest.mark.parametrize("D,N", [(d, n) for d, ns in SIZES.items() for n in ns])
def test_edges(D, N, causal, window, dtype, device):
    _compare(1, 4, 2, N, D, causal, window, dtype, device, layout="bnhd" if N % 2 else "bhnd")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("feature", ["segments", "softcap", "dropout"])
@pytest.mark.parametrize("D,N,causal,window", [(512, 97, True, 0), (512, 70, False, 0), (256, 161, True, 50),
                                               (256, 140, False, 0), (128, 260, True, 0), (128, 200, True, 70),
                                               (64, 300, True, 0), (64, 390, False, 0)])
def test_features(D, N, causal, window, feature, dtype, device):
    _compare(3, 3, 1, N, D, causal, window, dtype, device, feature)


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window", [
    (1, 8, 1, 1024, 512, False, 0),    # 256 row blocks: the last grid of one round
    (1, 8, 1, 1025, 512, False, 0),    # 264: the general forward
    (1, 8, 1, 2048, 512, True, 0),     # 512, causal
    (1, 8, 1, 2049, 512, True, 0),
    (1, 8, 4, 2000, 256, True, 0),
    (1, 8, 1, 1000, 256, True, 512),
    (2, 4, 4, 1024, 64, True, 0),
    (1, 16, 4, 1024, 128, True, 0),
    (1, 16, 4, 1023, 128, True, 0),
    (3, 8, 2, 640, 128, True, 0),      # 480 blocks
    (3, 8, 2, 639, 128, True, 0),      # below 640 tokens: the general forward
    (1, 8, 4, 3072, 256, True, 0),     # 768: the last below 4096 tokens
    (1, 8, 4, 3073, 256, True, 0),
    (1, 8, 4, 4095, 64, True, 0),      # 1024 blocks, one token short
    (1, 8, 4, 4096, 128, True, 0),     # 1024, from 4096 tokens
    (1, 4, 1, 8100, 64, True, 0),
    (1, 8, 4, 2048, 64, False, 0),     # 512, no mask
    (1, 5, 5, 1537, 256, False, 0),
    (2, 4, 4, 2049, 128, False, 0),
])
def test_rule_edges(B, Hq, Hkv, N, D, causal, window, device):
    _compare(B, Hq, Hkv, N, D, causal, window, torch.bfloat16, device, oracle=False)


@pytest.mark.parametrize("dtype,jump", [(torch.float16, 20.0), (torch.bfloat16, 60.0), (torch.bfloat16, 40.0)])
@pytest.mark.parametrize("D,N,first", [(512, 150, 100), (512, 150, 149), (256, 300, 200), (256, 300, 40),
                                       (128, 500, 400), (64, 900, 700)])
def test_late_large_scores(D, N, first, dtype, jump, device):
    """Scores far above a key group's first tile, in some groups only: the workgroup redoes its rows
    with the exact row max (at 40 nats in bf16 the margin still holds and nothing is redone)."""
    from gemma_triton_flash_attn_amd.attention import _forward

    g = torch.Generator().manual_seed(9)
    u = torch.ones(D) / D ** 0.5
    q = torch.randn(1, 4, N, D, generator=g) * 0.1 + u * 4.0
    k = torch.randn(1, 2, N, D, generator=g) * 0.1
    k[:, :, first:] += u * (jump * D ** 0.5 / 4.0)
    v = torch.randn(1, 2, N, D, generator=g)
    q, k, v = (t.to(device=device, dtype=dtype) for t in (q, k, v))
    o, lse = _forward(q, k, v, True, 0, D ** -0.5, True)
    o_ref, lse_ref = orc.forward(_np(q), _np(k), _np(v), True, 0)
    a_ref, _ = orc.forward(_np(q), _np(k), np.abs(_np(v)), True, 0)
    assert torch.isfinite(o).all()
    bound = U[dtype] * (a_ref + np.abs(o_ref)) + 1e-3  # 1e-3: fp32 scores of size ~ 60 under exp
    assert bool((np.abs(_np(o) - o_ref) <= bound).all()), np.abs(_np(o) - o_ref).max()
    assert float(np.abs(_np(lse[..., :N]) - lse_ref).max()) <= 1e-3
