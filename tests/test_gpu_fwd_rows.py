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

from conftest import exact64, make_inputs
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


def _compare(B, Hq, Hkv, N, D, causal, window, dtype, device, feature="plain", layout="bhnd"):
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


# The grids on both sides of each line of the rule.
EDGES = [
    (1, 8, 1, 1024, 512, False, 0),    # 256 row blocks: the last grid of one round
    (1, 8, 1, 1025, 512, False, 0),    # 264: the general forward
    (1, 8, 1, 2048, 512, True, 0),     # 512, causal
    (1, 8, 1, 2049, 512, True, 0),
    (1, 8, 4, 2000, 256, True, 0),
    (1, 8, 1, 1000, 256, True, 512),   # 256, windowed: the last small grid
    (1, 8, 1, 1040, 256, True, 512),
    (1, 4, 2, 2048, 64, True, 700),
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
]


@pytest.mark.parametrize("feature", ["plain", "segments"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,window", EDGES)
def test_rule_edges(B, Hq, Hkv, N, D, causal, window, dtype, feature, device):
    """Both forwards, whichever the rule picks, against 64 bits, in every 32-row block of every head.

    The roundings of P and of O are independent, each uniform within half a unit in the last place (u / 2
    relative, at most), so on random V a block's error is about sqrt(2 / 3) u / 2 of its norm; 2 u is five
    times that, and a single 32-key tile lost or read twice changes a row of n keys by sqrt(32 / n), eight
    times the bound and more up to 8192 keys in bf16. A block whose rows see nothing is zero. 1e-6 per
    element: fp32 sums, subnormal P in fp16."""
    from gemma_triton_flash_attn_amd.attention import _forward

    print(f"case B={B} {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype} {feature}", flush=True)
    g = torch.Generator(device=device).manual_seed(N + D)
    q, k, v = (torch.randn(B, h, N, D, generator=g, device=device).to(dtype) for h in (Hq, Hkv, Hkv))
    segs = _tables(B, N, device) if feature == "segments" else None
    window = 0 if window >= N else window
    want = exact64(q, k, v, causal, window, segs)

    def blocks(t):
        return torch.nn.functional.pad(t, (0, 0, 0, -N % 32)).view(B, Hq, -1, 32 * D).norm(dim=-1)

    for bkv in (0, GENERAL_BKV[D]):
        o, lse = _forward(q, k, v, causal, window, D ** -0.5, True, block_kv=bkv, segments=segs)
        assert bool((blocks(o.double() - want) <= 2 * U[dtype] * blocks(want) + 1e-6 * (32 * D) ** 0.5).all()), bkv
        if bkv == 0:
            rows = lse[..., :N]
        else:
            fin = torch.isfinite(rows)
            assert torch.equal(fin, torch.isfinite(lse[..., :N]))
            assert float((rows - lse[..., :N])[fin].abs().max()) <= 1e-4


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


def _odd(kind, k, v, j):
    """Key j made to score +-inf (by the sign of q's first element) or NaN, or its V to hold an infinity."""
    if kind == "inf_key":
        k[:, :, j, 0] = float("inf")
    elif kind == "nan_key":
        k[:, :, j, 5] = float("nan")
    else:
        v[:, :, j, 3] = float("inf")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["inf_key", "nan_key", "inf_value"])
@pytest.mark.parametrize("D,N", [(512, 230), (256, 300), (128, 500), (64, 900)])
@pytest.mark.parametrize("where", [0.02, 0.2, 0.55, 0.97])
def test_infinities_and_nans(where, D, N, kind, dtype, device):
    """One key that is not finite, in one key group's tiles only. A row that scores it +inf or NaN is NaN
    in every column and in its LSE, a row that scores it -inf is what it is without that key, a
    row that does not see it (causal, in an earlier tile) is what it is without it; an infinity in V
    reaches its own column of the rows that see it. As the general forward, and as 64 bits: 4 u of a
    row's norm covers the roundings of P and O (about sqrt(2 / 3) u / 2), and one of n <= 900 keys taken
    or left out is 1 / sqrt(n) of it."""
    from gemma_triton_flash_attn_amd.attention import _forward

    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(1, h, N, D, generator=g).to(dtype) for h in (4, 2, 2))
    q[..., 0] = torch.where(q[..., 0].abs() < 0.1, 0.5, q[..., 0])
    j = int(where * N)
    clean = exact64(q, k, v, True).to(device)
    without = (torch.arange(N) != j).expand(N, N) & (torch.arange(N)[:, None] >= torch.arange(N))
    s = (q.double() @ k.double().repeat_interleave(2, 1).transpose(2, 3)) * D ** -0.5
    s = s.masked_fill(~without, float("-inf"))
    skipped = torch.nan_to_num(torch.softmax(s, -1)) @ v.double().repeat_interleave(2, 1)
    _odd(kind, k, v, j)
    q, k, v, skipped = (t.to(device) for t in (q, k, v, skipped))
    rows = torch.arange(N, device=device)

    def near(o, want):
        return (o.double() - want).norm(dim=-1) <= 4 * U[dtype] * want.norm(dim=-1) + 1e-5

    for bkv in (0, GENERAL_BKV[D]):
        o, lse = _forward(q, k, v, True, 0, D ** -0.5, True, block_kv=bkv)
        early = rows < j // 128 * 128
        assert bool(near(o, clean)[:, :, early].all())
        late = o[:, :, j:]
        if kind == "inf_value":
            assert not bool(torch.isfinite(late[..., 3]).any())
            others = [c for c in range(D) if c != 3]
            assert bool(near(late[..., others], clean[:, :, j:][..., others]).all())
            continue
        nan = torch.ones_like(q[..., 0], dtype=torch.bool) if kind == "nan_key" else q[..., 0] > 0
        nan = nan & (rows >= j)
        assert bool(o[nan].isnan().all()) and bool(lse[..., :N][nan].isnan().all())
        if kind == "inf_key":
            # (row j = 0 sees that key alone: no key is left)
            rest = (rows >= max(j, 1)) & ~nan
            assert bool(torch.isfinite(lse[..., :N][rest]).all())
            assert bool(near(o, skipped)[rest].all())
