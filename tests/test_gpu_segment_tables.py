"""Segment tables built by the library's kernels (gfa_segments.hip) against the tensor operations of
segments.py on the CPU (equal, whole numbers), at the edges of their 1024-token workgroups."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 1023, 1024, 1025, 2049, 5000]


def _positions(kind, B, N):
    g = torch.Generator().manual_seed(N)
    pos = torch.arange(N).repeat(B, 1)
    if kind == "packed":
        for b in range(B):
            cuts = [0] + sorted(int(x) for x in torch.randint(1, max(N, 2), (7,), generator=g)) + [N]
            for a, e in zip(cuts, cuts[1:]):
                pos[b, a:e] = torch.arange(max(0, e - a))
    elif kind == "each":  # every token restarts
        pos.zero_()
    elif kind == "offset":  # one run that does not start at 0, and a restart at the last token
        pos += 17
        pos[-1, -1] = 3
    return pos


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("kind", ["plain", "packed", "each", "offset"])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_positions(kind, N, dtype, device):
    import gemma_triton_flash_attn_amd as gfa

    pos = _positions(kind, 3, N).to(dtype)
    want = gfa.segments.from_position_ids(pos)
    wide = torch.zeros(3, N + 5, dtype=dtype, device=device)
    wide[:, :N] = pos.to(device)
    for p in (pos.to(device), wide[:, :N]):
        got = gfa.segments.from_position_ids(p)
        assert isinstance(got, gfa.segments.SegmentTables)
        assert all(torch.equal(a.cpu(), b) and a.dtype == torch.int32 for a, b in zip(got, want))
    row = gfa.segments.from_position_ids(pos[:1].to(device).expand(4, N))  # one row for the batch
    assert all(torch.equal(a.cpu(), b[:1].expand(4, N)) for a, b in zip(row, want))


@pytest.mark.parametrize("N", SIZES)
@pytest.mark.parametrize("dtype", [torch.bool, torch.int64])
def test_masks(N, dtype, device):
    import gemma_triton_flash_attn_amd as gfa

    i = torch.arange(N)
    rows = [i < N, i < (N + 1) // 2, i >= N // 3, (i >= N // 4) & (i < 1 + N // 2), i < 0, i == N - 1]
    mask = torch.stack(rows).to(dtype)
    want = gfa.segments.from_padding_mask(mask)
    got = gfa.segments.from_padding_mask(mask.to(device))
    assert all(torch.equal(a.cpu(), b) for a, b in zip(got, want))
    if N >= 3:
        holed = mask.clone()
        holed[0, N // 2] = 0
        for m in (holed, holed[:1]):
            with pytest.raises(ValueError, match="contiguous"):
                gfa.segments.from_padding_mask(m.to(device))


@pytest.mark.parametrize("N", [70, 1500])
def test_adapter(N, device):
    """The adapter with position ids and masks: the same output as with tables built by hand, and a
    mask with holes still refused."""
    import gemma_triton_flash_attn_amd as gfa

    g = torch.Generator().manual_seed(N)
    q = torch.randn(2, N, 4, 256, generator=g).to(device, torch.bfloat16).transpose(1, 2)
    k, v = (torch.randn(2, N, 2, 256, generator=g).to(device, torch.bfloat16).transpose(1, 2) for _ in range(2))
    mod = SimpleNamespace(head_dim=256, is_causal=True)

    def want(segs):
        return gfa.attention_flash_gqa(q, k, v, causal=True, segments=segs).transpose(1, 2)

    plain, _ = gfa.triton_gqa_attention(mod, q, k, v, None, position_ids=torch.arange(N, device=device)[None])
    assert torch.equal(plain, want(None))
    pos = _positions("packed", 2, N)
    packed, _ = gfa.triton_gqa_attention(mod, q, k, v, None, position_ids=pos.to(device))
    assert torch.equal(packed, want(tuple(t.to(device) for t in gfa.segments.from_position_ids(pos))))
    mask = torch.arange(N)[None] < torch.tensor([[N], [N // 2]])
    padded, _ = gfa.triton_gqa_attention(mod, q, k, v, mask.to(device))
    assert torch.equal(padded, want(tuple(t.to(device) for t in gfa.segments.from_padding_mask(mask))))
    mask[1, 3] = False
    with pytest.raises(NotImplementedError, match="contiguous"):
        gfa.triton_gqa_attention(mod, q, k, v, mask.to(device))
    # three rows of ids for two rows of tokens: unpacked ids describe no segments, as before
    odd, _ = gfa.triton_gqa_attention(mod, q, k, v, None, position_ids=torch.arange(N, device=device).repeat(3, 1))
    assert torch.equal(odd, plain)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning", "ignore::DeprecationWarning")
@pytest.mark.parametrize("source", ["mask", "positions"])
def test_traced_tables_follow_the_batch(source, device):
    """Tables built inside a jit trace are part of it: they follow the batch that the trace is given,
    not the one it was traced with."""
    import gemma_triton_flash_attn_amd as gfa

    N = 80
    build = gfa.segments.from_padding_mask if source == "mask" else gfa.segments.from_position_ids
    i = torch.arange(N, device=device)[None]

    def batch(a, b):
        cut = torch.tensor([[a], [b]], device=device)
        return i < cut if source == "mask" else torch.where(i < cut, i, i - cut)

    def tables(t):
        return torch.stack(tuple(build(t)))

    traced = torch.jit.trace(tables, (batch(N, 30),), check_trace=False)
    for a, b in ((N, 30), (17, 60)):
        same = torch.equal(traced(batch(a, b)), tables(batch(a, b)))
        assert same, (a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,N,D,causal,window,same", [
    (8, 1, 333, 256, True, 512, True), (8, 1, 1024, 512, True, 0, True), (8, 1, 2500, 512, True, 0, True),
    (8, 1, 2048, 128, True, 0, True), (8, 4, 3073, 256, True, 0, True), (4, 1, 8200, 64, True, 0, True),
    (8, 1, 3000, 256, True, 512, True), (8, 8, 1700, 64, False, 0, False), (8, 4, 2100, 256, True, 0, False),
    (8, 4, 3072, 256, True, 0, False), (8, 1, 4096, 128, True, 0, False), (4, 1, 8192, 64, True, 0, False),
    (8, 4, 2048, 256, False, 0, False),
])
def test_ids_without_restarts(Hq, Hkv, N, D, causal, window, same, dtype, device):
    """Position ids of one run, which a model hands over in every layer, become a table of one segment
    per row. Outputs and gradients equal those without a table bit for bit where the same kernels
    run (``same``); where only a call without a table takes the small-grid forward, both outputs
    carry P rounded against their own reference maxima and their own rounding: with A = softmax
    |V| they differ by at most 2 u (A + |O|), u = 2^-8 in bf16 and 2^-11 in fp16, plus fp32 sums
    (1e-4)."""
    import gemma_triton_flash_attn_amd as gfa

    print(f"case {Hq}:{Hkv} N={N} D={D} causal={causal} window={window} {dtype}", flush=True)
    g = torch.Generator(device=device).manual_seed(N)
    q, k, v, do = (torch.randn(1, N, h, D, generator=g, device=device).to(dtype).transpose(1, 2)
                   for h in (Hq, Hkv, Hkv, Hq))
    mod = SimpleNamespace(head_dim=D, is_causal=causal)
    kw = dict(sliding_window=window or None, position_ids=torch.arange(N, device=device)[None])
    with torch.no_grad():
        out = gfa.triton_gqa_attention(mod, q, k, v, None, **kw)[0].transpose(1, 2)
        plain = gfa.attention_flash_gqa(q, k, v, causal, window)
        one = gfa.segments.from_lengths([N], N, device=device)
        assert torch.equal(out, gfa.attention_flash_gqa(q, k, v, causal, window, segments=one))
        if not same:
            a = gfa.attention_flash_gqa(q, k, v.abs(), causal, window)
            u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
            assert bool(((out.float() - plain.float()).abs() <= 2 * u * (a.float() + plain.float().abs()) + 1e-4).all())
            return
    assert torch.equal(out, plain)
    grads = []
    for ids in (True, False):
        t = [x.detach().requires_grad_(True) for x in (q, k, v)]
        o = (gfa.triton_gqa_attention(mod, *t, None, **kw)[0].transpose(1, 2) if ids
             else gfa.flash_attn_gqa_train(*t, causal, window))
        grads.append(torch.autograd.grad(o, t, do))
    assert all(torch.equal(a, b) for a, b in zip(*grads))


def test_default_device(device):
    """Under a default device (torch.set_default_device, torch.device as a context), which puts tensors made
    without a device on the GPU, tables and calls are the same and take the same path."""
    import gemma_triton_flash_attn_amd as gfa
    from gemma_triton_flash_attn_amd import _lib

    N = 100
    g = torch.Generator().manual_seed(1)
    q = torch.randn(2, 4, N, 64, generator=g).to(device, torch.bfloat16)
    k, v = (torch.randn(2, 2, N, 64, generator=g).to(device, torch.bfloat16) for _ in range(2))
    mod = SimpleNamespace(head_dim=64, is_causal=True)
    mask = (torch.arange(N)[None] < torch.tensor([[N], [40]])).to(device)
    pos = _positions("packed", 2, N).to(device)

    def calls():
        assert _lib.plain_setting()
        with torch.no_grad():
            out = [gfa.triton_gqa_attention(mod, q, k, v, mask)[0],
                   gfa.triton_gqa_attention(mod, q, k, v, None, position_ids=pos)[0],
                   *gfa.segments.from_padding_mask(mask), *gfa.segments.from_position_ids(pos)]
        t = [x.detach().requires_grad_(True) for x in (q, k, v)]
        return out + list(torch.autograd.grad(gfa.triton_gqa_attention(mod, *t, mask)[0].sum(), t))

    want = calls()
    with torch.device(device):
        assert all(torch.equal(a, b) for a, b in zip(calls(), want))
