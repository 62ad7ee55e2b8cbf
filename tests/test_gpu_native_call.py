"""The C++ host path (csrc/gfa_torch.cpp) against the Python autograd function it stands in for: the same
kernels on the same arguments, so outputs and gradients are equal bit for bit, and the same behaviour
with saved-tensor hooks, checkpointing, function transforms, forward mode, streams and errors."""
from __future__ import annotations

import threading
import time
from types import SimpleNamespace

import pytest
import torch

from conftest import make_inputs

pytestmark = pytest.mark.gpu


def _python(q, k, v, causal=False, slide_size=0, scale=None, segments=None, softcap=None, dropout_p=0.0):
    import gemma_triton_flash_attn_amd as gfa

    return gfa.FlashAttnGQAFunction.apply(q, k, v, causal, slide_size, scale, segments, softcap, dropout_p)


def _both(q, k, v, do, **kw):
    import gemma_triton_flash_attn_amd as gfa

    res = []
    for fn in (gfa.flash_attn_gqa_train, _python):
        torch.manual_seed(11)  # dropout seeds come from torch's generator
        qq, kk, vv = (t.detach().requires_grad_(True) for t in (q, k, v))
        o = fn(qq, kk, vv, **kw)
        res.append((o, *torch.autograd.grad(o, (qq, kk, vv), do)))
    return res


def _equal(q, k, v, do, **kw):
    (o, *g), (op, *gp) = _both(q, k, v, do, **kw)
    assert "FlashAttnGQAFunction" not in o.grad_fn.name() and "FlashAttnGQAFunction" in op.grad_fn.name()
    for a, b in zip((o, *g), (op, *gp)):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,N,causal,window", [(512, 70, True, 0), (256, 300, True, 64), (128, 33, False, 0),
                                               (64, 200, True, 0)])
@pytest.mark.parametrize("feature", ["plain", "segments", "softcap", "dropout", "scale"])
def test_equals_python_function(D, N, causal, window, dtype, feature, device):
    import gemma_triton_flash_attn_amd as gfa

    kw = {"plain": {}, "segments": {}, "softcap": {"softcap": 20.0}, "dropout": {"dropout_p": 0.25},
          "scale": {"scale": 0.07}}[feature]
    if feature == "segments":
        kw = {"segments": gfa.segments.from_lengths([N, N // 2], N, device=device)}
    q, k, v, do = make_inputs(2, 4, 2, N, D, dtype, device, seed=N, layout="bnhd" if D % 512 else "bhnd")
    _equal(q, k, v, do, causal=causal, slide_size=window, **kw)


def test_layouts(device):
    """Layouts the ABI addresses in place, and ones it copies: rows that are no multiple of 8 elements,
    a broadcast or sliced dO, another dtype of dO."""
    N, D = 50, 128
    q, k, v, do = make_inputs(2, 4, 2, N, D, torch.bfloat16, device, seed=3)
    _equal(q, k, v, do[:, :1, :1, :].expand_as(q), causal=True)
    _equal(q, k, v, do.transpose(2, 3).contiguous().transpose(2, 3), causal=True)
    wide = torch.zeros(2, 4, N, D + 4, dtype=torch.bfloat16, device=device)
    wide[..., :D] = q
    _equal(wide[..., :D], k, v, do, causal=True)
    _equal(q[:1].expand(2, 4, N, D), k, v, do, causal=False)
    big = torch.zeros(2, 4, 2 * N, D, dtype=torch.bfloat16, device=device)
    big[:, :, ::2] = q
    _equal(big[:, :, ::2], k, v, do, causal=True, slide_size=7)


def test_inference_entry_points(device):
    import gemma_triton_flash_attn_amd as gfa

    q, k, v, _ = make_inputs(2, 4, 2, 90, 256, torch.bfloat16, device, seed=5, layout="bnhd")
    want = _python(q, k, v, True, 40)
    assert torch.equal(gfa.attention_flash_gqa(q, k, v, True, 40), want)
    assert not gfa.attention_flash_gqa(q.clone().requires_grad_(True), k, v, True, 40).requires_grad
    mod = SimpleNamespace(head_dim=256, is_causal=True)
    out, _ = gfa.triton_gqa_attention(mod, q, k, v, None, sliding_window=40)
    assert torch.equal(out, want.transpose(1, 2)) and out.is_contiguous()
    # the adapter under autograd: the op's gradients
    grads = []
    for fn in (lambda a, b, c: gfa.triton_gqa_attention(mod, a, b, c, None, sliding_window=40)[0],
               lambda a, b, c: gfa.flash_attn_gqa_op(a, b, c, True, 40, scale=256 ** -0.5).transpose(1, 2)):
        t = [x.detach().requires_grad_(True) for x in (q, k, v)]
        o = fn(*t)
        grads.append(torch.autograd.grad(o, t, torch.ones_like(o)))
    assert all(torch.equal(a, b) for a, b in zip(*grads))
    # dropout in a module that trains without gradients
    torch.manual_seed(2)
    a, _ = gfa.triton_gqa_attention(mod, q, k, v, None, dropout=0.3)
    torch.manual_seed(2)
    assert torch.equal(a, _python(q, k, v, True, 0, 256 ** -0.5, None, None, 0.3).transpose(1, 2))


def test_hooks_checkpoint_and_transforms(device):
    import gemma_triton_flash_attn_amd as gfa
    from torch.utils.checkpoint import checkpoint

    q, k, v, do = make_inputs(1, 4, 2, 64, 128, torch.bfloat16, device, seed=6)
    _, want = _both(q, k, v, do, causal=True)
    packed = []
    t = [x.detach().requires_grad_(True) for x in (q, k, v)]
    with torch.autograd.graph.saved_tensors_hooks(lambda x: packed.append(x.shape) or x.cpu(), lambda x: x.to(device)):
        o = gfa.flash_attn_gqa_train(*t, True)
    assert len(packed) == 5  # q, k, v, O, LSE
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(o, t, do), want[1:]))
    for reentrant in (False, True):
        o = checkpoint(lambda a, b, c: gfa.flash_attn_gqa_train(a, b, c, True), *t, use_reentrant=reentrant)
        o.backward(do)
        assert all(torch.equal(x.grad, b) for x, b in zip(t, want[1:]))
        for x in t:
            x.grad = None
    # saved inputs changed in place before the backward are an error, as ever
    z = q * 1.0
    z.requires_grad_(True)
    y = z * 1.0
    o = gfa.flash_attn_gqa_train(y, k, v, True)
    y.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.backward(do)
    # function transforms and forward mode: refused, as by the Python function
    for fn in (gfa.flash_attn_gqa_train, _python):
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda a: fn(a, k, v, True).float().sum())(q)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(q, torch.ones_like(q))
            with pytest.raises((RuntimeError, NotImplementedError)):
                torch.autograd.forward_ad.unpack_dual(fn(dual, k, v, True))


def test_errors(device):
    import gemma_triton_flash_attn_amd as gfa
    from gemma_triton_flash_attn_amd import _lib

    q, k, v, do = make_inputs(1, 4, 2, 64, 128, torch.bfloat16, device, seed=7)
    with pytest.raises(_lib.GfaError, match="16-byte aligned") as e:  # contiguous but off by one element
        base = torch.zeros(q.numel() + 1, dtype=q.dtype, device=device)
        gfa.flash_attn_gqa_train(base[1:].view(q.shape), k, v, True)
    assert e.value.status == 1
    t = q.detach().requires_grad_(True)
    o = gfa.flash_attn_gqa_train(t, k, v, True)
    with pytest.raises(_lib.GfaError, match="dout is not 16-byte aligned") as e:  # raised on an engine thread
        o.backward(base[1:].view(q.shape))
    assert e.value.status == 1
    for bad, exc in ((dict(softcap=-1.0), ValueError), (dict(dropout_p=1.0), ValueError),
                     (dict(softcap=2.0, dropout_p=0.1), NotImplementedError), (dict(slide_size=-1), ValueError)):
        with pytest.raises(exc):
            gfa.flash_attn_gqa_train(q, k, v, True, **bad)
    with pytest.raises(TypeError):
        gfa.flash_attn_gqa_train(q.float(), k, v, True)
    with pytest.raises(ValueError, match="GPU tensors"):
        gfa.flash_attn_gqa_train(q.cpu(), k.cpu(), v.cpu(), True)


def test_streams_and_threads(device):
    """Calls on side streams from several threads at once, each forward and backward on its own."""
    import gemma_triton_flash_attn_amd as gfa

    cases, got = [], {}
    for i in range(4):
        q, k, v, do = make_inputs(1, 4, 2, 100 + 40 * i, 256, torch.bfloat16, device, seed=i)
        cases.append((q, k, v, do, _both(q, k, v, do, causal=True)[1]))
    torch.cuda.synchronize()

    def work(i):
        q, k, v, do, _ = cases[i]
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                t = [x.detach().requires_grad_(True) for x in (q, k, v)]
                o = gfa.flash_attn_gqa_train(*t, True)
                got[i] = (o, *torch.autograd.grad(o, t, do))
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for i, (*_, want) in enumerate(cases):
        assert all(torch.equal(a, b) for a, b in zip(got[i], want))


def test_other_threads_run_during_a_call(device):
    """The interpreter lock is free while a call allocates (here 2 GiB from the driver) and launches:
    another Python thread runs in the middle half of the call."""
    import gemma_triton_flash_attn_amd as gfa

    q = torch.zeros(1, 64, 131072, 128, dtype=torch.bfloat16, device=device)
    k = q[:, :1]
    for call in (lambda: gfa.attention_flash_gqa(q, k, k, True, 64), lambda: gfa.flash_attn_gqa_train(q, k, k, True, 64)):
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        ticks, stop = [], threading.Event()

        def spin():
            while not stop.is_set():
                ticks.append(time.perf_counter())

        th = threading.Thread(target=spin)
        th.start()
        time.sleep(0.01)
        t0 = time.perf_counter()
        call()
        t1 = time.perf_counter()
        stop.set()
        th.join()
        quarter = (t1 - t0) / 4
        assert any(t0 + quarter < t < t1 - quarter for t in ticks), t1 - t0
