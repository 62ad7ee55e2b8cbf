"""Gradients through the transformers adapter's C++ node against the registered op gfa::attn_fwd that
the adapter is made of wherever it is traced or compiled: the same gradients, and the same answer to
what a plain backward is not (second order, batched gradients, dispatch modes, compiled autograd)."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from conftest import make_inputs

pytestmark = pytest.mark.gpu

N, D = 96, 128
MOD = SimpleNamespace(head_dim=D, is_causal=True)
FEATURES = ["plain", "packed", "softcap", "dropout"]


def _inputs(device, seed=1):
    q, k, v, do = make_inputs(1, 4, 2, N, D, torch.bfloat16, device, seed=seed, layout="bnhd")
    return [t.requires_grad_(True) for t in (q, k, v)], do.transpose(1, 2)


def _kw(feature, device):
    pos = torch.arange(N, device=device)
    return {"plain": {}, "packed": {"position_ids": torch.where(pos < 40, pos, pos - 40)[None]},
            "softcap": {"softcap": 20.0}, "dropout": {"dropout": 0.2}}[feature]


def _adapter(t, kw):
    import gemma_triton_flash_attn_amd as gfa

    torch.manual_seed(5)  # dropout seeds come from torch's generator
    return gfa.triton_gqa_attention(MOD, *t, None, **kw)[0]


def _op(t, kw):
    import gemma_triton_flash_attn_amd as gfa

    torch.manual_seed(5)
    kw = dict(kw)
    pos = kw.pop("position_ids", None)
    segs = None if pos is None else gfa.segments.from_position_ids(pos)
    return gfa.flash_attn_gqa_op(*t, True, segments=segs, softcap=kw.get("softcap"),
                                 dropout_p=kw.get("dropout", 0.0)).transpose(1, 2)


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("feature", FEATURES)
def test_second_order_refused(feature, device):
    """create_graph gives the first-order gradients; differentiating them again is an error, as for
    the op (no formula), never a result without the second-order terms."""
    t, do = _inputs(device)
    kw = _kw(feature, device)
    want = torch.autograd.grad(_op(t, kw), t, do)
    for fn in (_adapter, _op):
        got = torch.autograd.grad(fn(t, kw), t, do, create_graph=True)
        assert all(torch.equal(a, b) and a.requires_grad for a, b in zip(got, want))
        with pytest.raises(RuntimeError, match="no autograd formula"):
            (got[0].float().square().sum() + t[0].float().sum()).backward()
        assert all(x.grad is None for x in t)


@pytest.mark.parametrize("feature", FEATURES)
def test_batched_gradients(feature, device):
    t, do = _inputs(device)
    kw = _kw(feature, device)
    dos = torch.stack([do, 2 * do, do.flip(1)])
    got = torch.autograd.grad(_adapter(t, kw), t, dos, is_grads_batched=True)
    for i in range(3):
        want = torch.autograd.grad(_op(t, kw), t, dos[i].contiguous())
        assert all(torch.equal(a[i], b) for a, b in zip(got, want))


@pytest.mark.parametrize("feature", FEATURES)
def test_dispatch_mode_in_backward(feature, device):
    t, do = _inputs(device)
    kw = _kw(feature, device)
    out = _adapter(t, kw)
    with _Seen() as seen:
        got = torch.autograd.grad(out, t, do)
    assert "gfa.attn_bwd.default" in seen.names
    assert all(torch.equal(a, b) for a, b in zip(got, torch.autograd.grad(_op(t, kw), t, do)))


@pytest.mark.parametrize("feature", FEATURES)
@pytest.mark.parametrize("entry", ["adapter", "train"])
def test_compiled_autograd(entry, feature, device):
    """Compiled autograd takes the node into one graph, and its graph serves other inputs and other
    dropout seeds."""
    import gemma_triton_flash_attn_amd as gfa

    kw = _kw(feature, device)
    torch._dynamo.reset()
    for seed in (1, 2, 3):
        t, do = _inputs(device, seed)

        def out():
            torch.manual_seed(seed)
            if entry == "adapter":
                return gfa.triton_gqa_attention(MOD, *t, None, **kw)[0]
            segs = gfa.segments.from_position_ids(kw["position_ids"]) if feature == "packed" else None
            return gfa.flash_attn_gqa_train(*t, True, segments=segs, softcap=kw.get("softcap"),
                                            dropout_p=kw.get("dropout", 0.0)).transpose(1, 2)

        want = torch.autograd.grad(out(), t, do)
        o = out()
        with torch._dynamo.compiled_autograd._enable(torch.compile(backend="aot_eager", fullgraph=True)):
            o.backward(do)
        assert all(torch.equal(x.grad, b) for x, b in zip(t, want))


class _SeenFunctions(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("grad", [True, False])
def test_function_modes_and_profiler(grad, device):
    """A torch-function mode sees the op, and a profiler lists it by name, with and without gradients."""
    t, do = _inputs(device)
    with torch.set_grad_enabled(grad):
        with _SeenFunctions() as seen:
            out = _adapter(t, {})
        assert any("gfa.attn_fwd" in n for n in seen.names)
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
            again = _adapter(t, {})
            if grad:
                again.backward(do)
    assert torch.equal(out, again)
    names = {e.key for e in prof.key_averages()}
    assert "gfa::attn_fwd" in names and ("gfa::attn_bwd" in names) == grad


def test_negated_views_and_zero_gradients(device):
    """Inputs and gradients whose values are not what lies in their memory: views that negate on reading,
    and a zero gradient without memory."""
    t, do = _inputs(device)
    plain = [x.detach() for x in t]
    neg = torch._neg_view(-plain[0])
    assert neg.is_neg() and torch.equal(_adapter([neg, *plain[1:]], {}), _adapter(plain, {}))
    leaves = [neg.requires_grad_(True), *t[1:]]
    out, want = _adapter(leaves, {}), torch.autograd.grad(_op(t, {}), t, do)
    got = torch.autograd.grad(out, leaves, torch._neg_view(-do))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    zero = torch._efficientzerotensor(do.shape, dtype=do.dtype, device=device)
    assert all(not x.any() for x in torch.autograd.grad(_adapter(t, {}), t, zero))
