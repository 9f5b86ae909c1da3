"""The routing kernels (csrc/moe_route.hip) against the torch op sequences they replace."""

from __future__ import annotations

import pytest
import torch

import kernels
from kernels._hip import plain
from kernels.moe_routing import _Route, combine_rows, route_topk, sort_by_expert

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,E,k", [(1, 1, 1), (3, 8, 2), (5, 64, 8), (7, 65, 3), (513, 256, 8)])
def test_topk(dev, T, E, k, dtype):
    """Same experts as torch's topk (ties aside: the logits are distinct), weights within the
    rounding of one exp and two divisions (2^-20 relative)."""
    g = torch.Generator().manual_seed(T * E)
    logits = (torch.stack([torch.randperm(E, generator=g) for _ in range(T)]).float() / 32 - 2).to(dtype).to(dev)
    w, e = route_topk(logits, k)
    probs = torch.softmax(logits.double(), dim=-1)
    want, idx = torch.topk(probs, k, dim=-1)
    assert torch.equal(e, idx) and e.dtype == torch.int64 and w.dtype == torch.float32
    want = want / want.sum(-1, keepdim=True)
    assert float(((w.double() - want).abs() - 2.0 ** -20 * want).max()) <= 0


def test_topk_ties_infinities_and_strides(dev):
    x = torch.full((4, 9), float("-inf"), device=dev)
    x[0] = 1.0                                   # all equal: the lowest experts, equal weights
    x[1, 5], x[1, 2] = 3.0, 3.0
    x[2, 7] = 0.0                                # one finite logit: weight 1, then zeros
    x[3] = torch.arange(9.0, device=dev)
    wide = torch.cat([x, x], 1)[:, :9]           # a row stride
    for t in (x, wide):
        w, e = route_topk(t, 3)
        assert e[0].tolist() == [0, 1, 2] and torch.allclose(w[0], torch.full((3,), 1 / 3, device=dev))
        assert e[1, :2].tolist() == [2, 5] and w[1].tolist() == [0.5, 0.5, 0.0]
        assert int(e[2, 0]) == 7 and w[2].tolist() == [1.0, 0.0, 0.0] and len(set(e[2].tolist())) == 3
        assert e[3].tolist() == [8, 7, 6]
    y = x.clone()
    y[3, 4] = float("nan")
    w, e = route_topk(y, 3)  # a NaN logit: NaN weights, as softmax gives, experts in range
    assert torch.isnan(w[3]).all() and int(e.min()) >= 0 and int(e.max()) < 9


def test_topk_keeps_gradients(dev):
    """Logits that need gradients, and transforms, take the differentiable torch ops."""
    x = torch.randn(6, 8, device=dev, requires_grad=True)
    w, _ = route_topk(x, 2)
    w[:, 0].sum().backward()
    assert x.grad is not None and x.grad.abs().sum() > 0
    _, t = torch.func.jvp(lambda v: route_topk(v, 2)[0], (x.detach(),), (torch.ones_like(x),))
    assert t.shape == (6, 2)
    assert torch.vmap(lambda v: route_topk(v, 2)[0])(x.detach().reshape(2, 3, 8)).shape == (2, 3, 2)


def test_traces_and_modes_see_the_torch_ops(dev):
    """Under a trace the result depends on the traced input (a kernel's would be a constant), and
    dispatch and function modes see topk; torch's default device alone changes nothing."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    a, b = (torch.randn(4, 8, generator=torch.Generator().manual_seed(i)).to(dev) for i in range(2))
    want = route_topk(b, 2)
    for traced in (torch.jit.trace(lambda t: route_topk(t, 2), a), make_fx(lambda t: route_topk(t, 2))(a),
                   make_fx(lambda t: route_topk(t, 2), pre_dispatch=True)(a)):
        w, e = traced(b)
        assert torch.equal(e, want[1]) and torch.allclose(w, want[0])
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    for mode in (Dispatch, Function):
        seen.clear()
        with mode():
            route_topk(a, 2)
        assert any("topk" in n for n in seen), seen
    with torch.device(dev):
        assert plain(a) and _Route.takes(want[1], 8)


@pytest.mark.parametrize("T,k,E", [(1, 1, 1), (1, 2, 8), (37, 2, 3), (512, 2, 8), (1025, 1, 256), (4096, 8, 64)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_sort(dev, T, k, E, dtype):
    idx = torch.randint(0, E, (T, k), generator=torch.Generator().manual_seed(T + E)).to(dtype).to(dev)
    assert _Route.takes(idx, E)
    r = _Route(idx, E)
    r.check()
    tok, counts, pos = sort_by_expert(idx.long(), E)
    assert torch.equal(r.token_of_slot.long(), tok) and torch.equal(r.pos, pos)
    assert torch.equal(r.seg_off[1:].long(), counts.cumsum(0)) and int(r.seg_off[0]) == 0


def test_sort_refuses_ids_outside(dev):
    idx = torch.tensor([[0, 9], [1, 2], [-1, 1]], device=dev)
    r = _Route(idx, 3)
    with pytest.raises(RuntimeError, match="negative"):
        r.check()
    assert r.seg_off.tolist() == [0, 1, 3, 4] and r.pos.tolist() == [[0, -1], [1, 3], [-1, 2]]
    assert r.token_of_slot.tolist() == [0, 1, 2, 1, -1, -1]
    with pytest.raises(ValueError, match="past the 3"):
        _Route(idx[:2], 3).check()
    assert not _Route.takes(torch.zeros(kernels.ROUTE_MAX + 1, 1, dtype=torch.int64, device=dev), 3)
    assert not _Route.takes(idx[:0], 3) and not _Route.takes(idx.float(), 3)


@pytest.mark.parametrize("T,D", [(1, 8), (3, 1000), (255, 4104), (256, 4096), (300, 20)])
def test_combine_columns_over_blocks(dev, T, D):
    """Every column is written once, whichever block owns it (fp32 sums of two products)."""
    g = torch.Generator().manual_seed(D)
    x, w = torch.randn(2 * T, D, generator=g).to(dev), torch.rand(T, 2, generator=g).to(dev)
    pos = torch.randperm(2 * T, generator=g).reshape(T, 2).to(dev)
    want = (x.double()[pos] * w.double()[:, :, None]).sum(1)
    assert float(((combine_rows(x, w, pos).double() - want).abs() - 2.0 ** -22 * (x.double()[pos].abs() * w[:, :, None]).sum(1)).max()) <= 0


def test_sort_under_a_default_device(dev):
    """The word that the kernel reports in is pinned host memory whatever torch's default device."""
    with torch.device(dev):
        r = _Route(torch.tensor([[1, 0], [2, 2]]), 3)
    r.check()
    assert r.bad.device.type == "cpu" and r.bad.is_pinned() and r.seg_off.tolist() == [0, 1, 2, 4]
