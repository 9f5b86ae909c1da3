"""Top-k routing and expert-sorted dispatch: the harness around the grouped INT4
GEMM (kernels.moe_grouped). Same conventions as the reference:

- route_topk: softmax in fp32 over router logits, top-k, renormalised
  (train/model.py:158-162);
- sort_by_expert: stable sort of the T*k (token, slot) assignments by expert,
  per-expert counts and the inverse permutation (kernels/moe_routing.py:116-130);
- gather_rows: out[i] = x[idx[i]] (kernels/moe_routing.py:89-97).

- combine_rows: out[t] = sum_k w[t, k] * expert_out[pos[t, k]], one gfx950 block per
  output row, no atomics (kernels/moe_routing.py:52-76, 100-113);
- combine_partials: the same over the fp32 partial products of a K-split expert GEMM;
- moe_dispatch_combine: the routed MoE forward (kernels/moe_routing.py:133-153). When
  the experts are SwiGLU MLPs whose projections are INT4 QuantLinear with stacked
  buffers (serve.quantize.quantize_model stacks them), the per-expert loop becomes two
  grouped launches and the combine (kernels.moe_grouped.int4_expert_mlp_combine);
  otherwise each expert module runs on its segment as in the reference.

sort and gather are index bookkeeping on the device (torch ops).
"""

from __future__ import annotations

import torch

import kernels
from kernels._hip import dt_code, ld, plain, require_hip, stream


_ROUTE_DT = (torch.float32, torch.float16, torch.bfloat16)


def route_topk(logits: torch.Tensor, k: int):
    """(weights [T, k] fp32, experts [T, k] int64)."""
    if (plain(logits) and logits.dim() == 2 and logits.dtype in _ROUTE_DT and logits.stride(1) == 1
            and 0 < k <= min(logits.shape[1], kernels.ROUTE_MAX_TOP) and logits.shape[1] <= kernels.ROUTE_MAX_EXPERTS
            and logits.stride(0) >= logits.shape[1]):
        T, E = logits.shape
        weights = torch.empty(T, k, dtype=torch.float32, device=logits.device)
        experts = torch.empty(T, k, dtype=torch.int64, device=logits.device)
        kernels.check(kernels.lib().mlsx_route_topk(
            logits.data_ptr(), dt_code(logits.dtype, "route_topk"), logits.stride(0), T, E, k, weights.data_ptr(),
            experts.data_ptr(), stream(logits.device)), "route_topk")
        return weights, experts
    probs = torch.softmax(logits.float(), dim=-1)
    weights, experts = torch.topk(probs, k, dim=-1)
    weights = weights / weights.sum(dim=-1, keepdim=True)
    return weights, experts


def sort_by_expert(experts_idx: torch.Tensor, n_experts: int):
    """(token_of_slot [T*k], counts [E], pos [T, k]) for expert-contiguous dispatch."""
    T, k = experts_idx.shape
    flat = experts_idx.reshape(-1)
    order = torch.argsort(flat, stable=True)
    counts = torch.bincount(flat, minlength=n_experts)
    pos = torch.empty_like(order)
    pos[order] = torch.arange(T * k, device=flat.device)
    return order // k, counts, pos.reshape(T, k)


class _Route:
    """sort_by_expert in one launch, as the grouped kernels take it: token_of_slot (int32), the
    segment offsets (int32 [E + 1]) and pos (int64 [T, k]). check() raises for expert ids outside
    [0, E), which the kernel leaves out; it waits for that launch alone, so the caller
    enqueues the layer's GEMMs first."""

    @staticmethod
    def takes(experts_idx: torch.Tensor, n_experts: int) -> bool:
        return (plain(experts_idx) and experts_idx.dim() == 2 and experts_idx.dtype in (torch.int64, torch.int32)
                and 0 < experts_idx.numel() <= kernels.ROUTE_MAX and 0 < n_experts <= kernels.ROUTE_MAX_EXPERTS)

    def __init__(self, experts_idx: torch.Tensor, n_experts: int):
        dev = experts_idx.device
        idx = experts_idx.to(torch.int64).contiguous()
        n = idx.numel()
        ints = torch.empty(n + n_experts + 1, dtype=torch.int32, device=dev)
        self.token_of_slot, self.seg_off = ints[:n], ints[n:]
        self.pos = torch.empty(idx.shape, dtype=torch.int64, device=dev)
        # (the host allocator does not know of the launch that writes it: wait() before it goes)
        self.bad = torch.empty(1, dtype=torch.int32, device="cpu", pin_memory=True)
        kernels.check(kernels.lib().mlsx_route_sort(
            idx.data_ptr(), n, idx.shape[1], n_experts, self.token_of_slot.data_ptr(), self.seg_off.data_ptr(),
            self.pos.data_ptr(), self.bad.data_ptr(), stream(dev)), "moe_dispatch_combine")
        self.done = torch.cuda.Event()
        self.done.record(torch.cuda.current_stream(dev))
        self.n_experts = n_experts

    def wait(self) -> None:
        self.done.synchronize()

    def check(self) -> None:
        self.wait()
        bad = int(self.bad)
        if bad == 2:
            raise RuntimeError("moe_dispatch_combine: negative expert index")
        if bad:
            raise ValueError(f"moe_dispatch_combine: expert index past the {self.n_experts} experts")


def gather_rows(x: torch.Tensor, idx: torch.Tensor) -> torch.Tensor:
    return x.index_select(0, idx.to(torch.int64))


def _combine_dt(dtype: torch.dtype, what: str) -> int:
    """dtype code of a combine operand: the three GEMM dtypes and fp64."""
    return kernels.MLS_F64 if dtype == torch.float64 else dt_code(dtype, what)


def combine_rows(expert_out: torch.Tensor, weights: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """out[t] = sum_k weights[t, k] * expert_out[pos[t, k]], output in expert_out's dtype,
    accumulated in fp32, or in fp64 when expert_out is fp64 (the reference's ACC64, which
    its fp64 gradcheck relies on; kernels/moe_routing.py:54-72, 100-113)."""
    dev = require_hip("combine_rows", expert_out, weights, pos)
    T, K = pos.shape
    D = expert_out.shape[1]
    x = expert_out if expert_out.stride(1) == 1 else expert_out.contiguous()
    w = weights.contiguous()
    p = pos.to(torch.int64).contiguous()
    out = torch.empty(T, D, dtype=x.dtype, device=dev)
    kernels.check(kernels.lib().mls_moe_combine(
        x.data_ptr(), _combine_dt(x.dtype, "combine_rows"), ld(x), x.shape[0], 1, 0, w.data_ptr(),
        _combine_dt(w.dtype, "combine_rows weights"), p.data_ptr(), T, K, out.data_ptr(),
        _combine_dt(out.dtype, "combine_rows"), ld(out), D, stream(dev)), "combine_rows")
    return out


def combine_partials(partials: torch.Tensor, weights: torch.Tensor, pos: torch.Tensor,
                     out_dtype: torch.dtype) -> torch.Tensor:
    """combine_rows over the fp32 partial products [splits, rows, D] of a K-split expert
    GEMM: out[t] = sum_k weights[t, k] * sum_p partials[p, pos[t, k]], in out_dtype."""
    dev = require_hip("combine_partials", partials, weights, pos)
    S, R, D = partials.shape
    T, K = pos.shape
    x = partials.contiguous()
    w = weights.contiguous()
    p = pos.to(torch.int64).contiguous()
    out = torch.empty(T, D, dtype=out_dtype, device=dev)
    kernels.check(kernels.lib().mls_moe_combine(
        x.data_ptr(), dt_code(x.dtype, "combine_partials"), D, R, S, R * D, w.data_ptr(),
        dt_code(w.dtype, "combine_partials weights"), p.data_ptr(), T, K, out.data_ptr(),
        dt_code(out_dtype, "combine_partials"), ld(out), D, stream(dev)), "combine_partials")
    return out


def moe_dispatch_combine(flat: torch.Tensor, weights: torch.Tensor, experts_idx: torch.Tensor,
                         expert_modules) -> torch.Tensor:
    """Routed MoE forward (kernels/moe_routing.py:133-153): sort the (token, slot)
    assignments by expert, gather the rows, run every expert on its contiguous segment,
    combine weighted by the router. flat [T, D], weights [T, k], experts_idx [T, k]."""
    from kernels.moe_grouped import int4_expert_mlp_combine, segment_offsets
    from serve.quantize import stacked_int4_experts

    n_experts = len(expert_modules)
    st = stacked_int4_experts(expert_modules)
    quantized = st is not None and flat.dtype in (torch.bfloat16, torch.float16)
    if quantized and _Route.takes(experts_idx, n_experts):
        route = _Route(experts_idx, n_experts)
        try:
            out = int4_expert_mlp_combine(flat, route.seg_off, st["w_gate"][0], st["w_gate"][1], st["w_up"][0],
                                          st["w_up"][1], st["w_down"][0], st["w_down"][1], st["group_size"], weights,
                                          route.pos, a_rows=route.token_of_slot)
        except BaseException:
            route.wait()
            raise
        route.check()
        return out
    token_of_slot, counts, pos = sort_by_expert(experts_idx, n_experts)
    if quantized:
        # the gather runs inside the gate/up kernel's activation load (a_rows)
        return int4_expert_mlp_combine(flat, segment_offsets(counts), st["w_gate"][0], st["w_gate"][1],
                                       st["w_up"][0], st["w_up"][1], st["w_down"][0], st["w_down"][1],
                                       st["group_size"], weights, pos, a_rows=token_of_slot)
    dispatched = gather_rows(flat, token_of_slot)
    expert_out = torch.empty_like(dispatched)
    start = 0
    for e, cnt in enumerate(counts.tolist()):
        if cnt:
            expert_out[start:start + cnt] = expert_modules[e](dispatched[start:start + cnt])
        start += cnt
    return combine_rows(expert_out, weights, pos)
