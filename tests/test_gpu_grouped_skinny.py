"""The grouped INT4 GEMMs for few rows an expert (csrc/grouped_skinny.hip) against float64.

Bounds: weights are exact, so an fp32 sum's error is that of K terms up to 8 |x| s: K 2^-24 of their
root sum of squares covers it at these K; a 16-bit output rounds once (2^-8, 2^-11). And against
the chunk kernel (csrc/gemm_grouped.hip), which takes calls of more rows: the same bits."""

from __future__ import annotations

import pytest
import torch

import kernels
from kernels.moe_grouped import int4_grouped_gate_up, int4_grouped_matmul, int4_grouped_matmul_partial, segment_offsets

pytestmark = pytest.mark.gpu

ROUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _weights(dev, E, N, K, group, sdt, seed):
    g = torch.Generator().manual_seed(seed)
    q = torch.randint(0, 256, (E, N, K // 2), generator=g, dtype=torch.uint8)
    s = (torch.rand(E, N, K // group, generator=g) * 0.02 + 0.01).to(sdt)
    v = torch.stack([q & 15, q >> 4], 3).reshape(E, N, K).double() - 8
    w = (v.reshape(E, N, K // group, group) * s.double()[..., None]).reshape(E, N, K)
    return q.to(dev), s.to(dev), w.to(dev)


def _rows(dev, counts, K, dtype, seed):
    return torch.randn(sum(counts), K, generator=torch.Generator().manual_seed(seed)).to(dtype).to(dev)


def _product(x, w, counts):
    out, at = [], 0
    for e, c in enumerate(counts):
        out.append(x[at:at + c].double() @ w[e].t())
        at += c
    return torch.cat(out)


def _slack(x, s, K):
    return K * 2.0 ** -24 * 8.0 * x.double().square().sum(1, keepdim=True).sqrt() * float(s.max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,N,K,group,sdt", [
    ([1], 8, 128, 128, torch.float16), ([3, 0, 5, 1], 100, 256, 64, torch.float32),
    ([0, 17, 1, 2], 64, 384, 128, torch.float16),     # a segment of two row tiles, one at a time
    ([40, 1, 20, 3], 130, 1024, 256, torch.float16),  # several passes of two row tiles
    ([7, 8, 0, 1], 65, 2048, 64, torch.float16), ([2, 2], 4096, 4096, 128, torch.float16),
])
def test_grouped(dev, counts, N, K, group, sdt, dtype):
    q, s, w = _weights(dev, len(counts), N, K, group, sdt, N + K)
    x = _rows(dev, counts, K, dtype, K)
    cnt = torch.tensor(counts, device=dev)
    want, slack = _product(x, w, counts), _slack(x, s, K)
    y = int4_grouped_matmul(x, q, s, cnt, group)
    assert float(((y.double() - want).abs() - ROUND[dtype] * want.abs() - slack).max()) <= 0
    if K // 2 % 128 == 0 and K // 2 % group == 0:
        part = int4_grouped_matmul_partial(x, q, s, cnt, group, 2)
        halves = torch.stack([_product(x[:, h], w[:, :, h], counts) for h in (slice(0, K // 2), slice(K // 2, K))])
        assert float(((part.double() - halves).abs() - slack).max()) <= 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,H,K,group", [([3, 0, 5, 1], 70, 256, 64), ([20, 1, 2, 2], 33, 512, 128), ([1, 1], 1024, 2048, 128)])
def test_gate_up_with_gather(dev, counts, H, K, group, dtype):
    """silu(gate) * up of gathered rows; an index outside the matrix reads zeros."""
    E, M, T = len(counts), sum(counts), 12
    (qg, sg, wg), (qu, su, wu) = (_weights(dev, E, H, K, group, torch.float16, 7 + i) for i in range(2))
    x = _rows(dev, [T], K, dtype, 3)
    idx = torch.randint(0, T, (M,), generator=torch.Generator().manual_seed(M)).to(dev)
    idx[0], idx[M - 1] = T, -1
    xs = torch.where(((idx >= 0) & (idx < T))[:, None], x[idx.clamp(0, T - 1)], torch.zeros_like(x[:1]))
    h = int4_grouped_gate_up(x, qg, sg, qu, su, segment_offsets(torch.tensor(counts, device=dev)), group, a_rows=idx)
    g, u = _product(xs, wg, counts), _product(xs, wu, counts)
    want, d = g * torch.sigmoid(g) * u, _slack(xs, sg, K)
    # |silu'| <= 1.1 and silu in fp32 with the device's exp: 2^-20 of the result
    bound = (ROUND[dtype] + 2.0 ** -20) * want.abs() + 1.1 * d * u.abs() + g.abs() * d + d * d
    assert float(((h.double() - want).abs() - bound).max()) <= 0


def _takes(M, E, K, group, splits=1):
    return kernels.lib().mlsx_int4_grouped_few_rows(M, E, K, group, splits) == 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts,N,K,group,sdt,splits", [
    ([5, 0, 16, 2], 150, 384, 128, torch.float32, 3),    # an edge of columns, three steps
    ([1, 9], 96, 2048, 64, torch.float16, 2), ([3, 1], 64, 896, 64, torch.float32, 1),
    ([11, 14, 8, 15], 5632, 2048, 128, torch.float16, 4),   # two row tiles, blocks few and ranges long
    ([9, 40, 0, 7, 12, 3, 13, 12], 3072, 2048, 128, torch.float16, 1), ([30, 1], 128, 2048, 512, torch.float32, 1),
    ([2] * 8, 512, 2048, 256, torch.float16, 2), ([2, 2], 64, 14336, 64, torch.float32, 1),  # 224 groups' scales in LDS
])
def test_rows_are_the_chunk_kernels(dev, counts, N, K, group, sdt, splits, dtype):
    """A row gets the same bits here and in a call of so many rows that the chunk kernel takes it,
    with infinities and NaN among them: plain, in partial products, and gate/up."""
    E, M = len(counts), sum(counts)
    extra = 16 * E + 1  # more rows for expert 0, behind its own
    assert _takes(M, E, K, group, splits) and not _takes(M + extra, E, K, group, splits)
    (q, s, _), (qu, su, _) = (_weights(dev, E, N, K, group, sdt, K + i) for i in range(2))
    x = _rows(dev, counts, K, dtype, N)
    x[0, 3], x[M // 2, K - 1], x[M - 1, K // 2] = float("inf"), float("-inf"), float("nan")
    big = torch.cat([x[:counts[0]], _rows(dev, [extra], K, dtype, 1), x[counts[0]:]])
    few, many = torch.tensor(counts, device=dev), torch.tensor([counts[0] + extra, *counts[1:]], device=dev)

    def same(a, b):
        b = torch.cat([b[..., :counts[0], :], b[..., counts[0] + extra:, :]], -2)
        bad = torch.isnan(a)
        assert a.shape == b.shape and bad.any() and not bad.all()
        assert torch.equal(bad, torch.isnan(b)) and torch.equal(a[~bad], b[~bad])

    same(int4_grouped_matmul(x, q, s, few, group), int4_grouped_matmul(big, q, s, many, group))
    same(int4_grouped_gate_up(x, q, s, qu, su, few, group), int4_grouped_gate_up(big, q, s, qu, su, many, group))
    same(int4_grouped_matmul_partial(x, q, s, few, group, splits),
         int4_grouped_matmul_partial(big, q, s, many, group, splits))


def test_infinities_as_fp32(dev):
    """fp32 scales (no scale table): an infinite x gives what fp32 arithmetic gives, +-inf, and NaN
    only at weights of zero."""
    q, s, w = _weights(dev, 2, 200, 512, 128, torch.float32, 1)
    x = _rows(dev, [2, 3], 512, torch.bfloat16, 2)
    x[1, 70], x[3, 511] = float("inf"), float("-inf")
    y = int4_grouped_matmul(x, q, s, torch.tensor([2, 3], device=dev), 128).float()
    want = torch.cat([x[:2].float() @ w[0].float().t(), x[2:].float() @ w[1].float().t()])
    inf = torch.isinf(want)
    assert inf.any() and torch.equal(y[inf], want[inf]) and torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.isfinite(y[torch.isfinite(want)]).all()
