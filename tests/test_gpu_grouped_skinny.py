"""The grouped INT4 GEMMs for few rows an expert (csrc/grouped_skinny.hip) against float64.

Bounds: a group's products are summed with an offset of 136 (bf16) or 1032 (fp16) a weight that
is taken off afterwards, so an fp32 sum's error is that of terms up to 1032 |x| s: K 2^-24 of
their root sum of squares covers it at these K; a 16-bit output rounds once (2^-8, 2^-11)."""

from __future__ import annotations

import pytest
import torch

from kernels.moe_grouped import int4_grouped_gate_up, int4_grouped_matmul, int4_grouped_matmul_partial, segment_offsets

pytestmark = pytest.mark.gpu

ROUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
OFF = {torch.bfloat16: 136.0, torch.float16: 1032.0}


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
    return K * 2.0 ** -24 * OFF[x.dtype] * x.double().square().sum(1, keepdim=True).sqrt() * float(s.max())


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
