"""The K-split weight-only GEMMs (csrc/gemm_ksplit.hip) through int8_matmul / int4_matmul, at
the edges of their tiles, ranges and ragged K, against float64.

Bounds: 16-bit outputs round once (2^-9 bf16, 2^-12 fp16, of the value) on fp32 sums whose
error is below 2^-17 of the terms' root sum of squares at these K; fp32 outputs have that
error alone, plus 2^-16 of each term where x is taken as two bf16 parts."""

from __future__ import annotations

import pytest
import torch

import kernels
from kernels.dequant_matmul import int4_matmul, int8_matmul

pytestmark = pytest.mark.gpu

ROUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}


def _weights(dev, bits, N, K, group, sdt, seed):
    g = torch.Generator().manual_seed(seed)
    if bits == 8:
        q = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
        s = (torch.rand(N, generator=g) + 0.1).to(sdt)
        w = q.double() * s.double()[:, None]
    else:
        q = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8)
        s = (torch.rand(N, K // group, generator=g) + 0.1).to(sdt)
        v = torch.stack([q & 15, q >> 4], 2).reshape(N, K).double() - 8
        w = (v.reshape(N, K // group, group) * s.double()[:, :, None]).reshape(N, K)
    return q.to(dev), s.to(dev), w.to(dev)


def _run(bits, x, q, s, group):
    return int8_matmul(x, q, s) if bits == 8 else int4_matmul(x, q, s, group)


def _check(y, x, w, what, split=False):
    want, terms = x.double() @ w.t(), (x.double().square() @ w.square().t()).sqrt()
    bound = ROUND[x.dtype] * want.abs() + (2.0 ** -14 if split else 2.0 ** -17) * terms
    excess = float(((y.double() - want).abs() - bound).max())
    assert excess <= 0, f"{what}: worst excess {excess:.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bits,M,N,K,group", [
    (8, 65, 4102, 1376, 0), (8, 300, 4096, 1376, 0), (8, 129, 2056, 2720, 0), (8, 1149, 1336, 2720, 0),
    (8, 257, 1000, 4096, 0), (8, 5, 64, 20512, 0),
    (4, 17, 130, 64, 32), (4, 65, 260, 320, 32), (4, 65, 4102, 1376, 32), (4, 16, 4096, 11008, 32), (4, 333, 1024, 11008, 128),
    (4, 700, 520, 4096, 64), (4, 257, 1000, 2048, 256), (4, 2048, 512, 4096, 32),
])
def test_shapes(dev, bits, M, N, K, group, dtype):
    """Ragged rows, columns and K (a multiple of 32) with NaN beside the operand's rows: whatever
    a tile reads past K or M must not reach a result. (All but the smallest two INT4 sizes are
    ones the K-split kernels take: more rows than the skinny and medium kernels serve faster.)"""
    q, s, w = _weights(dev, bits, N, K, group, torch.float32 if M % 2 else torch.float16, K + M)
    pad = torch.full((M + 1, K + 32), float("nan"), device=dev, dtype=dtype)
    x = pad[:M, :K]
    x.copy_(torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(dtype))
    split = dtype == torch.float32 and K % 64 == 0 and (bits == 8 or group % 64 == 0)
    _check(_run(bits, x, q, s, group), x, w, f"int{bits} {M}x{N}x{K} g{group} {dtype}", split)


@pytest.mark.parametrize("M,N,K", [(1, 300, 11008), (2, 300, 11008), (16, 200, 4128)])
@pytest.mark.parametrize("bits", [4, 8])
def test_fp32_rows_past_the_register_kernels(dev, bits, M, N, K):
    """fp32 decode rows whose x does not fit the register GEMV's registers: three bf16 parts,
    which add up to x, so the result is as close to float64 as fp32 sums are."""
    q, s, w = _weights(dev, bits, N, K, 32, torch.float32, K)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(dev)
    _check(_run(bits, x, q, s, 32), x, w, f"int{bits} {M}x{N}x{K}", bits == 8 and M > 1 and K % 64 == 0)


@pytest.mark.parametrize("layout", ["transposed", "row_broadcast", "group_broadcast", "padded"])
def test_scale_strides(dev, layout):
    """Every scale layout that the general path takes (group and row strides of any size)."""
    M, N, K, group = 333, 264, 2048, 64
    q, s, _ = _weights(dev, 4, N, K, group, torch.float16, 3)
    G = K // group
    s = {"transposed": lambda: s.t().contiguous().t(), "row_broadcast": lambda: s[:1].expand(N, G),
         "group_broadcast": lambda: s[:, :1].expand(N, G),
         "padded": lambda: torch.cat([s, s], 1)[:, :G]}[layout]()
    v = torch.stack([q & 15, q >> 4], 2).reshape(N, K).double() - 8
    w = (v.reshape(N, G, group) * s.double()[:, :, None]).reshape(N, K)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(1)).bfloat16().to(dev)
    _check(int4_matmul(x, q, s, group), x, w, layout)


@pytest.mark.parametrize("bits,K,group", [(4, 2048, 32), (4, 2048, 64), (4, 2048, 128), (4, 2048, 256), (8, 2080, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_non_finite_rows(dev, bits, K, group, dtype):
    """Infinities and NaN in x reach exactly the outputs that fp32 arithmetic gives them."""
    M, N = 333, 1032
    q, s, w = _weights(dev, bits, N, K, group, torch.float32, 5)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(2)).to(dtype).to(dev)
    x[3, 7], x[40, K - 1], x[332, 100], x[7, 0], x[7, 900] = float("inf"), float("-inf"), float("nan"), float("inf"), float("inf")
    y, want = _run(bits, x, q, s, group).float(), x.float() @ w.float().t()
    bad = ~torch.isfinite(want)
    assert bad.any() and torch.equal(torch.isnan(y), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(y[inf], want[inf]) and torch.isfinite(y[~bad]).all()


def test_graph_replays_match_eager(dev):
    """A split call under capture: the partial products' workspace belongs to the graph."""
    q, s, _ = _weights(dev, 4, 1024, 4096, 128, torch.float16, 9)
    x = torch.randn(333, 4096, generator=torch.Generator().manual_seed(4)).bfloat16().to(dev)
    assert kernels.lib().mlsx_wq_workspace(4, 333, 1024, 4096, kernels.MLS_BF16, 128) > 0
    want = int4_matmul(x, q, s, 128)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = int4_matmul(x, q, s, 128)
    for i in range(3):
        graph.replay()
        junk = int4_matmul(x * (i + 2), q, s, 128)  # eager work between the replays
        torch.cuda.synchronize()
        assert torch.equal(y, want) and not torch.equal(junk, want)


def test_short_workspace_takes_the_general_path(dev):
    """Without the workspace the call still runs (on the general entry point's kernels)."""
    M, N, K = 333, 512, 4096
    q, s, w = _weights(dev, 8, N, K, 0, torch.float32, 11)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(4)).bfloat16().to(dev)
    c = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    rc = kernels.lib().mlsx_int8_gemm(x.data_ptr(), kernels.MLS_BF16, K, q.data_ptr(), K, s.data_ptr(), kernels.MLS_F32,
                                      c.data_ptr(), kernels.MLS_BF16, N, M, N, K, None, 0,
                                      torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    _check(c, x, w, "no workspace")


@pytest.mark.parametrize("dtype,bits,M,N,K,group", [
    (torch.float32, 4, 17000, 72, 4128, 32),     # three parts of x past the bound: rows in two launches
    (torch.bfloat16, 4, 12289, 4104, 7456, 32),  # a forced split whose partial products pass it
])
def test_rows_in_several_launches(dev, dtype, bits, M, N, K, group):
    """More rows than the workspace's bound allows, the last launch ragged, with strides on both
    sides; every 97th row and the launches' edges against float64."""
    q, s, w = _weights(dev, bits, N, K, group, torch.float32, 3)
    x = torch.randn(M, K + 32, generator=torch.Generator().manual_seed(6)).to(dtype).to(dev)[:, :K]
    assert kernels.lib().mlsx_wq_workspace(bits, M, N, K, kernels.MLS_F32 if dtype == torch.float32 else kernels.MLS_BF16,
                                           group) <= 768 << 20
    y = _run(bits, x, q, s, group)
    at = torch.tensor(sorted({*range(0, M, 97), 4095, 4096, 8191, 8192, M - 1}), device=dev)
    _check(y[at], x[at], w, f"{M}x{N}x{K}")


@pytest.mark.parametrize("bits,K,group", [(8, 4096, 0), (4, 4096, 64)])
def test_weights_at_8_of_16_bytes_keep_fp32(dev, bits, K, group):
    """fp32 x with weights that are 8- but not 16-byte aligned multiplies in fp32, as the general
    path's split asks for 16. A chain of K fp32 sums rounds by 2^-24 sqrt(K) / 2 of the norm (2e-6
    here, 1.1e-6 measured); two bf16 parts of x, which keep 2^-16 of it, have 4.9e-6."""
    M, N = 333, 1024
    assert kernels.lib().mlsx_wq_ksplit(bits, M, N, K, kernels.MLS_F32, group) > 0  # (aligned, it is split)
    q, s, w = _weights(dev, bits, N, K, group, torch.float32, 8)
    flat = torch.empty(q.numel() + 8, dtype=q.dtype, device=dev)[8:]
    off = flat.view(q.shape).copy_(q)
    assert off.data_ptr() % 16 == 8
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(6)).to(dev)
    want = x.double() @ w.t()
    assert float((_run(bits, x, off, s, group) - want).norm() / want.norm()) < 2.0 ** -24 * K ** 0.5 / 2


@pytest.mark.parametrize("scale", [1e-36, 1e-40, 1.0, 1e34])
@pytest.mark.parametrize("bits,M,N,K,group", [(4, 200, 264, 2048, 32), (8, 300, 264, 2080, 0)])
def test_three_parts_hold_every_value(dev, bits, M, N, K, group, scale):
    """fp32 x in three bf16 parts is x itself at every magnitude, so the outputs are as close to float64
    as fp32 sums are (the smallest: to the last place of a subnormal output)."""
    assert kernels.lib().mlsx_wq_ksplit(bits, M, N, K, kernels.MLS_F32, group) > 0
    q, s, w = _weights(dev, bits, N, K, group, torch.float32, 12)
    x = (torch.randn(M, K, generator=torch.Generator().manual_seed(6)) * scale).to(dev)
    y, want = _run(bits, x, q, s, group).double(), x.double() @ w.t()
    terms = (x.double().square() @ w.square().t()).sqrt()
    assert float(((y - want).abs() - 2.0 ** -17 * terms - 2.0 ** -148).max()) <= 0
