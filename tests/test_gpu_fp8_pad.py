"""The padded fp8 encoders and the amax kernel behind FP8Linear's steps."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from kernels.fp8_matmul import (E4M3_MAX, E5M2_MAX, amax_scales, encode_padded, fp8_matmul, quantize_e4m3,
                                quantize_e5m2)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e5m2", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("R,C,off", [(1, 1, 0), (64, 64, 0), (63, 65, 0), (65, 63, 0), (130, 300, 0), (100, 128, 4), (128, 176, 0)])
def test_encode_padded(dev, R, C, off, dtype, e5m2):
    """Both layouts bit-identical to the plain encoders, zero bytes in the padding, and e4m3
    NaN codes kept only in a copy whose reduction axis needs no padding (exact: bytes)."""
    g = torch.Generator().manual_seed(R * 31 + C)
    x = (torch.randn(R, C + off, generator=g) * 300).to(dtype).to(dev)[:, off:]
    x[R // 2, C // 2] = float("nan")
    x[0, 0] = float("inf")
    bits, bits_t = encode_padded(x, 0.37, e5m2=e5m2)
    want = (quantize_e5m2 if e5m2 else quantize_e4m3)(x.contiguous(), 0.37)
    zeroed = torch.where((want & 0x7F) == 0x7F, torch.zeros_like(want), want)
    Rp, Cp = (R + 63) // 64 * 64, (C + 63) // 64 * 64
    assert bits.shape == (R, Cp) and bits_t.shape == (C, Rp)
    assert torch.equal(bits[:, :C], want if e5m2 or C % 64 == 0 else zeroed)
    assert torch.equal(bits_t[:, :R], (want if e5m2 or R % 64 == 0 else zeroed).t())
    assert not bits[:, C:].any() and not bits_t[:, R:].any()
    alone, none = encode_padded(x, 0.37, e5m2=e5m2, transposed=False)
    assert none is None and torch.equal(alone, bits)


@pytest.mark.parametrize("M,N,K", [(16, 16, 65), (100, 48, 130), (300, 260, 1000)])
def test_padded_gemm_matches_ragged(dev, M, N, K):
    """The padded operands through the matrix cores against the same operands at the ragged
    K: fp32 sums of exact products in two orders, |d| <= K 2^-24 sum |a b|."""
    g = torch.Generator().manual_seed(K)
    a, b = torch.randn(M, K, generator=g).to(dev), torch.randn(N, K, generator=g).to(dev)
    got = fp8_matmul(encode_padded(a, 0.1, transposed=False)[0], encode_padded(b, 0.1, transposed=False)[0], 0.1, 0.1)
    qa, qb = quantize_e4m3(a, 0.1), quantize_e4m3(b, 0.1)
    want = fp8_matmul(qa, qb, 0.1, 0.1)
    va, vb = (q.view(torch.float8_e4m3fn).double() for q in (qa, qb))
    bound = K * 2.0 ** -24 * 0.01 * (va.abs() @ vb.abs().t())
    assert float(((got - want).double().abs() - bound).max()) <= 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,off", [(1, 0), (7, 1), (4096, 0), (1_000_003, 0), (5_000_001, 3)])
def test_amax_scales(dev, n, off, dtype):
    """Bit-identical to torch's amax and to a host division rounded to fp32, aligned or not."""
    x = torch.randn(n + off, generator=torch.Generator().manual_seed(n)).to(dtype).to(dev)[off:]
    x[n // 2] = -9.5
    y = torch.zeros(33, device=dev)  # an all-zero tensor takes the floor
    amax, scale = amax_scales([x, y], E4M3_MAX).cpu()
    want = float(x.abs().amax())
    assert float(amax[0]) == want and float(amax[1]) == 0.0
    assert float(scale[0]) == np.float32(want / E4M3_MAX) and float(scale[1]) == np.float32(1e-12)
    for bad in (float("inf"), float("nan")):
        x[0] = bad
        got = amax_scales([x], E5M2_MAX).cpu()
        assert np.array_equal(got.numpy().ravel(), np.float32([bad, bad]), equal_nan=True)


def test_amax_scales_declines(dev):
    """A layout or dtype that the kernel does not read is left to torch's own ops."""
    x = torch.randn(8, 8, device=dev)
    assert amax_scales([x.t()], 1.0) is None and amax_scales([x[:0]], 1.0) is None
    assert amax_scales([x.double()], 1.0) is None and amax_scales([x.cpu()], 1.0) is None
