"""The fp32 weight gradient on the matrix cores (csrc/gemm_dw.hip) against float64: tile and stage
edges, strided operands, values far apart, infinities and NaN, and the calls that stay torch's."""

from __future__ import annotations

import pytest
import torch

import kernels
from kernels._hip import ld, stream

gpu = pytest.mark.gpu


def _dw(dy, x, pad=0):
    M, N = dy.shape
    K = x.shape[1]
    lib = kernels.lib()
    need = lib.mlsx_dw_fp32_workspace(M, N, K)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=dy.device)  # NaN parts wherever one is left unwritten
    out = torch.full((N, K + pad), 7.0, device=dy.device)
    kernels.check(lib.mlsx_dw_fp32(dy.data_ptr(), ld(dy), x.data_ptr(), ld(x), out.data_ptr(), K + pad, M, N, K,
                                   ws.data_ptr(), need, stream(dy.device)), "weight gradient")
    assert (out[:, K:] == 7.0).all()
    return out[:, :K]


def _bound(dy, x):
    """Three parts carry every value whole; the products left out are below 3 * 2^-24 of |dy||x|, and
    the two sums round at most once per MFMA and product, 2^-24 of the running |dy||x| each."""
    steps = 6 * (-(-dy.shape[0] // 32)) + 34
    return (dy.double().abs().t() @ x.double().abs()) * (steps + 3) * 2.0**-24 + 1e-300


@gpu
@pytest.mark.parametrize("M,N,K,pad", [
    (1, 1, 1, 0), (31, 16, 128, 0), (33, 129, 127, 1), (64, 256, 257, 0), (65, 383, 4, 4), (97, 130, 66, 3),
    (256, 2048, 2048, 0), (300, 4000, 4001, 0),
])
def test_against_float64(M, N, K, pad):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    wide = torch.randn(M, N + 5, generator=g, device="cuda")
    dy = wide[:, 5:] if pad % 2 else wide[:, :N].contiguous()  # (odd pad: rows of an odd stride)
    x = torch.randn(M, K, generator=g, device="cuda") * 1e-3
    err = (_dw(dy, x, pad).double() - dy.double().t() @ x.double()).abs()
    assert (err <= _bound(dy, x)).all()


@gpu
def test_values_far_apart():
    g = torch.Generator(device="cuda").manual_seed(0)
    s = torch.logspace(-14, 14, 192, device="cuda")[:, None]
    dy = torch.randn(192, 160, generator=g, device="cuda") * s
    x = torch.randn(192, 200, generator=g, device="cuda") / s
    err = (_dw(dy, x).double() - dy.double().t() @ x.double()).abs()
    assert (err <= _bound(dy, x)).all()


@gpu
def test_non_finite_as_fp32():
    """Small integers: the finite outputs are exact and the others follow from IEEE products."""
    g = torch.Generator(device="cuda").manual_seed(0)
    dy = torch.randint(-3, 4, (96, 300), generator=g, device="cuda").float()
    x = torch.randint(-3, 4, (96, 200), generator=g, device="cuda").float()
    dy[3, 5], dy[9, 77], x[3, 100], x[20, 9] = float("inf"), float("-inf"), float("inf"), float("nan")
    want = (dy.cpu()[:, :, None] * x.cpu()[:, None, :]).sum(0)
    assert torch.equal(torch.nan_to_num(_dw(dy, x).cpu(), 7.5, 8.5, 9.5), torch.nan_to_num(want, 7.5, 8.5, 9.5))
    assert want.isnan().any() and want.isinf().any()


@gpu
@pytest.mark.parametrize("sd,sx", [(1e-36, 1.0), (1e4, 1e-38), (1e-20, 1e-16), (1e34, 1e-36), (3e33, 1e2), (1e16, 1e17), (1e-41, 1e20)])
def test_every_scale_keeps_its_bits(sd, sx):
    """Values near fp32's smallest, whole or beside ordinary columns, and values and sums so large that
    the parts pass bf16's range, are as close to float64 as fp32 sums are."""
    g = torch.Generator(device="cuda").manual_seed(1)
    dy = torch.randn(96, 300, generator=g, device="cuda")
    x = torch.randn(96, 200, generator=g, device="cuda")
    for cols in (slice(None), slice(7, 9)):
        a, b = dy.clone(), x.clone()
        a[:, cols] *= sd
        b[:, cols] *= sx
        err = (_dw(a, b).double() - a.double().t() @ b.double()).abs()
        assert (err <= _bound(a, b) + 96 * 2.0**-149).all()


@gpu
def test_infinity_times_the_smallest_values():
    """An infinity times a value whose parts are small stays an infinity of its sign, as in fp32."""
    dy = torch.logspace(-44.5, 5, 257, device="cuda").repeat(40, 1) * torch.where(torch.arange(257, device="cuda") % 2 == 0, 1.0, -1.0)
    x = torch.ones(40, 130, device="cuda")
    x[11, 3] = float("-inf")
    got = _dw(dy, x)[:, 3]
    assert torch.equal(got, dy[11] * x[11, 3]) and torch.isinf(got).all()


@gpu
def test_route():
    """Where the kernel serves the gradient, and where torch must: a gradient of the gradient,
    16-bit and few tokens."""
    from kernels.int8_ste import _weight_grad
    g = torch.Generator(device="cuda").manual_seed(0)
    dy = torch.randn(1024, 2048, generator=g, device="cuda")
    x = torch.randn(2048, 1024, generator=g, device="cuda").t()  # a transposed view
    assert torch.equal(_weight_grad(dy, x), _dw(dy, x.contiguous()))
    xr = x.contiguous().requires_grad_()
    out = _weight_grad(dy, xr)
    assert out.grad_fn is not None
    assert torch.equal(out, dy.t() @ xr)
    assert torch.equal(_weight_grad(dy.half(), x.half()), dy.half().t() @ x.half())
    assert torch.equal(_weight_grad(dy[:8], x[:8]), dy[:8].t() @ x[:8])


def test_sizes_and_errors():
    lib = kernels.lib()
    assert lib.mlsx_dw_fp32_workspace(33, 10, 20) == 6 * 64 * 30
    assert lib.mlsx_dw_fp32_workspace(0, 10, 20) == 0
    assert lib.mlsx_dw_fp32_workspace(1 << 23, 10, 20) == 0  # 32-bit offsets of a block's rows
    assert lib.mlsx_dw_fp32_pays(2048, 4096, 4096) == 1
    assert lib.mlsx_dw_fp32_pays(255, 4096, 8192) == 0  # few tokens
    assert lib.mlsx_dw_fp32_pays(1023, 2048, 2048) == 0 and lib.mlsx_dw_fp32_pays(1024, 2048, 2048) == 1
    assert lib.mlsx_dw_fp32_pays(2048, 1024, 1024) == 0  # 64 tiles
    assert lib.mlsx_dw_fp32_pays(65536, 8192, 8192) == 0  # 6 GiB of parts
    with pytest.raises(ValueError):
        kernels.check(lib.mlsx_dw_fp32(64, 8, 64, 8, 64, 8, 4, 8, 8, 64, 10, None), "short workspace")
    with pytest.raises(NotImplementedError):
        kernels.check(lib.mlsx_dw_fp32(64, 8, 64, 8, 64, 8, 0, 8, 8, 64, 1 << 20, None), "no rows")
