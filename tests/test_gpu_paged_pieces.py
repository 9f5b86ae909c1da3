"""Paged attention over contexts cut into pieces: lengths at the edges of a piece, of a table, and
batches whose lengths differ by orders of magnitude, against float64."""

from __future__ import annotations

import pytest
import torch

import kernels
from kernels.paged_attention import paged_attention_decode

pytestmark = pytest.mark.gpu


def _want(q, k, v, tab, lens, bs):
    out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
    for i, n in enumerate(lens):
        n = min(n, tab.shape[1] * bs)
        if n > 0:
            ids = tab[i, :-(-n // bs)].long()
            kk, vv = (t[ids].transpose(0, 1).reshape(q.shape[1], -1, q.shape[2])[:, :n].double() for t in (k, v))
            p = torch.softmax((kk * q[i].double()[:, None]).sum(-1) * q.shape[2] ** -0.5, -1)
            out[i] = (p[:, :, None] * vv).sum(1)
    return out


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float32, 64), (torch.float32, 24)])
@pytest.mark.parametrize("lens,H,bs,extra", [
    ([128], 2, 16, 0), ([129], 2, 16, 0), ([127, 1, 0, 256, 257], 3, 16, 0),
    ([3000, 1, 17, 0, 900], 4, 16, 5),       # a table wider than any context
    ([5000, 5000], 1, 8, 0), ([1024 + 1], 2, 1, 0),   # more than 64 blocks a piece
    ([40] * 300 + [2000], 2, 32, 0),         # past 256 sequences: the length from the table's width
    ([2048] * 3, 32, 16, -20),               # contexts past the table's end are cut there
    ([500, 3, 129], 4, 16, 1000),            # a table 32 times as wide as the longest context
    ([40] * 299 + [900, 2000], 8, 16, 4000), ([300] * 260, 16, 16, 600),
])
def test_pieces(dev, lens, H, bs, extra, dtype, D):
    g = torch.Generator().manual_seed(len(lens) + max(lens))
    n, per = len(lens), max(-(-max(lens) // bs) + extra, 1)
    used = [min(-(-v // bs), per) for v in lens]
    ids = torch.randperm(sum(used) + 3, generator=g).to(torch.int32)
    tab, at = torch.full((n, per), -7, dtype=torch.int32), 0  # unused entries are invalid ids
    for i, u in enumerate(used):
        tab[i, :u] = ids[at:at + u]
        at += u
    shape = (sum(used) + 3, H, bs, D)
    k, v = (torch.randn(*shape, generator=g).to(dtype).to(dev) for _ in range(2))
    q, tab = torch.randn(n, H, D, generator=g).to(dtype).to(dev), tab.to(dev)
    y = paged_attention_decode(q, k, v, tab, torch.tensor(lens, dtype=torch.int32, device=dev))
    want = _want(q, k, v, tab, lens, bs)
    # softmax and its sums in fp32 (2^-13 of the values' scale covers exp and 5000 terms), then one rounding
    bound = 2.0 ** -13 * v.double().abs().amax() + (0 if dtype == torch.float32 else 2.0 ** -8) * want.abs()
    assert float(((y.double() - want).abs() - bound).max()) <= 0


@pytest.mark.parametrize("lens,H", [([4096], 8), ([4096] * 8, 4), ([700, 1, 90], 4), ([200] * 300, 2)])
def test_pieces_do_not_depend_on_the_tables_width(dev, lens, H):
    """The contexts alone say how they are cut: a table 32 times as wide gives the same bits (a cut
    at other tokens would round differently), so it is walked by as many wavefronts."""
    bs, D, n = 16, 64, len(lens)
    g = torch.Generator().manual_seed(n)
    need = -(-max(lens) // bs)
    k, v = (torch.randn(64, H, bs, D, generator=g).bfloat16().to(dev) for _ in range(2))
    q = torch.randn(n, H, D, generator=g).bfloat16().to(dev)
    wide = torch.randint(0, 64, (n, 32 * need), generator=g, dtype=torch.int32).to(dev)
    ctx = torch.tensor(lens, dtype=torch.int32, device=dev)
    # (a table at least 64 pieces wide: the grid's room for pieces is the same in both)
    mid = max(need, 64 * 128 // bs)
    assert torch.equal(paged_attention_decode(q, k, v, wide[:, :mid], ctx), paged_attention_decode(q, k, v, wide, ctx))


def test_workspace_sizes():
    L = kernels.lib()
    assert L.mlsx_paged_attention_workspace(4, 8, 64, 16, 8) == 0                  # one piece
    assert L.mlsx_paged_attention_workspace(4, 8, 64, 16, 9) == 4 * 8 * 2 * 66
    assert L.mlsx_paged_attention_workspace(1, 1, 64, 16, 1 << 20) == 64 * 66      # at most 64 splits
    assert L.mlsx_paged_attention_workspace(0, 8, 64, 16, 9) == 0
    assert L.mlsx_paged_attention_workspace(40, 32, 128, 16, 1 << 16) == 40 * 32 * 13 * 130  # about 16384 wavefronts
    assert L.mlsx_paged_attention_workspace(300, 32, 128, 16, 44) == 0             # enough wavefronts uncut
