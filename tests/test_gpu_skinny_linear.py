"""A_compBT of a few rows: the kernel that streams the decoded weight against
FP64, at the edges of its tiles, its waves' shares of the columns and its range
of rows, and the calls it leaves to the library."""
from __future__ import annotations

import pytest
import torch

from losslessly_compressed_tensors_amd.kernels import fused
from losslessly_compressed_tensors_amd.operations import A_compBT, compress

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _values(*shape, seed=0, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to(
        torch.bfloat16).to(DEV)


@pytest.mark.parametrize("tokens", [1, 3, 15, 16])
@pytest.mark.parametrize("rows,cols", [(1, 8), (15, 24), (17, 32), (33, 264), (1000, 1032),
                                       (768, 4096), (4100, 520), (8200, 1000), (12300, 72)])
def test_skinny_linear(tokens, rows, cols):
    a, w = _values(tokens, cols), _values(rows, cols, seed=1, scale=0.05)
    out = fused.skinny_linear(a, w)
    exact = a.double() @ w.double().T
    size = a.double().abs() @ w.double().abs().T
    # At most `cols` FP32 additions, then one BF16 rounding (8 significant bits).
    assert bool(((out.double() - exact).abs()
                 <= cols * 2.0 ** -24 * size + 2.0 ** -8 * exact.abs()).all())


def test_routes():
    w = _values(192, 128, seed=1, scale=0.05)
    comp = compress(w)
    a = _values(4, 128)
    torch.testing.assert_close(A_compBT(a, comp), a @ w.T)
    wide = _values(4, 256)[:, ::2]                       # made contiguous first
    torch.testing.assert_close(A_compBT(wide, comp), wide @ w.T)
    leaf = a.clone().requires_grad_()
    A_compBT(leaf, comp).sum().backward()                # autograd sees the product
    torch.testing.assert_close(leaf.grad, w.float().sum(0).to(torch.bfloat16).expand(4, -1),
                               rtol=2 ** -7, atol=2 ** -7)
    assert fused.skinny_linear(_values(fused.MAX_SKINNY_TOKENS + 1, 128), w) is None
    assert fused.skinny_linear(a.float(), w.float()) is None
    assert fused.skinny_linear(_values(4, 12), _values(8, 12)) is None
