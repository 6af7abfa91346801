"""The one-pass kernels of the layers' dense steps against the expressions
they replace, at the edges of their accesses, row groups and register chunks."""
from __future__ import annotations

import pytest
import torch

from losslessly_compressed_tensors_amd.components import ops
from losslessly_compressed_tensors_amd.kernels import fused

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF = 2.0 ** -8      # BF16 rounding, relative: half of the last of 8 significand bits
STEP = 2.0 ** -24     # FP32 rounding, relative


def _values(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(
        torch.bfloat16).to(DEV)


@pytest.mark.parametrize("n", [1, 7, 8, 2047, 2048, 2049, 100003])
def test_relu_square(n):
    z, grad = _values(n), _values(n, seed=1)
    special = torch.tensor([float("nan"), float("inf"), -float("inf"), -0.0, 0.0, 3e38, -1e-40],
                           dtype=torch.bfloat16, device=DEV)[:n]
    z[-len(special):] = special
    grad[0] = float("inf")
    relu, square = fused.relu_square(z)
    assert torch.equal(relu.nan_to_num(9.0), z.relu().nan_to_num(9.0))
    assert torch.equal(square.nan_to_num(9.0), z.relu().square().nan_to_num(9.0))
    want = (grad * (2 * relu)).masked_fill(relu == 0, 0)
    again = fused.relu_square_backward(grad, relu)
    assert torch.equal(grad.isnan(), want.isnan())
    assert torch.equal(grad.nan_to_num(9.0), want.nan_to_num(9.0))
    assert torch.equal(again.nan_to_num(9.0), square.nan_to_num(9.0))


@pytest.mark.parametrize("rows,cols", [(1, 8), (31, 64), (33, 72), (257, 8), (1024, 8200),
                                       (8191, 768), (4099, 3080)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_column_sum(rows, cols, dtype, monkeypatch):
    monkeypatch.setattr(fused, "_MIN_SUM_ROWS", 1)
    g = _values(rows, cols)
    out = fused.column_sum(g, dtype)
    assert out.dtype == dtype
    exact, size = g.double().sum(0), g.double().abs().sum(0)
    # At most `rows` FP32 additions, then one BF16 rounding.
    assert bool(((out.double() - exact).abs() <= rows * STEP * size + HALF * exact.abs()).all())


@pytest.mark.parametrize("rows,cols", [(1, 4), (5, 252), (2051, 256), (4100, 260), (4097, 768),
                                       (33, 1000), (9, 1028), (3, 2052), (7, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rms_norm(rows, cols, dtype):
    x, grad = _values(rows, cols), _values(rows, cols, seed=1)
    x[0] = 0
    gain = (1 + 0.1 * _values(cols, seed=2).float()).to(dtype)
    w = gain.to(torch.bfloat16)
    y, rstd = fused.rms_norm(x, gain)
    ref_y, ref_rstd = torch.ops.aten._fused_rms_norm.default(x, [cols], w, None)
    assert rstd.shape == ref_rstd.shape and y.shape == x.shape
    # Sums of `cols` squares in two orders, a division and a reciprocal root.
    assert bool(((rstd - ref_rstd).abs() <= (cols + 8) * STEP * ref_rstd).all())
    h = x.double() * rstd.double()
    assert bool(((y.double() - h * w.double()).abs()
                 <= 1.01 * HALF * (h * w.double()).abs() + 1e-38).all())

    grad_x, grad_gain, rebuilt = fused.rms_norm_backward(grad, x, rstd, gain, dtype, True)
    assert torch.equal(rebuilt, y.view(-1, cols)) and grad_gain.dtype == dtype
    assert torch.equal(rebuilt, (x.float() * rstd * w.float()).to(torch.bfloat16))
    d = grad.double() * w.double()
    mean = (d * h).mean(1, keepdim=True)
    exact = rstd.double() * (d - h * mean)
    size = rstd.double() * (d.abs() + h.abs() * (d * h).abs().mean(1, keepdim=True))
    assert bool(((grad_x.double() - exact).abs()
                 <= (cols + 8) * STEP * size + 1.01 * HALF * exact.abs()).all())
    terms = grad.double() * h
    assert bool(((grad_gain.double() - terms.sum(0)).abs()
                 <= (rows + 4) * STEP * terms.abs().sum(0) + 1.01 * HALF * terms.sum(0).abs()
                 ).all())
    bare = fused.rms_norm_backward(grad, x, rstd, gain, dtype, False)
    assert torch.equal(bare[0], grad_x) and torch.equal(bare[1], grad_gain) and bare[2] is None


def test_what_the_kernels_leave_to_aten():
    x = _values(64, 256)
    assert fused.relu_square(x.t()) is None                        # strided
    assert fused.relu_square(x.float()) is None                    # another type
    assert fused.relu_square(x.view(-1)[1:]) is None               # not 16-byte aligned
    assert fused.relu_square(x[:0]) is None                        # empty
    assert fused.relu_square(x.cpu()) is None                      # on the host
    leaf = x.clone().requires_grad_()
    assert fused.relu_square(leaf) is None                         # autograd has to see it
    with torch.no_grad():
        assert fused.relu_square(leaf) is not None
        with torch.autocast("cuda", dtype=torch.float16):
            assert fused.relu_square(x) is None
    assert fused.column_sum(_values(1024, 12), torch.float32) is None
    assert fused.column_sum(_values(1023, 16), torch.float32) is None   # ATen is faster
    assert fused.rms_norm(_values(8, 4100), _values(4100)) is None
    assert fused.rms_norm(_values(8, 256), _values(1, 256)) is None


@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_a_trace_records_the_operations():
    """A traced norm computes its own inputs' norm."""
    first, x = _values(16384, 256), _values(16384, 256, seed=1)
    gain = 1 + 0.1 * _values(256, seed=2)
    assert fused.norm_pays(first, gain)
    traced = torch.jit.trace(lambda t: ops.rms_norm(t, gain), (first,))
    y, rstd = torch.ops.aten._fused_rms_norm.default(x, [256], gain, None)
    again = traced(x)
    assert torch.equal(again[0], y) and torch.equal(again[1], rstd)
