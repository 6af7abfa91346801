"""CPU: which tensors the fused dense kernels take (``kernels/fused.py``), with
the device and the launch stood in for."""
from __future__ import annotations

import types

import pytest
import torch

from losslessly_compressed_tensors_amd import operations
from losslessly_compressed_tensors_amd.components import layers, ops
from losslessly_compressed_tensors_amd.kernels import fused


@pytest.fixture
def no_launch(monkeypatch):
    """Every tensor counts as the kernels' own; a launch fails the test."""
    monkeypatch.setattr(fused, "native", lambda *tensors: True)
    monkeypatch.setattr(fused, "_stream", lambda tensor: 0)
    monkeypatch.setattr(fused.hip, "call", lambda name, *args: pytest.fail(f"launched {name}"))


@pytest.mark.parametrize("shape", [(5, 8, 3), (5, 8, 8), (2, 8, 5, 3)])
@pytest.mark.filterwarnings("ignore:The use of `x.T`")
def test_few_row_product_takes_matrices_only(no_launch, monkeypatch, shape):
    """A weight of more dimensions keeps the library's broadcast product."""
    a = torch.randn(4, 8).to(torch.bfloat16)
    w = torch.randn(shape).to(torch.bfloat16)
    assert fused.skinny_linear(a, w) is None
    monkeypatch.setattr(operations, "decompress", lambda record: w)
    try:
        expected = a @ w.T
    except RuntimeError as error:     # refused before, refused the same way
        with pytest.raises(type(error)):
            operations.A_compBT(a, types.SimpleNamespace(shape=w.shape))
        return
    assert torch.equal(operations.A_compBT(a, types.SimpleNamespace(shape=w.shape)), expected)


def test_few_row_product_takes_matching_columns_only(no_launch):
    a = torch.zeros(4, 8, dtype=torch.bfloat16)
    assert fused.skinny_linear(a, torch.zeros(5, 16, dtype=torch.bfloat16)) is None


def test_tensors_past_the_launch_limits_are_left_to_aten(no_launch):
    def empty(*shape):
        return torch.empty(*shape, dtype=torch.bfloat16, device="meta")

    assert fused.rms_norm(empty(2 ** 26 - 3, 64), empty(64)) is None
    assert fused.rms_norm(empty(2 ** 31, 4), empty(4)) is None
    assert fused.relu_square(empty(2 ** 33 + 8)) is None
    assert fused.relu_square_backward(empty(2 ** 35), empty(2 ** 35)) is None
    assert fused.skinny_linear(empty(16, 8), empty(2 ** 29 - 63, 8)) is None


def test_small_calls_stay_with_aten(no_launch):
    """Where ATen's call takes less time than a launch of the row kernels."""
    for rows, cols in ((1, 256), (64, 768), (1024, 64)):
        x = torch.randn(rows, cols).to(torch.bfloat16)
        gain = torch.ones(cols, dtype=torch.bfloat16)
        y, rstd = ops._forward(x, gain)
        want = torch.ops.aten._fused_rms_norm.default(x, [cols], gain, None)
        assert torch.equal(y, want[0]) and torch.equal(rstd, want[1])
    g = torch.randn(1024, 64).to(torch.bfloat16)
    for dtype in (torch.bfloat16, torch.float32):
        assert torch.equal(layers._bias_grad(g, dtype), g.sum(0).to(dtype))


def test_where_the_row_kernels_pay():
    """Both sides of each line, at sizes where both were timed."""
    def empty(rows, cols, dtype=torch.bfloat16):
        return torch.empty(rows, cols, dtype=dtype, device="meta")

    def gain(cols, dtype=torch.bfloat16):
        return torch.empty(cols, dtype=dtype, device="meta")

    for rows, cols, pays in ((0, 256, False), (1, 64, False), (8192, 64, False), (16384, 64, False),
                             (8192, 768, False), (8192, 1024, False), (16384, 256, True),
                             (4096, 2048, False), (4096, 3072, False), (2048, 4096, False),
                             (4096, 4096, True), (8192, 2048, True)):
        assert fused.norm_pays(empty(rows, cols), gain(cols)) == pays, (rows, cols)
        assert fused.norm_pays(empty(rows, cols), gain(cols, torch.float32))
    for rows, cols, pays in ((0, 256, False), (16, 768, False), (4096, 64, False),
                             (8192, 64, True), (2048, 768, False), (4096, 768, True),
                             (2048, 1024, False), (1024, 2048, False), (2048, 2048, True),
                             (512, 3072, False), (1024, 3072, True), (256, 4096, False),
                             (512, 4096, True)):
        assert fused.norm_backward_pays(empty(rows, cols)) == pays, (rows, cols)
    assert not fused.norm_pays(torch.empty((), dtype=torch.bfloat16), gain(1))
    for rows, cols, bf16, fp32 in ((1023, 4096, False, False), (1024, 64, False, False), (1536, 64, False, True),
                                   (1024, 128, False, True), (8192, 8, False, False),
                                   (16384, 64, False, True), (4096, 128, False, True),
                                   (2048, 256, False, True), (4096, 256, True, True),
                                   (1536, 768, False, True), (2048, 768, True, True),
                                   (1024, 3072, True, True), (8192, 768, True, True)):
        assert fused.column_sum_pays(empty(rows, cols), torch.bfloat16) == bf16, (rows, cols)
        assert fused.column_sum_pays(empty(rows, cols), torch.float32) == fp32, (rows, cols)


class _DeviceTensor:
    """What ``native`` asks of a tensor, for one on device ``index``."""

    is_cuda = True
    requires_grad = False

    def __init__(self, index: int = 0):
        self.index = index

    def get_device(self):
        return self.index

    def is_contiguous(self):
        return True

    def numel(self):
        return 8

    def data_ptr(self):
        return 1 << 20

    def is_conj(self):
        return False

    is_neg = is_conj


@pytest.fixture
def device_tensors(monkeypatch):
    """``native`` on stand-ins for device tensors, the current device being 0."""
    monkeypatch.setattr(fused, "_PLAIN", (_DeviceTensor,))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
    monkeypatch.setattr(torch._C._functorch, "is_functorch_wrapped_tensor", lambda tensor: False)
    return _DeviceTensor


def test_every_tensor_is_on_the_current_device(device_tensors):
    here, there = device_tensors(0), device_tensors(1)
    assert fused.native(here) and fused.native(here, here, here)
    assert not fused.native(there)
    assert not fused.native(here, there)
    assert not fused.native(here, here, there)
    assert not fused.native(there, here)


def test_host_tensors_are_left_to_aten():
    assert not fused.native(torch.zeros(8))     # also without any device


@pytest.mark.filterwarnings("ignore::DeprecationWarning")
def test_tracing_and_transforms_see_atens_operations(device_tensors, monkeypatch):
    x = device_tensors()
    assert fused.native(x)
    seen = []

    def traced(value):
        seen.append(fused.native(x))
        return value + 1

    torch.jit.trace(traced, (torch.zeros(2),), check_trace=False)
    assert seen and not any(seen)
    with torch.autograd.forward_ad.dual_level():
        assert not fused.native(x)

    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not fused.native(x)
    monkeypatch.setattr(torch._C._functorch, "is_functorch_wrapped_tensor", lambda tensor: True)
    assert not fused.native(x)                  # vmap, grad and the other transforms
