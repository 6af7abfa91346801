"""The reservations of a batched launch: made in job order under one hold of
the arena lock, after the deferred frees, each against what the jobs before it
left, whatever order the jobs' blocks finish in."""
from __future__ import annotations

import pytest
import torch

from gpu_util import require_gpu
from losslessly_compressed_tensors_amd.comp_format import DistType, Distribution
from losslessly_compressed_tensors_amd.kernels import dispatch
from losslessly_compressed_tensors_amd.operations import (
    a_compA_add_b_B_batch, compress_batch, decompress)
from losslessly_compressed_tensors_amd.tensor_buffer import (
    STATUS_EMPTY, STATUS_FREED, STATUS_OK, TensorBuffer)

pytestmark = pytest.mark.gpu
DIST = Distribution(DistType.GAUSSIAN)


@pytest.fixture(autouse=True)
def _gpu():
    require_gpu()


def _tensor(n, seed):
    """Values whose exponents spread too far for some streams."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(n, generator=g)
    x[torch.randperm(n, generator=g)[: n // 3]] *= 2.0 ** -20
    return x.to(torch.bfloat16).cuda()


# Ones of no overflow between them, and jobs of 1 to 40 blocks, the first and
# the last among the longest.
SIZES = [40 * 32768, 5, 32768, 3 * 32768 + 7, 70000, 9, 12 * 32768, 40000, 33, 2 * 32768,
         100, 5 * 32768, 1, 65536, 17 * 32768, 39 * 32768 - 1]


def _descriptor(record):
    return [int(v) for v in record.fallback_descriptor.cpu()]


def _first_fit(records, capacity):
    """What one first-fit allocator over [0, capacity) gives the records in
    order: (offset, size, status) each."""
    start, out = 0, []
    for r in records:
        request = int(r.fallback_used.item()) + 2 * int(r.fallback_count.item())
        size = -(-request // 16) * 16
        if request == 0:
            out.append((-1, 0, STATUS_EMPTY))
        elif start + size > capacity:
            out.append((-1, 0, None))
        else:
            out.append((start, size, STATUS_OK))
            start += size
    return out


@pytest.mark.parametrize("count", [1, 2, 16])
@pytest.mark.parametrize("room", [1.0, 0.6])
def test_reservations_follow_job_order(count, room):
    tensors = [_tensor(n, i) for i, n in enumerate(SIZES[:count])]
    large = TensorBuffer(1 << 24, device="cuda")
    records = compress_batch(tensors, DIST, buffer=large)
    whole = sum(size for _, size, _ in _first_fit(records, 1 << 24))
    assert whole > 0
    capacity = max(16, int(whole * room) // 16 * 16)
    buffer = TensorBuffer(capacity, device="cuda")
    for again in range(2):
        records = compress_batch(tensors, DIST, buffer=buffer)
        expected = _first_fit(records, capacity)
        for x, record, (offset, size, status) in zip(tensors, records, expected):
            got = _descriptor(record)
            assert got[:2] == [offset, size]
            if status is None:
                assert got[2] not in (STATUS_OK, STATUS_EMPTY)
            else:
                assert got[2] == status
                assert torch.equal(decompress(record).view(torch.int16), x.view(torch.int16))
        assert bool(buffer.failures()) == (None in [s for _, _, s in expected])
        # The frees of all of them wait for the next batch's reservations.
        kept = records
        for record, (_, _, status) in zip(records, expected):
            if status == STATUS_OK:
                record.free()
    records = compress_batch(tensors, DIST, buffer=buffer)
    assert [_descriptor(r)[:2] for r in records] == [list(e[:2]) for e in expected]
    assert all(_descriptor(r)[2] == STATUS_FREED
               for r, (_, _, status) in zip(kept, expected) if status == STATUS_OK)


def test_update_reservations_follow_job_order():
    alpha = torch.tensor([1.0], device="cuda")
    beta = torch.tensor([0.25], device="cuda")
    tensors = [_tensor(n, i) for i, n in enumerate(SIZES[:8])]
    others = [_tensor(n, 50 + i) for i, n in enumerate(SIZES[:8])]
    source = TensorBuffer(1 << 24, device="cuda")
    buffer = TensorBuffer(1 << 24, device="cuda")
    records = compress_batch(tensors, DIST, buffer=source)
    results = a_compA_add_b_B_batch(records, alpha, others, beta, buffer=buffer)
    expected = _first_fit(results, 1 << 24)
    assert [tuple(_descriptor(r)[:3]) for r in results] == expected
    for x, y, result in zip(tensors, others, results):
        want = torch.addcmul(x.float(), y.float(), beta).to(torch.bfloat16)
        assert torch.allclose(decompress(result).float(), want.float(), rtol=2 ** -7, atol=1e-30)


@pytest.mark.parametrize("epoch", [1, 0x7FFFFFFF, 0x80000000, 0x80000001, 0xFFFFFFFF])
@pytest.mark.parametrize("update", [False, True])
def test_requests_are_told_from_unwritten_words(epoch, update, monkeypatch):
    """At every epoch, the one whose top bit is its only one among them, a zeroed
    control array holds no request: each record has its reservation."""
    tensors = [_tensor(n, i) for i, n in enumerate(SIZES[:8])]
    source = TensorBuffer(1 << 24, device="cuda")
    buffer = TensorBuffer(1 << 24, device="cuda")
    records = compress_batch(tensors, DIST, buffer=source)
    calls = []
    monkeypatch.setattr(dispatch, "_control_arrays", {})
    monkeypatch.setattr(dispatch, "_next_fused_epoch", lambda: calls.append(1) or epoch)
    if update:
        one = torch.tensor([1.0], device="cuda")
        results = a_compA_add_b_B_batch(records, one, [torch.zeros_like(x) for x in tensors], one,
                                        buffer=buffer)
    else:
        results = compress_batch(tensors, DIST, buffer=buffer)
    assert len(calls) == 1      # an epoch serves one launch
    assert [tuple(_descriptor(r)[:3]) for r in results] == _first_fit(results, 1 << 24)
    assert not buffer.failures()
    for x, result in zip(tensors, results):
        # (x + 0 turns -0 into 0.)
        want = x + torch.zeros_like(x) if update else x
        assert torch.equal(decompress(result).view(torch.int16), want.view(torch.int16))
