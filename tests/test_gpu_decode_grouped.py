"""GPU: the grouped decoder (several symbols per table lookup) at the sizes where
its tiles, its streams' ends and its choice against the other decoders change.
The codec is lossless, so a decode is right exactly when it restores the input."""
import numpy as np
import pytest
import torch

from gpu_util import require_gpu
from losslessly_compressed_tensors_amd.codec.decode import decode_batch
from losslessly_compressed_tensors_amd.codec.geometry import geometry
from losslessly_compressed_tensors_amd.comp_format import Distribution, DistType, NoiseLevel
from losslessly_compressed_tensors_amd.kernels import hip
from losslessly_compressed_tensors_amd.operations import compress, decompress

pytestmark = pytest.mark.gpu

LAYOUTS = [(DistType.GAUSSIAN, NoiseLevel.CLEAN), (DistType.LAPLACE, NoiseLevel.CLEAN),
           (DistType.EMPIRICAL, NoiseLevel.SPARSE), (DistType.GAUSSIAN, NoiseLevel.MEDIUM),
           (DistType.LAPLACE, NoiseLevel.HIGH)]


def _values(kind: str, n: int) -> torch.Tensor:
    rng = np.random.default_rng(n)
    if kind == "bits":       # every exponent: escapes, and overflow in every stream
        bits = rng.integers(0, 65536, size=n, dtype=np.uint16)
    elif kind == "zeros":    # one symbol: the longest or the shortest codes
        bits = np.zeros(n, dtype=np.uint16)
    else:                    # few overflowing streams, whose tails are short
        x = torch.from_numpy(rng.standard_normal(n, dtype=np.float32)).to(torch.bfloat16)
        return x.cuda()
    return torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda()


@pytest.mark.parametrize("family,noise", LAYOUTS)
@pytest.mark.parametrize("kind", ["normal", "bits", "zeros"])
def test_grouped_decode_restores_tile_and_block_edges(family, noise, kind):
    """Ends inside and at the edges of a row, a 32-row unit, a 64-row tile and
    a block."""
    require_gpu()
    print(f"case grouped {family.name} {noise.name} {kind}", flush=True)
    dist = Distribution(family, noise_level=noise)
    block = geometry(dist)[0]
    for n in (1, 7, 8, 255, 256, 257, 32 * 256 - 1, 32 * 256 + 5, 64 * 256, 64 * 256 + 1,
              block - 1, block, block + 1, 3 * block + 64 * 256 + 131):
        x = _values(kind, n)
        assert torch.equal(decompress(compress(x, dist)).view(torch.int16), x.view(torch.int16)), n


@pytest.mark.parametrize("family,noise", LAYOUTS)
@pytest.mark.parametrize("run", [1, 2, 3, 5, 30, 64, 70])
def test_runs_of_escapes(family, noise, run):
    """Rows of 256 values whose exponents no code has, `run` at a time at every
    distance from a tile's edges, in all lanes and in every third."""
    require_gpu()
    print(f"case runs {family.name} {noise.name} {run}", flush=True)
    dist = Distribution(family, noise_level=noise)
    block = geometry(dist)[0]
    generator = torch.Generator(device="cuda").manual_seed(run)
    x = torch.randn(3 * block + 777, device="cuda", generator=generator).to(torch.bfloat16)
    rows = x[:3 * block].view(-1, 256)
    start, far = 0, 2.0 ** -70
    for gap in range(1, 40):
        rows[start:start + run] *= far
        start += run + gap
    rows[block // 256:2 * block // 256, 1::3] *= far
    record = compress(x, dist)
    assert torch.equal(decompress(record).view(torch.int16), x.view(torch.int16))
    assert torch.equal(decode_batch([record, record])[1].view(torch.int16), x.view(torch.int16))


@pytest.mark.parametrize("family,noise", LAYOUTS)
@pytest.mark.parametrize("mode", [1, 2, 4])
def test_each_decoder_restores_whole_and_partial_blocks(family, noise, mode):
    """The wide, the compact and the grouped kernel pinned, singly and in one
    batched launch, on values of every exponent and with few overflows."""
    require_gpu()
    print(f"case pinned {mode} {family.name} {noise.name}", flush=True)
    dist = Distribution(family, noise_level=noise)
    block = geometry(dist)[0]
    hip.call("lct_set_decoder", mode)
    try:
        for kind in ("normal", "bits"):
            tensors = [_values(kind, n) for n in (777, block, 2 * block - 1, 2 * block + 33 * 256 + 5)]
            records = [compress(x, dist) for x in tensors]
            for x, record, y in zip(tensors, records, decode_batch(records)):
                assert torch.equal(decompress(record).view(torch.int16), x.view(torch.int16))
                assert torch.equal(y.view(torch.int16), x.view(torch.int16))
    finally:
        hip.call("lct_set_decoder", 0)


@pytest.mark.parametrize("blocks", [767, 768, 1024, 1600])
def test_decode_around_the_grids_held_at_once(blocks):
    """W = 25: 768 workgroups of the grouped kernel and 1024 of the wide one are
    resident at once; single decodes and one batched launch of two tensors on
    either side of both, whole and ragged."""
    require_gpu()
    print(f"case grids {blocks}", flush=True)
    dist = Distribution(DistType.LAPLACE)
    block = geometry(dist)[0]
    generator = torch.Generator(device="cuda").manual_seed(blocks)
    for n in (blocks * block, blocks * block - 333):
        x = torch.randn(n, device="cuda", generator=generator).to(torch.bfloat16)
        whole = compress(x, dist)
        assert torch.equal(decompress(whole).view(torch.int16), x.view(torch.int16))
        half = (blocks // 2) * block
        parts = [x[:half], x[half:]]
        for y, part in zip(decode_batch([compress(p, dist) for p in parts]), parts):
            assert torch.equal(y.view(torch.int16), part.view(torch.int16))


@pytest.mark.parametrize("family,noise,blocks",
                         [(DistType.GAUSSIAN, NoiseLevel.CLEAN, (1024, 1025, 1410, 2049)),
                          (DistType.GAUSSIAN, NoiseLevel.MEDIUM, (769, 1410, 2049, 3073)),
                          (DistType.LAPLACE, NoiseLevel.HIGH, (769, 1281, 1537)),
                          (DistType.EMPIRICAL, NoiseLevel.SPARSE, (769, 1025, 1153)),
                          (DistType.LAPLACE, NoiseLevel.CLEAN, (1025, 1153))])
def test_decode_where_the_choice_changes(family, noise, blocks):
    """Grids on either side of the lines of choose_decoder, whole and ragged,
    single and batched."""
    require_gpu()
    dist = Distribution(family, noise_level=noise)
    block = geometry(dist)[0]
    for count in blocks:
        print(f"case choice {family.name} {noise.name} {count}", flush=True)
        generator = torch.Generator(device="cuda").manual_seed(count)
        x = torch.randn(count * block, device="cuda", generator=generator).to(torch.bfloat16)
        for y in (x, x[:-12345]):
            records = [compress(y, dist)]
            assert torch.equal(decompress(records[0]).view(torch.int16), y.view(torch.int16))
            cut = (count // 3) * block
            parts = [y[:cut], y[cut:]]
            for out, part in zip(decode_batch([compress(p, dist) for p in parts]), parts):
                assert torch.equal(out.view(torch.int16), part.view(torch.int16))
