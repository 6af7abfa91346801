"""GPU: the fused updates' four-symbol steps where they can go wrong: quads whose
codes exceed 32 bits, escapes at each place of a quad, streams that end inside
a half, and tensors that end inside a row, a quad, a half or a chunk.  Every
stored field against the oracle's re-encode of the oracle's components."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import (
    assert_matches_oracle,
    bits_of,
    oracle_compress,
    oracle_from_components,
    require_gpu,
)
from losslessly_compressed_tensors_amd.codec.geometry import geometry
from losslessly_compressed_tensors_amd.comp_format import Distribution, DistType, NoiseLevel
from losslessly_compressed_tensors_amd.operations import (
    a_compA_add_b_B, a_compA_add_compB, compA_mul_B, compress)

pytestmark = pytest.mark.gpu

ALPHA, BETA = float(np.float32(0.75)), float(np.float32(-0.5))
DISTS = [Distribution(DistType.GAUSSIAN), Distribution(DistType.LAPLACE, zero_prob=0.01),
         Distribution(DistType.EMPIRICAL, noise_level=NoiseLevel.SPARSE)]
IDS = ["gaussian-clean", "laplace-clean", "empirical-sparse"]


def _bits(n: int, seed: int, rare: int) -> torch.Tensor:
    """Normal values, every `rare`-th one a random bit pattern (an escape, as a
    rule): each stream holds escapes at every place of a quad, and with
    rare = 1 quads of up to 64 bits and streams that overflow early."""
    rng = np.random.default_rng(seed)
    x = torch.from_numpy(rng.standard_normal(n, dtype=np.float32)).to(torch.bfloat16)
    bits = x.view(torch.int16).numpy().copy()
    bits[::rare] = rng.integers(0, 65536, size=bits[::rare].size, dtype=np.uint16).view(np.int16)
    return torch.from_numpy(bits).view(torch.bfloat16)


@pytest.mark.parametrize("dist", DISTS, ids=IDS)
@pytest.mark.parametrize("rare", [1, 7, 263])
def test_update_edges(dist, rare):
    require_gpu()
    block = geometry(dist)[0]
    alpha = torch.tensor([ALPHA], device="cuda")
    beta = torch.tensor([BETA], device="cuda")
    for n in (1, 255, 257, 4 * 256 + 1, 8 * 256 - 1, 8 * 256, 16 * 256 + 129, 32 * 256 + 3,
              block - 1, block, block + 1, 2 * block + 7 * 256 + 33):
        print(f"case quads {dist.family.name} rare={rare} n={n}", flush=True)
        a, b = _bits(n, 1 + n, rare), _bits(n, 2 + n, rare)
        ca, cb = compress(a.cuda(), dist), compress(b.cuda(), dist)
        oa, ob = oracle_compress(a, dist), oracle_compress(b, dist)
        for result, (side, exponents) in (
                (a_compA_add_b_B(ca, alpha, b.cuda(), beta, dense_output=False),
                 oracle.pointwise(oa, bits_of(b), oracle.OP_SCALAR_MUL_ADD, ALPHA, BETA, False,
                                  False, policy=1)),
                (compA_mul_B(ca, b.cuda(), dense_output=False),
                 oracle.pointwise(oa, bits_of(b), oracle.OP_MULTIPLY, 1.0, 1.0, False, True,
                                  policy=1)),
                (a_compA_add_compB(ca, alpha, cb, dense_output=False),
                 oracle.dual(oa, ob, ALPHA, policy=1))):
            assert_matches_oracle(result, oracle_from_components(side, exponents, dist))
