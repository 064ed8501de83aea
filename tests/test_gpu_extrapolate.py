"""The layered extrapolation (extrapLayerKernel: four faces a thread, status
bytes looked at as words) bit for bit against the oracle on arrays whose rows,
planes and sizes are no multiples of four, down to the smallest, with few, many
and no valid faces, and after more layers than there are faces to fill."""
import numpy as np
import pytest

import oracle_lib as O
from ffengine import kernels as K
from test_gpu_kernels import same_bits, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 12, 40])
@pytest.mark.parametrize("share", [0.0, 0.002, 0.3])
@pytest.mark.parametrize("shape", [(3, 3, 3), (4, 3, 5), (5, 6, 7), (17, 9, 33), (30, 31, 29), (8, 64, 12)])
def test_extrapolate_ragged_bitexact(shape, share, layers):
    rng = np.random.default_rng(sum(shape) + layers)
    field = rng.standard_normal(shape).astype(np.float32)
    valid = (rng.random(shape) < share).astype(np.uint8)
    if share:
        valid[tuple(a // 2 for a in shape)] = 1
    say(f"extrapolate {shape} {share} {layers}")
    assert same_bits(K.extrapolate(field, valid, layers), O.extrapolate(field, valid, layers))
