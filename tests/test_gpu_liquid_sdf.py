"""The liquid SDF (liquidSDFKernel) bit for bit against the oracle at each
number of workgroups a block of cells is dealt to: 1, 2, 4, 8 and 16 as the grid
has 1 210, 729, 343, 216 and 125 blocks; one particle, none in most blocks, a
dense cluster, and particles on the faces of the domain."""
import numpy as np
import pytest

import oracle_lib as O
from ffengine import kernels as K
from test_gpu_kernels import same_bits, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["one", "sparse", "cluster"])
@pytest.mark.parametrize("n3", [(101, 103, 97), (83, 81, 85), (70, 61, 70), (60, 55, 51), (49, 50, 41)])
def test_liquid_sdf_splits_bitexact(n3, kind):
    rng = np.random.default_rng(sum(n3))
    dx = 1.0 / max(n3)
    size = np.array(n3) * dx
    if kind == "one":
        pos = size[None] * 0.37
    elif kind == "sparse":
        pos = rng.random((3000, 3)) * size
        pos[:300, 0] = 0.0
        pos[300:600, 2] = size[2] * (1 - 1e-6)
    else:
        pos = size * 0.5 + (rng.random((20000, 3)) - 0.5) * 13 * dx
    pos = pos.astype(np.float32)
    r = 0.5 * dx * np.sqrt(3.0)
    say(f"liquid_sdf {n3} {kind}")
    assert same_bits(K.liquid_sdf(n3, dx, pos, r), O.liquid_sdf(n3, dx, pos, r))
