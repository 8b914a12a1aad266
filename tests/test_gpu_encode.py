"""GPU: encoders at block counts that leave the last 64-block tile partial."""
import numpy as np
import pytest

import clibs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [clibs.Q8_0, clibs.Q4_K, clibs.Q6_K, clibs.IQ2_XXS])
@pytest.mark.parametrize("blocks", [1, 63, 65])
def test_encoded_blocks_of_partial_tiles(hip_ctx, orc, t, blocks):
    """Planes put in GGUF order on the device where the last 64-block tile is
    not whole: the reference's bytes."""
    x = clibs.gauss(7, f"pack.{blocks}", 256 * blocks, 0.02)
    assert np.array_equal(hip_ctx.quantize(t, x), clibs.quantize(orc, t, x))
