"""Edge sizes of the row-span and band kernels, bit for bit against the oracle.

Both kernels repeat the oracle's operations in its order, so the tolerance is
zero for every output.
"""
from __future__ import annotations

import pytest

from pybatchrender.envs.cartpole import CartPoleConfig, CartPoleGroundRenderer, CartPoleRenderer
from tests.test_gpu_parity import check_parity, ground_states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["uint8", "bfloat16", "float32"])
@pytest.mark.parametrize("width", [2, 5, 47, 63, 65, 127])
def test_rows_kernel_ragged_widths(cuda, width, dtype):
    """Tile widths that are no multiple of a lane's pixels: narrower than one
    lane, one pixel more or less than whole lanes, in both lane widths."""
    for cls in (CartPoleGroundRenderer, CartPoleRenderer):
        r = cls(CartPoleConfig(num_scenes=37, device="cuda", tile_resolution=(width, 21),
                               kernel="rows", output_dtype=dtype))
        r._step(ground_states(37, width).cuda())
        check_parity(r, f"rows width {width} {cls.__name__}")
        check_parity(r, f"rows width {width} {cls.__name__}, colour only", depth=False, vis=False)
