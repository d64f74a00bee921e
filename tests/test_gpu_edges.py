"""Edge sizes of the row-span and band kernels, bit for bit against the oracle.

Both kernels repeat the oracle's operations in its order, so the tolerance is
zero for every output.
"""
from __future__ import annotations

import pytest
import torch

from pybatchrender import PBRConfig, PBRRenderer, workloads
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


@pytest.mark.parametrize("cap", [0, 8])
@pytest.mark.parametrize("dtype", ["uint8", "bfloat16", "float32"])
@pytest.mark.parametrize("n", [2048, 2049])
def test_rows_kernel_record_forms(cuda, n, dtype, cap):
    """Small flat scenes on both sides of the scene count at which the
    32-record form takes over from the 64-record one: per-scene counts (some
    scenes empty), boxes around and through the near plane, short lists."""
    gen = torch.Generator("cpu").manual_seed(n + cap)
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=(31, 17), device="cuda",
                              kernel="rows", output_dtype=dtype, row_list_cap=cap))
    a = r.add_node("models/box", instances_per_scene=2,
                   model_pivot_relative_point=(0.5, 0.5, 0.5))
    a.set_transforms(workloads.random_transforms(n * 2, gen, pos_range=2.0,
                                                 scale_range=(0.5, 6.0)))
    a.set_colors(torch.rand(n * 2, 4, generator=gen))
    a.set_instance_counts(torch.randint(0, 3, (n,), generator=gen))
    b = r.add_node("models/quad", instances_per_scene=1, shared_across_scenes=True)
    b.set_transforms(workloads.random_transforms(1, gen, pos_range=1.0))
    b.set_colors(torch.rand(1, 4, generator=gen))
    b.set_instance_counts(torch.randint(0, 2, (n,), generator=gen))
    r.add_camera(z_near=0.3)
    eye = torch.stack([torch.rand(n, generator=gen) * 4 - 2, torch.full((n,), -5.0),
                       torch.rand(n, generator=gen) * 3], 1)
    r._pbr_cam.set_positions_and_lookat(eye, torch.zeros(3))
    r.add_light()
    r.setup_environment()
    check_parity(r, f"rows forms n={n} {dtype} cap={cap}")
    check_parity(r, f"rows forms n={n} {dtype} cap={cap}, colour only", depth=False, vis=False)


@pytest.mark.parametrize("n", [2048, 2049])
def test_posed_step_record_forms(cuda, n):
    """The posing launch in both forms: frames of the fused step."""
    r = CartPoleGroundRenderer(CartPoleConfig(num_scenes=n, device="cuda",
                                              tile_resolution=(33, 20)))
    pix = r.step(ground_states(n, 5).cuda())
    check_parity(r, f"posed step n={n}", depth=False, vis=False, got={"pixels": pix})
