"""The tile kernels (records in device memory) and their persistent queue, by
options that the band path leaves to them: a tile size or a bin capacity.

Frames repeat the oracle's operations in its order, so their tolerance is
zero."""
from __future__ import annotations

import pytest
import torch

from pybatchrender import PBRConfig, PBRRenderer, autotune, workloads
from tests.test_gpu_parity import _bits, check_parity
from tests.test_gpu_posed import _kernel_names
from tests.test_zz_no_alloc import _render, _same

pytestmark = pytest.mark.gpu

# (tile_size, bin_capacity)
TILES = [(0, 1904), (0, 1024), (8, 0), (32, 0)]


def _draws_records(r) -> None:
    names = _kernel_names(lambda: r.render())
    if names:
        assert any("tile_raster_kernel" in s for s in names), names
        assert not any("bands_kernel" in s for s in names), names


@pytest.mark.parametrize("persistent", [False, True])
@pytest.mark.parametrize("ts,cap", TILES)
def test_tile_records_uneven_batch(cuda, ts, cap, persistent):
    r = workloads.uneven_batch(num_scenes=64, resolution=84, max_instances=96, seed=11,
                               kernel="tiles", tile_size=ts, bin_capacity=cap,
                               persistent=persistent)
    for k in range(2):
        check_parity(r, f"tiles {ts}, bins {cap}, persistent {persistent}, launch {k}")
    _draws_records(r)


@pytest.mark.parametrize("wide", [False, True])
def test_tile_records_few_persistent_workgroups(cuda, wide):
    """A queue of many more (scene, tile) items than workgroups."""
    r = workloads.many_cubes(num_scenes=70, resolution=64, instances=20, seed=2, kernel="tiles",
                             tile_size=16, persistent=True, output_dtype="float32")
    r.workgroups = 300 if wide else 3
    for k in range(2):
        check_parity(r, f"{r.workgroups} workgroups, launch {k}")


@pytest.mark.parametrize("persistent", [False, True])
def test_tile_records_many_tiny_and_empty_scenes(cuda, persistent):
    """Counts of 0, 1 or 2 boxes over 700 scenes with runs of empty scenes: a
    256-slot setup step crosses many scenes, so the setup's walk from the previous
    slot's scene and its binary-search fallback both run."""
    n = 700
    gen = torch.Generator("cpu").manual_seed(11)
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=(24, 24), device="cuda",
                              kernel="tiles", bin_capacity=1904, persistent=persistent))
    box = r.add_node("models/box", instances_per_scene=8,
                     model_pivot_relative_point=(0.5, 0.5, 0.5))
    counts = torch.randint(0, 3, (n,), generator=gen, dtype=torch.int32)
    counts[100:180] = 0
    counts[400:420] = 8
    box.set_instance_counts(counts)
    box.set_transforms(workloads.random_transforms(n * 8, gen, pos_range=1.0,
                                                   scale_range=(0.5, 1.2)))
    box.set_colors(torch.rand(n * 8, 4, generator=gen))
    r.add_camera(fov_y_deg=60.0, z_near=0.1, z_far=50.0)
    r._pbr_cam.set_positions_and_lookat(torch.tensor([[0.0, -5.0, 1.0]]).repeat(n, 1),
                                        torch.zeros(3))
    r.add_light()
    r.setup_environment()
    check_parity(r, f"700 tiny and empty scenes (persistent={persistent})")
    _draws_records(r)


@pytest.mark.parametrize("ts,cap", [(0, 1904), (32, 0)])
def test_tile_records_persistent_graph_replays(cuda, ts, cap):
    """The persistent queue in a hipGraph: its head is reset in every replay."""
    r = workloads.uneven_batch(num_scenes=160, resolution=64, max_instances=24, seed=5,
                               kernel="tiles", tile_size=ts, bin_capacity=cap, persistent=True)
    g = r.capture_step(depth=True, vis=True)
    gen = torch.Generator("cpu").manual_seed(9)
    nodes = r._drawn_nodes()
    full = [n.instance_counts.clone() for n in nodes]
    for k in range(4):
        for n, f in zip(nodes, full):
            M = workloads.random_transforms(n.transforms_b44.shape[0], gen)
            n.transforms_b44.copy_(M.to(n.transforms_b44.device))
            n.instance_counts.copy_(
                (f.cpu() - torch.randint(0, 3, f.shape, generator=gen)).clamp(min=0).to(f.device))
        got = {key: v.clone() for key, v in g().items()}
        torch.cuda.synchronize()
        assert not g.overflowed()
        out = check_parity(r, f"graph replay {k}, tiles {ts}")
        for key in ("pixels", "depth", "vis"):
            assert torch.equal(_bits(got[key]), _bits(out["got"][key])), f"replay {k}: {key}"


@pytest.mark.parametrize("persistent", [False, True])
def test_tile_records_noalloc(cuda, persistent):
    """pbr_render_noalloc's scratch memory under the records and the queue, the
    second batch on what the first left."""
    for n in (160, 37):
        r = workloads.uneven_batch(num_scenes=n, resolution=84, max_instances=48, seed=n,
                                   kernel="tiles", bin_capacity=1904, persistent=persistent)
        _same(_render(r, noalloc=True), _render(r, noalloc=False), f"N={n}")


def test_autotune_persistent_candidates_reach_the_queue(cuda):
    """Every persistent tile candidate runs the tile kernels, not the band
    path, which ignores the queue and its size."""
    r = workloads.uneven_batch(num_scenes=24, resolution=48, max_instances=16, seed=1)
    want = r.render()["pixels"].cpu()
    seen = 0
    for cand in autotune.candidates(r):
        if cand["kernel"] == "tiles" and cand["persistent"]:
            autotune._apply(r, cand)
            assert torch.equal(r.render()["pixels"].cpu(), want), cand
            _draws_records(r)
            seen += 1
    assert seen >= 12
