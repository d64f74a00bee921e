"""Edge sizes of the row-span, band, backward, steering and copy kernels.

Frames repeat the oracle's operations in its order, so their tolerance is
zero; gradients are held to bounds of their float32 sums.
"""
from __future__ import annotations

import pytest
import torch

from pybatchrender import PBRConfig, PBRRenderer, _native, diff, workloads
from pybatchrender.envs.cartpole import CartPoleConfig, CartPoleGroundRenderer, CartPoleRenderer
from pybatchrender.envs.steering import SteeringConfig, SteeringRenderer
from pybatchrender.renderer.mesh import Mesh
from tests.test_gpu_parity import _bits, check_parity, ground_states
from tests.test_gpu_posed import _kernel_names

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


@pytest.mark.parametrize("n,dtype", [(7168, "float32"), (11264, "bfloat16"), (1536, "float32"),
                                     (1536, "bfloat16"), (1536, "uint8")])
def test_rows_kernel_store_forms(cuda, n, dtype):
    """Which stores are streaming depends on the output's bytes: the same
    pixels, alone and with depth and ids, as the scenes give in smaller batches."""
    st = ground_states(n, 3).cuda()
    vp = None  # the whole batch's: a view's aspect follows the batch's tile grid

    def frames(a, b):
        nonlocal vp
        r = CartPoleGroundRenderer(CartPoleConfig(num_scenes=b - a, device="cuda", kernel="rows",
                                                  output_dtype=dtype))
        r._step(st[a:b])
        if vp is None:
            vp = r._pbr_cam.VP_k44
        r._pbr_cam.VP_k44 = vp[a:b].clone()
        full = r.render(depth=True, vis=True)
        return r.render()["pixels"], full["pixels"], full["depth"], full["vis"]

    whole = frames(0, n)
    for a in range(0, n, 512):
        for x, y in zip(whole, frames(a, a + 512)):
            assert _bits(x[a:a + 512]).equal(_bits(y)), (a, x.dtype)


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


def _steering(n: int, seed: int) -> SteeringRenderer:
    g = torch.Generator("cpu").manual_seed(seed)
    r = SteeringRenderer(SteeringConfig(num_scenes=n, device="cuda", tile_resolution=(24, 20)))
    obs = torch.rand(n, 3, 4, generator=g) * torch.tensor([4.0, 30.0, 1.0, 1.0])
    r.build_obstacles(obs.cuda())
    fwd = torch.rand(n, 3, generator=g) - torch.tensor([0.5, -1.0, 0.5])
    r._pbr_cam.set_forward(fwd.cuda())
    return r


def _scene_bits(r: SteeringRenderer, pix: torch.Tensor) -> list[torch.Tensor]:
    cam = r._pbr_cam
    out = [pix, cam.eye_k3, cam.V_k44, cam.VP_k44]
    for nd in (r.player_node, r.left_border, r.right_border):
        out += [nd.transforms_b44, nd.rot3_b33, nd.scale_b11, nd.colors_b4]
    return [_bits(t) for t in out]


@pytest.mark.parametrize("cols", [2, 4, 7])
@pytest.mark.parametrize("n", [1, 3, 64, 65, 257])
def test_steering_step_launch_matches_tensor_operations(cuda, n, cols):
    """Every tensor the one-launch steering step writes, and its frame,
    against the same step by tensor operations: each layout of the state
    that is read in place, states with fewer rows, on the host, of another
    type, and in a scene's own buffer."""
    g = torch.Generator("cpu").manual_seed(100 * n + cols)
    a, b = _steering(n, 7), _steering(n, 7)
    b._step_device = lambda st: False
    base = torch.rand(n, cols, generator=g) * torch.tensor([3.0, 90.0] + [1.0] * (cols - 2))
    base[:: 3, 0] = -0.0
    dev = base.cuda()
    wide = torch.zeros(n, 2 * cols, device="cuda")
    wide[:, ::2] = dev
    for what, st in (("contiguous", dev), ("transposed", dev.t().contiguous().t()),
                     ("every second", wide[:, ::2]), ("host", base), ("double", dev.double()),
                     ("half the rows", dev[: (n + 1) // 2]), ("row", dev[0])):
        same = [x.equal(y) for x, y in zip(_scene_bits(a, a.step(st)), _scene_bits(b, b.step(st)))]
        assert all(same), f"n={n} cols={cols} {what}: {same}"
    if cols == 4:
        for r in (a, b):
            r.player_node.colors_b4.copy_(dev)
        same = [x.equal(y) for x, y in zip(_scene_bits(a, a.step(a.player_node.colors_b4)),
                                           _scene_bits(b, b.step(b.player_node.colors_b4)))]
        assert all(same), f"n={n}, state in the colour buffer: {same}"
    check_parity(a, f"steering n={n}", depth=False, vis=False,
                 got={"pixels": a.step(dev)})


@pytest.mark.parametrize("cols", [2, 4])
def test_steering_step_of_negated_memory(cuda, cols):
    """A state, or a tensor the step reads, whose memory holds the negatives
    of its values (torch's negative bit)."""
    g = torch.Generator("cpu").manual_seed(cols)
    a, b = _steering(65, 7), _steering(65, 7)
    b._step_device = lambda st: False
    z = torch.complex(torch.rand(65, cols, generator=g), torch.randn(65, cols, generator=g) * 2.0)
    state = z.cuda().conj().imag
    assert state.is_neg()
    same = [x.equal(y) for x, y in zip(_scene_bits(a, a.step(state)),
                                       _scene_bits(b, b.step(state.resolve_neg())))]
    assert all(same), same
    for r in (a, b):
        r._camera_eye_offset = torch._neg_view(r._camera_eye_offset)
    state = state.resolve_neg()
    same = [x.equal(y) for x, y in zip(_scene_bits(a, a.step(state)), _scene_bits(b, b.step(state)))]
    assert all(same), same


@pytest.mark.parametrize("what", ["subclass", "instance"])
def test_steering_step_calls_replaced_methods(cuda, what):
    """A subclass's or an object's own set_poses, set_colors and camera
    methods see the step's poses, colours and eye."""
    calls = []

    class Logged(SteeringRenderer):
        def set_poses(self, poses):
            calls.append("poses")
            super().set_poses(poses)

    def logged(obj, name):
        inner = getattr(obj, name)

        def method(*args, **kw):
            calls.append(name)
            return inner(*args, **kw)
        setattr(obj, name, method)

    r = _steering(5, 7)
    state = torch.rand(5, 4).cuda()
    r.step(state)
    if what == "subclass":
        r.__class__ = Logged
        r.step(state)
        assert calls == ["poses"]
        return
    for obj, name in ((r, "set_poses"), (r.player_node, "set_colors"),
                      (r._pbr_cam, "set_positions")):
        calls.clear()
        logged(obj, name)
        r.step(state)
        assert name in calls, name
        delattr(obj, name)


@pytest.mark.parametrize("shift_dst,shift_src", [(0, 0), (0, 1), (3, 0), (2, 2)])
def test_copy_segments(cuda, shift_dst, shift_src):
    """Copies and clears of 0 .. 70001 floats at aligned and odd addresses,
    and nothing written beside them."""
    sizes = [0, 1, 3, 4, 5, 255, 4096, 70001, 17]
    src = [torch.randn(n + shift_src + 8, device="cuda") for n in sizes]
    dst = [torch.full((n + shift_dst + 8,), 7.0, device="cuda") for n in sizes]
    want = [t.clone() for t in dst]
    segs = []
    for k, n in enumerate(sizes):
        clear = k % 3 == 1
        segs.append((dst[k].data_ptr() + 4 * shift_dst,
                     None if clear else src[k].data_ptr() + 4 * shift_src, 4 * n))
        want[k][shift_dst:shift_dst + n] = 0.0 if clear else src[k][shift_src:shift_src + n]
    _native.copy_segments(segs, _native.stream_ptr(src[0].device))
    for k, n in enumerate(sizes):
        assert torch.equal(dst[k], want[k]), f"segment {k} of {n} floats"
    with pytest.raises(RuntimeError, match="aligned"):
        _native.copy_segments([(dst[3].data_ptr() + 2, None, 4)], 0)


def test_gradients_from_unaligned_transforms(cuda):
    """Instance rows at an address that is no multiple of 16 are rendered
    through the copies the backward reads."""
    n = 9
    gen = torch.Generator("cpu").manual_seed(3)
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=(33, 20), device="cuda",
                              output_dtype="float32"))
    node = r.add_node("models/sphere", instances_per_scene=2)
    node.set_transforms(workloads.random_transforms(n * 2, gen, pos_range=1.0))
    node.set_colors(torch.rand(n * 2, 4, generator=gen))
    r.add_camera().set_positions_and_lookat(torch.tensor([0.0, -5.0, 1.0]), torch.zeros(3))
    r.add_light()
    r.setup_environment()
    gout = torch.randn(n, 3, 20, 33, generator=gen).cuda()

    def gradients():
        p = diff.scene_params(r)
        img = diff.render(r, p)
        # what the backward reads is frozen with the frame
        moved = node.transforms_b44
        saved = moved.clone()
        moved.zero_()
        grads = torch.autograd.grad(img, p.tensors(), gout)
        moved.copy_(saved)
        return [img.detach()] + [g.cpu() for g in grads]

    want = gradients()
    odd = torch.empty(node.transforms_b44.numel() + 1, device="cuda")[1:]
    odd = odd.reshape(node.transforms_b44.shape)
    odd.copy_(node.transforms_b44)
    node.transforms_b44 = odd
    got = gradients()
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:], want[1:]):
        # sums of float atomics in any order: a few hundred terms of 2^-24 each
        assert (a - b).abs().max() <= 2e-5 * b.abs().max() + 1e-30


def _strip_mesh(verts: int, tris: int, gen) -> Mesh:
    """A closed-looking blob of `tris` triangles on exactly `verts` vertices."""
    pos = torch.nn.functional.normalize(torch.randn(verts, 3, generator=gen), dim=1)
    tri = torch.stack([torch.randperm(verts, generator=gen)[:3] for _ in range(tris)])
    tri[0] = torch.tensor([0, verts // 2, verts - 1])
    return Mesh(pos.numpy(), pos.numpy(), tri.numpy())


@pytest.mark.parametrize("verts,tris", [(3, 1), (64, 63), (65, 64), (136, 256), (137, 256),
                                        (136, 257)])
@pytest.mark.parametrize("flat", [False, True])
def test_band_kernel_mesh_sizes(cuda, verts, tris, flat):
    """Meshes on both sides of what a wave's vertex table and triangle queue
    hold (beyond them the tile kernels draw), several instances a chunk."""
    gen = torch.Generator("cpu").manual_seed(verts + tris)
    n, k = 5, 7
    mesh = _strip_mesh(verts, tris, gen)
    if flat:
        mesh.normals[:] = mesh.normals[:1]
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=(45, 37), device="cuda",
                              kernel="tiles"))
    node = r.add_node(mesh, instances_per_scene=k)
    node.set_transforms(workloads.random_transforms(n * k, gen, pos_range=2.0,
                                                    scale_range=(0.2, 1.5)))
    node.set_colors(torch.rand(n * k, 4, generator=gen))
    node.set_instance_counts(torch.tensor([k, 0, 3, 1, k]))
    r.add_camera().set_positions_and_lookat(torch.tensor([0.0, -5.0, 1.0]), torch.zeros(3))
    r.add_light()
    r.setup_environment()
    check_parity(r, f"{verts} vertices, {tris} triangles")


@pytest.mark.parametrize("dtype", ["uint8", "bfloat16", "float32"])
@pytest.mark.parametrize("n,res", [(3, (33, 130)), (64, (40, 64)), (256, (21, 9)), (257, (21, 9)),
                                   (258, (20, 12)), (65, (128, 128))])
def test_band_kernel_forms(cuda, n, res, dtype):
    """Scene counts on both sides of the wide form and of its numbers of
    bands, frames of odd and of whole groups of four pixels: smooth and flat
    nodes, near-plane crossings of more triangles than the clip queue holds,
    long triangles beyond the frame, empty scenes."""
    gen = torch.Generator("cpu").manual_seed(n + res[0])
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=res, device="cuda", kernel="tiles",
                              output_dtype=dtype))
    for model, k, lo, hi in (("models/sphere", 3, 0.2, 1.0), ("models/cylinder", 3, 2.0, 9.0),
                             ("models/box", 9, 0.1, 30.0)):
        node = r.add_node(model, instances_per_scene=k)
        node.set_transforms(workloads.random_transforms(n * k, gen, pos_range=2.5,
                                                        scale_range=(lo, hi)))
        node.set_colors(torch.rand(n * k, 4, generator=gen))
        node.set_instance_counts(torch.randint(0, k + 1, (n,), generator=gen))
    r.add_camera(z_near=0.4)
    eye = torch.stack([torch.rand(n, generator=gen) * 4 - 2, torch.full((n,), -4.0),
                       torch.rand(n, generator=gen) * 3], 1)
    r._pbr_cam.set_positions_and_lookat(eye, torch.zeros(3))
    r.add_light()
    r.setup_environment()
    check_parity(r, f"band form n={n} {res} {dtype}")
    check_parity(r, f"band form n={n} {res} {dtype}, colour only", depth=False, vis=False)


@pytest.mark.parametrize("counts", [False, True])
@pytest.mark.parametrize("n", [1, 4, 16])
def test_band_kernel_few_scenes(cuda, n, counts):
    """Few scenes on both sides of the vertices per scene from which the tile
    kernels draw them (box: 24 vertices): the same frames as the oracle's, from
    the expected kernels; with instance counts it is the mean scene's vertices
    that decide."""
    line = (24576 + 6144 * n) // 24
    for k, band in ((line, True), (line + 1, False)):
        ips = 2 * k if counts else k
        r = workloads.many_cubes(num_scenes=n, resolution=33, instances=ips, seed=n, kernel="tiles",
                                 output_dtype="uint8", output_depth=False)
        if counts:  # k in the mean
            c = torch.full((n,), k)
            if n > 1:
                c[0], c[1] = 2 * k, 0
            r._drawn_nodes()[0].set_instance_counts(c)
        check_parity(r, f"n={n}, {k} of {ips} boxes", vis=False)
        names = _kernel_names(lambda: r.render())
        if names:
            assert any("bands_kernel" in s for s in names) == band, names
            assert any("tile_raster_kernel" in s for s in names) != band, names


@pytest.mark.parametrize("res,spheres", [((7, 40), 1), ((50, 17), 3), ((130, 33), 3),
                                         ((300, 16), 2), ((1000, 9), 2), ((64, 15), 8)])
def test_smooth_backward_pixel_sums(cuda, res, spheres):
    """The sorted smooth backward where a row is no whole run of eight pixels,
    a band takes several chunks of runs, the last band is short, and the
    visible slots take one pass or several.  Unlit, an instance's colour
    gradient is the sum of the output gradient over its pixels, so every
    pixel has to reach its own slot; a float32 sum of n terms in any order is
    within n 2^-24 of the sum of their magnitudes."""
    gen = torch.Generator("cpu").manual_seed(res[0])
    n, (W, H) = 2, res
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=res, device="cuda",
                              output_dtype="float32"))
    counts = (2, spheres)
    for model, k in zip(("models/box", "models/sphere"), counts):
        node = r.add_node(model, instances_per_scene=k)
        node.set_transforms(workloads.random_transforms(n * k, gen, pos_range=1.2,
                                                        scale_range=(0.5, 1.2)))
        node.set_colors(torch.rand(n * k, 4, generator=gen))
    r.add_camera().set_positions_and_lookat(torch.tensor([0.0, -5.0, 1.5]), torch.zeros(3))
    r.add_light(strength=0.0)
    r.setup_environment()
    gout = torch.randn(n, 3, H, W, generator=gen)
    p = diff.scene_params(r)
    grads = torch.autograd.grad(diff.render(r, p), p.colors, gout.cuda())
    vis = r.render(vis=True)["vis"].cpu()
    first = 0
    for got, k, ntri in zip(grads, counts, (12, 224)):
        for s in range(n):
            for i in range(k):
                lo = first + i * ntri
                mine = (vis[s] >= lo) & (vis[s] < lo + ntri)
                g = gout[s][:, mine].double()
                bound = mine.sum() * 2.0 ** -24 * g.abs().sum(1)
                err = (got[s * k + i, :3].cpu().double() - g.sum(1)).abs()
                assert (err <= bound).all(), (res, ntri, s, i, err, bound)
        first += k * ntri


@pytest.mark.parametrize("mesh", [1, 2, 5])
@pytest.mark.parametrize("res", [(64, 64), (50, 17), (130, 33), (300, 100)])
def test_smooth_backward_large_triangles(cuda, res, mesh):
    """Smooth triangles of many units of eight pixels each, whose sums are
    joined across a wave's lanes: one slot for whole waves, slots that change
    within a row of lanes, a last wave that is not full.  Unlit, a node's
    colour gradient is the sum of the output gradient over its pixels (bound as
    in test_smooth_backward_pixel_sums), also where one instance's gradient is
    infinite and its neighbour's is not."""
    W, H = res
    gen = torch.Generator("cpu").manual_seed(W + mesh)
    t = torch.linspace(-3.0, 3.0, mesh + 1)
    x, z = torch.meshgrid(t, t, indexing="ij")
    pos = torch.stack([x, 0.1 * x * z, z], -1).reshape(-1, 3)
    nrm = torch.stack([0.1 * x, -torch.ones_like(x), 0.1 * z], -1).reshape(-1, 3)
    a = (torch.arange(mesh)[:, None] * (mesh + 1) + torch.arange(mesh)).reshape(-1)
    b = a + mesh + 1
    tri = torch.cat([torch.stack([a, b, b + 1], 1), torch.stack([a, b + 1, a + 1], 1)])
    n = 3
    r = PBRRenderer(PBRConfig(num_scenes=n, tile_resolution=res, device="cuda",
                              output_dtype="float32"))
    node = r.add_node(Mesh(pos.numpy(), nrm.numpy(), tri.numpy()), instances_per_scene=2)
    eye = torch.eye(4).repeat(n * 2, 1, 1)
    eye[1::2, 0, 3] = 1.5  # the second plane covers the right part of the frame
    eye[1::2, 1, 3] = -0.7
    node.set_transforms(eye)
    node.set_colors(torch.rand(n * 2, 4, generator=gen))
    r.add_camera().set_positions_and_lookat(torch.tensor([0.0, -4.0, 0.3]), torch.zeros(3))
    r.add_light(strength=0.0)
    r.setup_environment()
    vis = r.render(vis=True)["vis"].cpu()
    inst = torch.where(vis >= 0, vis // len(tri), -1)
    assert all((inst[s] == i).sum() > W * H // 20 for s in range(n) for i in (0, 1))
    gout = torch.randn(n, 3, H, W, generator=gen)
    gout[2][:, inst[2] == 0] = float("inf")
    p = diff.scene_params(r)
    got = torch.autograd.grad(diff.render(r, p), p.colors, gout.cuda())[0].cpu()
    for s in range(n):
        for i in range(2):
            if (s, i) == (2, 0):
                assert not torch.isfinite(got[s * 2 + i, :3]).any()
                continue
            g = gout[s][:, inst[s] == i].double()
            bound = g.shape[1] * 2.0 ** -24 * g.abs().sum(1)
            err = (got[s * 2 + i, :3].double() - g.sum(1)).abs()
            assert (err <= bound).all(), (res, mesh, s, i, err, bound)


@pytest.mark.parametrize("mesh", [1, 5])
def test_smooth_backward_large_triangles_match_reference(cuda, mesh):
    """All gradients of lit smooth planes against the float64 reference."""
    from tests.test_diff import _assert_close, _kernel_and_reference

    t = torch.linspace(-3.0, 3.0, mesh + 1)
    x, z = torch.meshgrid(t, t, indexing="ij")
    pos = torch.stack([x, 0.1 * x * z, z], -1).reshape(-1, 3)
    nrm = torch.stack([0.1 * x, -torch.ones_like(x), 0.1 * z], -1).reshape(-1, 3)
    a = (torch.arange(mesh)[:, None] * (mesh + 1) + torch.arange(mesh)).reshape(-1)
    b = a + mesh + 1
    tri = torch.cat([torch.stack([a, b, b + 1], 1), torch.stack([a, b + 1, a + 1], 1)])
    r = PBRRenderer(PBRConfig(num_scenes=2, tile_resolution=(96, 96), device="cuda",
                              output_dtype="float32"))
    node = r.add_node(Mesh(pos.numpy(), nrm.numpy(), tri.numpy()), instances_per_scene=1)
    node.set_colors(torch.tensor([[0.3, 0.6, 0.5, 0.9], [0.8, 0.2, 0.4, 0.7]]))
    r.add_camera().set_positions_and_lookat(torch.tensor([0.2, -4.0, 0.3]), torch.zeros(3))
    r.add_light(ambient=(0.2, 0.2, 0.25), dir_dir=(0.1, 0.9, -0.3), dir_col=(0.9, 0.8, 0.7),
                strength=0.9)
    r.setup_environment()
    _assert_close(*_kernel_and_reference(r)[:2])
