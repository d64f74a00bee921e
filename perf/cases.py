"""Workloads whose time counts for users of the renderer.

Each listed case is one call a training or simulation program makes per step:

  step / graph   ``renderer.step(state)`` of the CartPole scenes, eager or as
                 the captured graph (few boxes, one launch per step)
  steering       ``renderer.step(observation)`` of the steering scenes
                 (smooth spheres on a long track, rails crossing the near
                 plane, a moving camera)
  cubes          ``renderer.render()`` of N scenes of random boxes
  uneven         ``renderer.render()`` of scenes whose instance counts differ
                 (boxes, UV spheres and cylinders)
  grad           ``diff.render`` and its gradients for a given output
                 gradient: flat boxes, or boxes and smooth spheres

``exact`` draws the same inputs in float64 with plain torch: coverage and the
visible triangle are decided on the 1/256-pixel window positions a rasteriser
snaps its float32 vertices to, everything else is float64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

LIGHT = dict(ambient=(0.2, 0.2, 0.2), dir_dir=(-0.3, 0.5, -0.8), dir_col=(0.8, 0.8, 0.8))
BACKGROUND = 0.41
DTYPES = {"uint8": torch.uint8, "bfloat16": torch.bfloat16, "float32": torch.float32}
# scene x triangle x pixel tests exact() takes on at most (about 20 s)
EXACT_TESTS = 1e11


def listed():
    return [
        # a few scenes: an evaluation loop or a debugger's single step, all latency
        {"name": "step_64", "kind": "step", "scene": "ground", "n": 64, "w": 64, "h": 64,
         "dtype": "uint8"},
        # the throughput configuration of this repository's benchmark
        {"name": "step_4096", "kind": "step", "scene": "ground", "n": 4096, "w": 64, "h": 64,
         "dtype": "uint8"},
        # the reference's own scene (rail, cart, pole) at the 84-pixel frames of pixel agents
        {"name": "step_rail_1000x84", "kind": "step", "scene": "rail", "n": 1000, "w": 84, "h": 84,
         "dtype": "uint8"},
        # the largest environment batch: bf16 frames and depth for a policy, from a captured step
        {"name": "graph_16384_bf16_depth", "kind": "graph", "scene": "ground", "n": 16384, "w": 64,
         "h": 64, "dtype": "bfloat16"},
        # the steering environment with its default track of 100 obstacles
        {"name": "steering_512", "kind": "steering", "n": 512, "obstacles": 100, "w": 64, "h": 64},
        # many small objects per scene, float32 + depth
        {"name": "cubes_1024x128_f32", "kind": "cubes", "n": 1024, "w": 128, "h": 128, "k": 64,
         "dtype": "float32", "depth": True},
        # odd sizes: a rectangular tile, no multiple of 4 or 64 in any of them
        {"name": "cubes_301_101x75", "kind": "cubes", "n": 301, "w": 101, "h": 75, "k": 23,
         "dtype": "uint8", "depth": False},
        # instance counts from 1 to 256 per scene, one work queue
        {"name": "uneven_8192x84", "kind": "uneven", "n": 8192, "w": 84, "h": 84, "k": 256,
         "dtype": "uint8", "queue": True},
        # the same at a small, odd size
        {"name": "uneven_700_61x45", "kind": "uneven", "n": 700, "w": 61, "h": 45, "k": 24,
         "dtype": "bfloat16", "queue": False},
        # image and gradients of the CartPole batch: flat shading, colours / light / normals
        {"name": "grad_flat_4096", "kind": "grad", "n": 4096, "w": 64, "h": 64, "boxes": 2,
         "spheres": 0},
        # inverse rendering of smooth objects at full size
        {"name": "grad_smooth_512x128", "kind": "grad", "n": 512, "w": 128, "h": 128, "boxes": 16,
         "spheres": 16},
        # a small fit: few views of few objects, odd frame
        {"name": "grad_smooth_40_90x70", "kind": "grad", "n": 40, "w": 90, "h": 70, "boxes": 3,
         "spheres": 5},
    ]


def _span(rng, lo, hi):
    """A whole number in [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "graph", "steering", "cubes", "uneven", "grad"))
    if kind in ("step", "graph"):
        w, h = rng.randint(32, 128), rng.randint(32, 128)
        n = min(_span(rng, 16, 16384), 16384 * 64 * 64 // (w * h))
        return {"kind": kind, "scene": rng.choice(("ground", "rail")), "n": n, "w": w, "h": h,
                "dtype": rng.choice(tuple(DTYPES))}
    if kind == "steering":
        return {"kind": kind, "n": _span(rng, 8, 512), "obstacles": rng.randint(10, 100),
                "w": rng.choice((48, 64, 84)), "h": 64}
    if kind == "cubes":
        w, h, k = rng.randint(32, 160), rng.randint(32, 160), _span(rng, 6, 96)
        n = min(_span(rng, 16, 2048), 1024 * 128 * 128 // (w * h), 1024 * 64 // k)
        return {"kind": kind, "n": n, "w": w, "h": h, "k": k, "dtype": rng.choice(tuple(DTYPES)),
                "depth": rng.random() < 0.5}
    if kind == "uneven":
        k = _span(rng, 8, 256)
        w, h = rng.randint(32, 100), rng.randint(32, 100)
        n = min(_span(rng, 32, 8192), 8192 * 84 * 84 // (w * h), 8192 * 256 // k)
        return {"kind": kind, "n": n, "w": w, "h": h, "k": k, "dtype": rng.choice(tuple(DTYPES)),
                "queue": rng.random() < 0.5}
    spheres = rng.choice((0, _span(rng, 1, 16)))
    boxes = _span(rng, 1, 16)
    w, h = rng.randint(32, 128), rng.randint(32, 128)
    n = min(_span(rng, 16, 4096), 512 * 128 * 128 // (w * h))
    if spheres:
        n = min(n, 512 * 32 // (boxes + spheres))
    return {"kind": kind, "n": n, "w": w, "h": h, "boxes": boxes, "spheres": spheres}


# --- meshes (counter-clockwise seen from outside) ---------------------------

def _box():
    pos, nrm, tri = [], [], []
    for axis in range(3):
        for sign in (1.0, -1.0):
            n = np.eye(3)[axis] * sign
            u = np.eye(3)[(axis + 1) % 3]
            v = np.cross(n, u)
            b = len(pos)
            for su, sv in ((-1, -1), (1, -1), (1, 1), (-1, 1)):
                pos.append(0.5 * (n + su * u + sv * v) + 0.5)
                nrm.append(n)
            tri += [(b, b + 1, b + 2), (b, b + 2, b + 3)]
    return np.array(pos), np.array(nrm), np.array(tri)


def _sphere(seg=16, rings=8):
    th = math.pi * np.arange(1, rings) / rings
    ph = 2.0 * math.pi * np.arange(seg) / seg
    ring = np.stack([np.outer(np.sin(th), np.cos(ph)), np.outer(np.sin(th), np.sin(ph)),
                     np.outer(np.cos(th), np.ones(seg))], -1).reshape(-1, 3)
    nrm = np.concatenate([[[0.0, 0.0, 1.0]], ring, [[0.0, 0.0, -1.0]]])
    at = lambda r, s: 1 + (r - 1) * seg + s % seg  # noqa: E731
    tri = [(0, at(1, s), at(1, s + 1)) for s in range(seg)]
    for r in range(1, rings - 1):
        for s in range(seg):
            tri += [(at(r, s), at(r + 1, s), at(r + 1, s + 1)),
                    (at(r, s), at(r + 1, s + 1), at(r, s + 1))]
    tri += [(len(nrm) - 1, at(rings - 1, s + 1), at(rings - 1, s)) for s in range(seg)]
    return 0.5 * nrm, nrm, np.array(tri)


def _cylinder(seg=32):
    ph = 2.0 * math.pi * np.arange(seg) / seg
    rim = np.stack([np.cos(ph), np.sin(ph), 0.0 * ph], -1)
    up = np.array([0.0, 0.0, 1.0])
    lo, hi = 0.5 * rim - 0.5 * up, 0.5 * rim + 0.5 * up
    pos = [lo, hi, hi, 0.5 * up[None], lo, -0.5 * up[None]]
    nrm = [rim, rim, np.tile(up, (seg + 1, 1)), np.tile(-up, (seg + 1, 1))]
    a, b = np.arange(seg), (np.arange(seg) + 1) % seg
    tri = [np.stack([a, b, seg + b], 1), np.stack([a, seg + b, seg + a], 1),
           np.stack([2 * seg + a, 2 * seg + b, np.full(seg, 3 * seg)], 1),
           np.stack([3 * seg + 1 + b, 3 * seg + 1 + a, np.full(seg, 4 * seg + 1)], 1)]
    return np.concatenate(pos), np.concatenate(nrm), np.concatenate(tri)


# --- inputs -----------------------------------------------------------------

class _Draws:
    """Random inputs on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator("cuda").manual_seed(int(seed))

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device="cuda")

    def whole(self, n, *shape):
        return torch.randint(0, n, shape, generator=self.gen, device="cuda")

    def transforms(self, rows, spread, lo, hi):
        """Random rotations (uniform quaternions) x scales in [lo, hi], positions in
        [-spread, spread]^3."""
        w, x, y, z = torch.nn.functional.normalize(self.normal(rows, 4), dim=1).unbind(1)
        R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                         2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                         2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1)
        M = torch.zeros(rows, 4, 4, device="cuda")
        M[:, :3, :3] = R.reshape(-1, 3, 3) * self.uniform(lo, hi, rows, 1, 1)
        M[:, :3, 3] = self.uniform(-spread, spread, rows, 3)
        M[:, 3, 3] = 1.0
        return M

    def colors(self, rows, lo=0.0, hi=1.0):
        c = torch.ones(rows, 4, device="cuda")
        c[:, :3] = self.uniform(lo, hi, rows, 3)
        return c

    def yaw(self, n, eye):
        """Per-scene camera positions: `eye` turned about z."""
        a = self.uniform(0.0, 2.0 * math.pi, n)
        return torch.stack([-eye[1] * torch.sin(a), eye[1] * torch.cos(a),
                            torch.full_like(a, eye[2])], 1)


def _cartpole_state(case, seed):
    """Positions and angles an agent meets before an episode ends."""
    d, n = _Draws(seed), case["n"]
    return torch.stack([d.uniform(-2.4, 2.4, n), d.uniform(-1.0, 1.0, n),
                        d.uniform(-0.21, 0.21, n), d.uniform(-0.5, 0.5, n)], 1)


def _objects(case, seed):
    """Nodes (mesh, instances per scene, transforms, colours, counts), camera positions and
    light of a scene of random objects."""
    d, n = _Draws(seed), case["n"]
    nodes = []
    if case["kind"] == "cubes":
        rows = n * case["k"]
        nodes.append((_box(), case["k"], d.transforms(rows, 3.0, 0.1, 0.5), d.colors(rows), None))
        eye, strength = (0.0, -8.0, 3.0), 1.0
    elif case["kind"] == "uneven":
        k = case["k"]
        total = torch.round(torch.exp(d.uniform(0.0, math.log(k), n))).clamp(1, k).long()
        choice = d.whole(3, n, k)
        active = torch.arange(k, device="cuda")[None] < total[:, None]
        for j, mesh in enumerate((_box(), _sphere(), _cylinder())):
            cnt = ((choice == j) & active).sum(1).to(torch.int32)
            nodes.append((mesh, k, d.transforms(n * k, 3.0, 0.1, 0.5), d.colors(n * k), cnt))
        eye, strength = (0.0, -8.0, 3.0), 1.0
    else:
        for mesh, k in ((_box(), case["boxes"]), (_sphere(), case["spheres"])):
            if k:
                rows = n * k
                nodes.append((mesh, k, d.transforms(rows, 1.8, 0.5, 1.0),
                              d.colors(rows, 0.1, 0.9), None))
        eye, strength = (0.0, -5.0, 1.8), 0.9
    return nodes, d.yaw(n, eye), strength


def _output_gradient(case, seed):
    """What a mean-squared loss against another frame sends back."""
    n, h, w = case["n"], case["h"], case["w"]
    return _Draws(seed + 1).normal(n, 3, h, w) * (2.0 / (n * 3 * h * w))


def prepare(case, seed):
    from pybatchrender_amd.config import PBRConfig
    from pybatchrender_amd.renderer.mesh import Mesh
    from pybatchrender_amd.renderer.renderer import PBRRenderer

    kind, n, res = case["kind"], case["n"], (case["w"], case["h"])
    if kind in ("step", "graph"):
        from pybatchrender_amd.envs.cartpole import renderer as scenes
        from pybatchrender_amd.envs.cartpole.config import CartPoleConfig

        cfg = CartPoleConfig(num_scenes=n, tile_resolution=res, device="cuda",
                             output_dtype=case["dtype"])
        r = {"ground": scenes.CartPoleGroundRenderer, "rail": scenes.CartPoleRenderer}[
            case["scene"]](cfg)
        state = _cartpole_state(case, seed)
        if kind == "graph":
            return {"step": r.capture_step(state, depth=True), "input": state}
        return {"step": r.step, "input": state}
    if kind == "steering":
        from pybatchrender_amd.envs.steering import SteeringConfig, SteeringRenderer

        d = _Draws(seed)
        cfg = SteeringConfig(num_scenes=n, tile_resolution=res, device="cuda",
                             number_of_obstacles=case["obstacles"])
        r = SteeringRenderer(cfg)
        track = torch.zeros(n, case["obstacles"], 4, device="cuda")
        track[:, :, 0] = d.whole(12, n, case["obstacles"]).float() * 2.0 - 11.0
        track[:, :, 1] = torch.arange(case["obstacles"], device="cuda") * 12.0 + 6.0
        track[:, :, 2] = (d.uniform(0.0, 1.0, n, case["obstacles"]) < 0.2).float()
        r.build_obstacles(track)
        # cars spread over the track, some of them just crashed
        obs = torch.stack([d.uniform(-11.0, 11.0, n), d.uniform(0.0, 12.0 * case["obstacles"], n),
                           d.uniform(18.0, 110.0, n), (d.uniform(0.0, 1.0, n) < 0.1).float(),
                           d.uniform(-11.0, 11.0, n), d.uniform(0.0, 1200.0, n)], 1)
        return {"step": r.step, "input": obs}
    nodes, eye, strength = _objects(case, seed)
    cfg = PBRConfig(num_scenes=n, tile_resolution=res, device="cuda",
                    output_dtype=case.get("dtype", "float32"),
                    output_depth=case.get("depth", False), persistent=case.get("queue", False))
    r = PBRRenderer(cfg)
    for mesh, k, M, col, cnt in nodes:
        node = r.add_node(Mesh(*mesh), instances_per_scene=k)
        node.set_transforms(M)
        node.set_colors(col)
        if cnt is not None:
            node.set_instance_counts(cnt)
    r.add_camera(fov_y_deg=55.0).set_positions_and_lookat(eye, torch.zeros(3))
    r.add_light(strength=strength, **LIGHT)
    r.setup_environment()
    if kind != "grad":
        return {"render": r.render}
    from pybatchrender_amd import diff

    return {"renderer": r, "params": diff.scene_params(r), "grad": _output_gradient(case, seed)}


def run(state):
    if "step" in state:
        return state["step"](state["input"])
    if "render" in state:
        return state["render"]()
    from pybatchrender_amd import diff

    p = state["params"]
    img = diff.render(state["renderer"], p)
    gv, gl, *gc = torch.autograd.grad(img, [p.vertices, p.light, *p.colors], state["grad"])
    return {"image": img, "vertices": gv, "light": gl, "colors": gc}


def work(case):
    """Frames written (and, for gradients, the output gradient and the visible triangle of
    every pixel read), instance rows (a 4x4 matrix and a colour) and view-projections read; 60
    operations per vertex, 40 per triangle, 10 per pixel (100 more for its gradients)."""
    n, px = case["n"], case["n"] * case["w"] * case["h"]
    kind = case["kind"]
    size = {"uint8": 1, "bfloat16": 2, "float32": 4}[case.get("dtype", "uint8")]
    if kind in ("step", "graph"):
        out = px * (3 * size + (4 if kind == "graph" else 0))
        return {"bytes": out + n * (16 + 2 * 80 + 64), "flops": n * (52 * 60 + 26 * 40) + px * 10}
    if kind == "steering":
        inst = n * (case["obstacles"] + 3)
        return {"bytes": px * 3 + inst * 80 + n * 64,
                "flops": inst * (114 * 60 + 224 * 40) + px * 10}
    if kind == "cubes":
        inst = n * case["k"]
        return {"bytes": px * (3 * size + (4 if case["depth"] else 0)) + inst * 80 + n * 64,
                "flops": inst * (24 * 60 + 12 * 40) + px * 10}
    if kind == "uneven":
        # the mean of round(exp(U(0, ln k))) is about (k - 1) / ln k
        inst = n * (case["k"] - 1) / math.log(case["k"])
        return {"bytes": px * 3 * size + inst * 80 + n * 76,
                "flops": inst * (89 * 60 + 121 * 40) + px * 10}
    inst = n * (case["boxes"] + case["spheres"])
    flops = n * (case["boxes"] * (24 * 60 + 12 * 40) + case["spheres"] * (114 * 60 + 224 * 40))
    return {"bytes": px * (12 + 12 + 4) + inst * (2 * 80 + 16) + n * 128,
            "flops": 2 * flops + px * 110}


# --- float64 reference ------------------------------------------------------

def _view_projection(n, w, h, eye, target, fov, near=0.05, far=100.0):
    """[n, 4, 4] float32 view-projections (z up); the aspect is that of the near-square atlas
    of n tiles."""
    cols = math.ceil(math.sqrt(n))
    rows = math.ceil(n / cols)
    f = 1.0 / math.tan(math.radians(fov) * 0.5)
    P = torch.zeros(4, 4)
    P[0, 0] = f / ((cols * w) / (rows * h))
    P[1, 1] = f
    P[2, 2] = (far + near) / (near - far)
    P[2, 3] = (2.0 * far * near) / (near - far)
    P[3, 2] = -1.0
    unit = torch.nn.functional.normalize
    fwd = unit(target - eye, dim=1)
    s = unit(torch.cross(fwd, torch.tensor([[0.0, 0.0, 1.0]], device=eye.device).expand_as(fwd),
                         dim=1), dim=1)
    u = torch.cross(s, fwd, dim=1)
    V = torch.eye(4, device=eye.device).repeat(n, 1, 1)
    V[:, 0, :3], V[:, 1, :3], V[:, 2, :3] = s, u, -fwd
    V[:, 0, 3], V[:, 1, 3], V[:, 2, 3] = -(s * eye).sum(1), -(u * eye).sum(1), (fwd * eye).sum(1)
    return torch.matmul(P.to(eye.device)[None], V)


def _as_uploaded(M):
    """A matrix as the node holds it: rotation part times its mean row norm."""
    R = M[:, :3, :3]
    s = sum(torch.linalg.norm(R[:, k], dim=1) for k in range(3)) / 3.0
    s = s.reshape(-1, 1, 1)
    M = M.clone()
    M[:, :3, :3] = (R / s) * s
    return M


def _mul(A, v):
    """A [.., r, c] times v [.., c or 3 plus an implied 1], summed left to right."""
    out = A[..., 0] * v[..., None, 0] + A[..., 1] * v[..., None, 1]
    out = out + A[..., 2] * v[..., None, 2]
    return out + A[..., 3] * (v[..., None, 3] if v.shape[-1] == 4 else 1.0)


def _scene(nodes, VP, w, h):
    """Per scene and triangle (draw order), for a batch of scenes: snapped window positions,
    clip w, depth plane, vertex normals, colour, and indices for gradients."""
    out = []
    n = VP.shape[0]
    for j, (mesh, k, M, col, cnt) in enumerate(nodes):
        dev = M.device
        pos = torch.tensor(mesh[0], dtype=torch.float32, device=dev)
        nrm = torch.tensor(mesh[1], dtype=torch.float32, device=dev).double()
        tri = torch.tensor(mesh[2], dtype=torch.long, device=dev)
        M = M.reshape(n, k, 1, 4, 4)
        clip = _mul(VP[:, None, None], _mul(M, pos))           # [n, k, V, 4] float32
        iw = 1.0 / clip[..., 3]
        X = torch.round((clip[..., 0] * iw + 1.0) * (0.5 * w) * 256.0).double()
        Y = torch.round((clip[..., 1] * iw + 1.0) * (0.5 * h) * 256.0).double()
        d = (clip[..., 2] * iw * 0.5 + 0.5).double()
        wide = _mul(VP.double()[:, None, None], _mul(M.double(), pos.double()))
        N = torch.nn.functional.normalize((M[..., :3, :3].double() * nrm[:, None, :]).sum(-1), dim=-1)
        pick = lambda a: a[:, :, tri].reshape(n, -1, 3, *a.shape[3:])  # noqa: E731
        T = k * len(tri)
        live = torch.ones(n, k, device=dev, dtype=torch.bool)
        if cnt is not None:
            live = torch.arange(k, device=dev)[None] < cnt[:, None]
        inst = torch.arange(k, device=dev).repeat_interleave(len(tri))
        out.append({
            "X": pick(X), "Y": pick(Y), "d": pick(d), "W": pick(wide[..., 3]), "N": pick(N),
            "D": pick(wide[..., 2] / wide[..., 3] * 0.5 + 0.5),
            "C": col.double().reshape(n, k, 4)[:, inst], "live": live[:, inst],
            "node": torch.full((n, T), j, device=dev), "inst": inst.expand(n, T),
            "tri": torch.arange(T, device=dev).remainder(len(tri)).expand(n, T),
            "smooth": torch.full((n, T), not bool((nrm[tri] == nrm[tri][:, :1]).all()), device=dev),
        })
    return {key: torch.cat([o[key] for o in out], 1) for key in out[0]}


def _plane(X, Y, d):
    """Depth plane (zx, zy, zc) through three window positions in 1/256 pixel."""
    x, y = X / 256.0, Y / 256.0
    ax, ay, bx, by = x[..., 1] - x[..., 0], y[..., 1] - y[..., 0], x[..., 2] - x[..., 0], y[..., 2] - y[..., 0]
    area = ax * by - bx * ay
    d1, d2 = d[..., 1] - d[..., 0], d[..., 2] - d[..., 0]
    zx, zy = (d1 * by - d2 * ay) / area, (d2 * ax - d1 * bx) / area
    return zx, zy, d[..., 0] - zx * x[..., 0] - zy * y[..., 0], area


def _visible(S, w, h):
    """[n, h, w] index of the triangle each pixel shows, -1 for background (row 0 = top)."""
    dev = S["X"].device
    jj, ii = torch.meshgrid(torch.arange(h - 1, -1, -1, device=dev),
                            torch.arange(w, device=dev), indexing="ij")
    px, py = (256.0 * ii + 128.0).reshape(-1), (256.0 * jj + 128.0).reshape(-1)
    X, Y = S["X"], S["Y"]
    zx, zy, zc, area = _plane(X, Y, S["d"])
    n, T = area.shape
    best = torch.full((n, w * h), 1.0, dtype=torch.float64, device=dev)
    win = torch.full((n, w * h), -1, dtype=torch.long, device=dev)
    step = max(1, int(2 ** 27 // (n * w * h)))
    f32 = lambda a: a.float().double()  # noqa: E731
    zx, zy, zc = f32(zx), f32(zy), f32(zc)
    for t0 in range(0, T, step):
        t = slice(t0, min(T, t0 + step))
        ok = (S["live"][:, t] & (area[:, t] > 0.0))[..., None].expand(-1, -1, w * h)
        for k in range(3):
            a, b = (k + 1) % 3, (k + 2) % 3
            dx, dy = X[:, t, b] - X[:, t, a], Y[:, t, b] - Y[:, t, a]
            edge = dx[..., None] * (py - Y[:, t, a, None]) - dy[..., None] * (px - X[:, t, a, None])
            top_left = (dy < 0) | ((dy == 0) & (dx < 0))
            ok = ok & ((edge > 0) | ((edge == 0) & top_left[..., None]))
        tz = f32(zy[:, t, None] * (py / 256.0) + zc[:, t, None])
        z = f32(zx[:, t, None] * (px / 256.0) + tz).clamp(0.0, 1.0)
        z = torch.where(ok, z, 2.0)
        zmin, at = z.min(1)
        take = zmin < best
        best = torch.where(take, zmin, best)
        win = torch.where(take, at + t0, win)
    return win.reshape(n, h, w)


def _shade(N, rgba, light):
    """light: direction (3), colour (3), ambient (3), strength."""
    L = torch.nn.functional.normalize(light[:3], dim=0)
    N = torch.nn.functional.normalize(N, dim=-1)
    lam = (N * L).sum(-1, keepdim=True).clamp(min=0.0)
    s = light[9].clamp(0.0, 1.0)
    return rgba[..., :3] * ((1.0 - s) + (light[6:9] + lam * light[3:6]) * s)


def _frames(S, win, w, h, light):
    """Colour [n, 3, h, w] and depth [n, h, w] of the visible triangles."""
    at = win >= 0
    s, y, x = at.nonzero(as_tuple=True)
    t = win[at]
    px, py = 256.0 * x + 128.0, 256.0 * (h - 1 - y) + 128.0
    X, Y, N = S["X"][s, t], S["Y"][s, t], S["N"][s, t]
    e = torch.stack([(X[:, (k + 2) % 3] - X[:, (k + 1) % 3]) * (py - Y[:, (k + 1) % 3])
                     - (Y[:, (k + 2) % 3] - Y[:, (k + 1) % 3]) * (px - X[:, (k + 1) % 3])
                     for k in range(3)], 1)
    bary = e / S["W"][s, t]
    mixed = (bary[..., None] * N).sum(1)
    col = _shade(torch.where(S["smooth"][s, t][:, None], mixed, N[:, 0]), S["C"][s, t], light)
    out = torch.full((*win.shape, 3), BACKGROUND, dtype=torch.float64, device=win.device)
    out[at] = col
    depth = torch.ones(win.shape, dtype=torch.float64, device=win.device)
    zx, zy, zc, _ = _plane(X, Y, S["D"][s, t])
    depth[at] = (zx * (px / 256.0) + zy * (py / 256.0) + zc).clamp(0.0, 1.0)
    return out.permute(0, 3, 1, 2), depth


def _gradients(nodes, VP, S, win, w, h, light, gout):
    """Gradients of sum(image * gout) with the visible triangles held: colours per node, the
    vertices of all meshes, the light."""
    leaf = lambda a: a.double().clone().requires_grad_(True)  # noqa: E731
    dev, n = VP.device, VP.shape[0]
    verts = [leaf(torch.tensor(np.concatenate(m[0][:2], 1), dtype=torch.float32, device=dev))
             for m in nodes]
    cols = [leaf(m[3]) for m in nodes]
    light = leaf(light)
    at = win >= 0
    s, y, x = at.nonzero(as_tuple=True)
    t = win[at]
    g = gout.permute(0, 2, 3, 1)[at].double()
    total = 0.0
    for j, (mesh, k, M, _, _) in enumerate(nodes):
        m = S["node"][s, t] == j
        sj, tj = s[m], t[m]
        row = sj * k + S["inst"][sj, tj]
        ids = torch.tensor(mesh[2], device=dev)[S["tri"][sj, tj]]
        v = verts[j][ids]                                       # [P, 3, 6]
        Mr = M.double()[row]
        Nw = torch.nn.functional.normalize((Mr[:, None, :3, :3] * v[:, :, None, 3:]).sum(-1), dim=-1)
        normal = Nw[:, 0]
        if bool(S["smooth"][sj[:1], tj[:1]].any()):
            clip = _mul(VP.double()[sj][:, None], _mul(Mr[:, None], v[..., :3]))
            cx = (x[m] + 0.5)[:, None]
            cy = (h - 1 - y[m] + 0.5)[:, None]
            hx = (clip[..., 0] + clip[..., 3]) * (0.5 * w) - cx * clip[..., 3]
            hy = (clip[..., 1] + clip[..., 3]) * (0.5 * h) - cy * clip[..., 3]
            u = torch.stack([hx[:, (i + 1) % 3] * hy[:, (i + 2) % 3]
                             - hx[:, (i + 2) % 3] * hy[:, (i + 1) % 3] for i in range(3)], 1)
            normal = (u[..., None] * Nw).sum(1)
        total = total + (_shade(normal, cols[j][row], light) * g[m]).sum()
    got = torch.autograd.grad(total, [*verts, light, *cols], allow_unused=True)
    got = [torch.zeros_like(p) if q is None else q for p, q in zip([*verts, light, *cols], got)]
    k = len(nodes)
    return torch.cat(got[:k]), got[k], got[k + 1:]


def _cartpole_nodes(case, seed):
    """The CartPole scenes as plain nodes: (mesh, 1, transforms, colours, None) per object."""
    n, state = case["n"], _cartpole_state(case, seed)
    box = _box()

    def placed(scale, pivot, colour, x=0.0, y=0.0, z=0.0, angle=None, mesh=box):
        pos = (mesh[0] - np.array(pivot)) * np.array(scale)
        M = torch.eye(4, device="cuda").repeat(n, 1, 1)
        if angle is not None:
            c, s = torch.cos(angle), torch.sin(angle)
            M[:, 0, 0], M[:, 0, 2], M[:, 2, 0], M[:, 2, 2] = c, s, -s, c
        M[:, 0, 3], M[:, 1, 3], M[:, 2, 3] = x, y, z
        col = torch.as_tensor(colour, dtype=torch.float32, device="cuda").expand(n, 4)
        return (pos, mesh[1], mesh[2]), 1, M, col, None

    x, th = state[:, 0], state[:, 2]
    if case["scene"] == "ground":
        quad = (np.array([(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0)], float),
                np.array([(0, 0, 1)] * 4, float), np.array([(0, 1, 2), (0, 2, 3)]))
        nodes = [placed((10.0, 10.0, 1.0), (0.5, 0.5, 0.0), (0.35, 0.55, 0.3, 1.0), mesh=quad),
                 placed((0.4, 0.2, 0.2), (0.5, 0.5, 0.5), (0.9, 0.3, 0.2, 1.0), x=x, z=0.1),
                 placed((0.05, 0.05, 1.0), (0.5, 0.5, 0.0), (0.95, 0.85, 0.3, 1.0), x=x, z=0.2,
                        angle=th)]
        return nodes, (0.0, -6.0, 1.5), 60.0, [-1.0, -1.0, -2.0, 0.8, 0.8, 0.8, 0.2, 0.2, 0.2, 1.0]
    t = torch.linspace(0.0, 1.0, n, device="cuda")[:, None]
    first, last = (torch.tensor(c, device="cuda") for c in ((0.6, 0.8, 1.0, 1.0),
                                                            (1.0, 0.6, 0.8, 1.0)))
    nodes = [placed((6.0, 0.05, 0.05), (0.5, 0.5, 0.5), (0.2, 0.2, 0.2, 1.0)),
             placed((1.2, 0.8, 0.5), (0.5, 0.5, 0.5), first + (last - first) * t, x=x),
             placed((0.1, 0.1, 2.0), (0.5, 0.5, 0.05), (1.0, 0.7, 0.2, 1.0), x=x, y=0.45, angle=th)]
    return nodes, (5.0, 5.0, 2.0), 55.0, [0.4, -0.6, -0.7, 1.0, 1.0, 1.0, 0.2, 0.2, 0.25, 1.0]


def exact(case, seed):
    kind, n, w, h = case["kind"], case["n"], case["w"], case["h"]
    if kind == "steering" or (case.get("dtype") == "uint8" and kind != "graph"
                              and not case.get("depth")):
        return None  # bytes: equal or not
    if kind in ("step", "graph"):
        nodes, eye, fov, light = _cartpole_nodes(case, seed)
        eye = torch.tensor(eye, device="cuda").expand(n, 3)
    else:
        nodes, eye, strength = _objects(case, seed)
        nodes = [(m, k, _as_uploaded(M), c, cnt) for m, k, M, c, cnt in nodes]
        fov = 55.0
        light = [*LIGHT["dir_dir"], *LIGHT["dir_col"], *LIGHT["ambient"], strength]
    tris = sum(k * len(m[2]) for m, k, *_ in nodes)
    if n * tris * w * h > EXACT_TESTS:
        return None
    light = torch.tensor(light, dtype=torch.float32, device="cuda").double()
    VP = _view_projection(n, w, h, eye, torch.zeros(3, device="cuda"), fov)
    images, depths, grads = [], [], None
    gout = _output_gradient(case, seed) if kind == "grad" else None
    step = max(1, min(n, int(2 ** 22 // max(tris, w * h))))
    for s0 in range(0, n, step):
        s1 = min(n, s0 + step)
        part = [(m, k, M[s0 * k:s1 * k], c[s0 * k:s1 * k], None if cnt is None else cnt[s0:s1])
                for m, k, M, c, cnt in nodes]
        S = _scene(part, VP[s0:s1], w, h)
        win = _visible(S, w, h)
        img, dep = _frames(S, win, w, h, light)
        images.append(img)
        depths.append(dep)
        if gout is not None:
            v, li, cs = _gradients(part, VP[s0:s1], S, win, w, h, light, gout[s0:s1])
            grads = ((v, li, [[c] for c in cs]) if grads is None else
                     (grads[0] + v, grads[1] + li, [a + [c] for a, c in zip(grads[2], cs)]))
    img, dep = torch.cat(images), torch.cat(depths)
    if kind == "grad":
        return {"image": img, "vertices": grads[0], "light": grads[1].cpu(),
                "colors": [torch.cat(c) for c in grads[2]]}
    if kind == "step":
        return img
    pixels = img if case["dtype"] != "uint8" else None
    if kind == "graph" or case.get("depth"):
        return {"pixels": pixels, "depth": dep}
    return {"pixels": pixels}
