"""Performance cases of the package: what its users have it do, through its
public entry points, from a single look-up of a thousand keys to tables of
sixteen million and grids of two hundred thousand blocks.

Ten kinds of work (the "op" of a case); each has a maker of its inputs and a
pass:

  find     look-ups with value rows in a standing HashMap
  set      a HashSet filled anew and asked for members
  map      a HashMap filled anew with value rows and read back by key
  update   a batch enters a standing HashMap, is read back and leaves again,
           and what stays is listed
  embed    HashEmbedding, forward and backward
  forward  SparseDenseGrid interpolation without gradients (rendering, export)
  train    one training pass over a grid: features, their gradient with respect
           to the positions, a loss of both, backward to the embeddings
  fuse     one depth frame integrated into a grid
  rays     near / far and samples of camera rays through a grid
  surface  block table, smoothing and surface mesh of a fused field

Values are float32 throughout, the only type the modules allocate.  Which index
a new key gets is left to the device, so standing tables are restored from a
state dict (as a program resumes from a checkpoint), which fixes it, and a pass
returns nothing that depends on the index of a key it has inserted itself.  The
rays and the fields whose outputs vary in length come from a geometry of the
case; a seed gives their order, the blocks' and the rows.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "torch-ash_amd"))
import ash  # noqa: E402

DEV = torch.device("cuda")
SPARSE = 128  # blocks per axis of the bounded grids


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one query of a few points against a small map (the size of the unit
        # tests): nothing but the latency of a call
        {"name": "find_small", "op": "find", "dim": 3, "stored": 10_000, "n": 1_000},
        # benchmark configuration 1: a million keys, half of them repeated
        {"name": "set_1m", "op": "set", "dim": 3, "n": 1_000_000, "unique": 0.5},
        # benchmark configuration 2, the headline: 16 M voxels with values
        {"name": "map_16m", "op": "map", "dim": 3, "n": 16_000_000},
        # a sliding window over a standing map: an odd batch comes and goes
        {"name": "update_64k", "op": "update", "dim": 3, "stored": 1_000_000, "n": 65_537},
        # trainable rows behind keys, one optimisation pass
        {"name": "embed_200k", "op": "embed", "dim": 3, "stored": 300_000, "n": 200_003, "e": 16},
        # a batch of points out of a small grid, as in an interactive viewer
        {"name": "forward_small", "op": "forward", "blocks": 2_000, "grid": 8, "e": 8, "n": 4_097,
         "rays": True, "interpolation": "linear"},
        # benchmark configuration 3: wide rows, unordered points, a tenth of
        # them outside the active blocks
        {"name": "forward_16ch", "op": "forward", "blocks": 200_000, "grid": 8, "e": 16,
         "n": 4_400_000, "rays": False, "interpolation": "linear"},
        # benchmark configuration 4: samples of 32768 rays, value loss and
        # gradient-norm loss, plain backward()
        {"name": "train_rays", "op": "train", "blocks": 200_000, "grid": 8, "e": 4,
         "n": 4_194_304, "interpolation": "smooth_step", "dense": False},
        # the scene reconstruction demo: rows of distance, colour and weight, a
        # batch of rays, one dense gradient for the whole pass
        {"name": "train_5ch", "op": "train", "blocks": 20_000, "grid": 8, "e": 5, "n": 131_072,
         "interpolation": "smooth_step", "dense": True},
        # benchmark configuration 5 with the demo's rows: a VGA frame with
        # colour, the number of touched blocks read back
        {"name": "fuse_vga", "op": "fuse", "width": 640, "height": 480, "cell": 0.015, "e": 5,
         "count": True},
        # the sampler in front of a training pass over 32768 rays
        {"name": "rays_32k", "op": "rays", "blocks": 200_000, "rays": 32_768, "samples": 128},
        # export after fusion
        {"name": "surface_60k", "op": "surface", "blocks": 60_000, "e": 5, "window": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("find", "set", "map", "update", "embed", "forward", "train", "fuse", "rays",
                     "surface"))
    dim = rng.choice((1, 2, 3, 3, 3, 4))
    if op == "find":
        return {"op": op, "dim": dim, "stored": _log(rng, 1_000, 8_000_000), "n": _log(rng, 100, 8_000_000)}
    if op == "set":
        return {"op": op, "dim": dim, "n": _log(rng, 1_000, 4_000_000), "unique": rng.choice((0.5, 0.9, 1.0))}
    if op == "map":
        return {"op": op, "dim": 3, "n": _log(rng, 1_000, 15_000_000)}
    if op == "update":
        return {"op": op, "dim": dim, "stored": _log(rng, 10_000, 4_000_000), "n": _log(rng, 100, 1_000_000)}
    if op == "embed":
        return {"op": op, "dim": dim, "stored": _log(rng, 1_000, 300_000), "n": _log(rng, 100, 400_000),
                "e": rng.choice((3, 8, 16, 32))}
    if op in ("forward", "train"):
        grid = rng.choice((4, 8, 8, 8, 16))
        e = rng.choice((1, 2, 3, 4, 5, 6, 7, 8, 12, 16))
        cells = 6_000_000 if grid == 16 else 50_000_000   # per grid: keeps a block count in hand
        most = min(200_000, cells // grid**3, 400_000_000 // (grid**3 * e))
        case = {"op": op, "blocks": _log(rng, 500, most), "grid": grid, "e": e,
                "interpolation": rng.choice(("linear", "smooth_step"))}
        if op == "forward":
            case.update(n=_log(rng, 100, 4_000_000), rays=rng.choice((True, False)))
        else:
            case.update(n=_log(rng, 1_000, min(2_000_000, 8_000_000 // e)), dense=rng.choice((True, False)))
        return case
    if op == "fuse":
        return {"op": op, "width": _log(rng, 150, 1_300), "height": _log(rng, 110, 1_000),
                "cell": rng.choice((0.012, 0.015, 0.02, 0.03)), "e": rng.choice((2, 5)),
                "count": rng.choice((True, False))}
    if op == "rays":
        return {"op": op, "blocks": _log(rng, 1_000, 200_000), "rays": _log(rng, 500, 100_000),
                "samples": rng.choice((32, 64, 128))}
    window, e = rng.choice((3, 3, 5, 7)), rng.choice((2, 5))
    return {"op": op, "blocks": _log(rng, 500, min(60_000, 8_100_000 // (e * window**3))), "e": e,
            "window": window}


# --------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV)


def _unit(g, n):
    d = torch.randn(n, 3, generator=g, device=DEV)
    return d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _on_spheres(radii, centres, n, g):
    """n points on the spheres' surfaces, spheres drawn by area."""
    pick = torch.multinomial(radii * radii, n, replacement=True, generator=g)
    return centres[pick] + radii[pick].unsqueeze(1) * _unit(g, n)


# bits per component of a packed key, and the range the keys are drawn from
_BITS = {1: 32, 2: 31, 3: 21, 4: 16}


def _pack(keys):
    b = _BITS[keys.shape[1]]
    code = torch.zeros(keys.shape[0], dtype=torch.int64, device=keys.device)
    for d in range(keys.shape[1]):
        code |= (keys[:, d].long() + (1 << (b - 1))) << (b * d)
    return code


def _unpack(code, dim):
    b = _BITS[dim]
    parts = [((code >> (b * d)) & ((1 << b) - 1)) - (1 << (b - 1)) for d in range(dim)]
    return torch.stack(parts, dim=1).int()


def _distinct_keys(n, dim, g):
    """n distinct keys in random order: surface voxels of spheres in three
    dimensions (benchmark configuration 2), uniform ones otherwise."""
    have = torch.empty(0, dtype=torch.int64, device=DEV)
    if dim == 3:
        radii = _rand(g, 64) * 2.5 + 0.5
        centres = _rand(g, 64, 3) * 40 - 20
    while have.numel() < n:
        m = n - have.numel() + n // 8 + 1024
        if dim == 3:
            keys = torch.floor(_on_spheres(radii, centres, m, g) / 0.01).int()
        else:
            half = {1: 1 << 28, 2: 1 << 16, 4: 1 << 8}[dim]
            keys = torch.randint(-half, half, (m, dim), generator=g, device=DEV, dtype=torch.int32)
        have = torch.unique(torch.cat([have, _pack(keys)]))
    return _unpack(have[torch.randperm(have.numel(), generator=g, device=DEV)[:n]], dim).contiguous()


def _queries(keys, n, hit, g):
    """n keys of which a share `hit` is stored, the others moved out of range."""
    q = keys[torch.randint(keys.shape[0], (n,), generator=g, device=DEV)]
    away = {1: 1 << 29, 2: 1 << 18, 3: 100_000, 4: 1 << 10}[keys.shape[1]]
    q[:, 0] += (_rand(g, n) >= hit).int() * away
    return q.contiguous()


def _restore(engine, keys):
    """Key i under index i, through the engine's state dict."""
    n, cap = keys.shape[0], engine.capacity
    state = {
        "_heap": torch.arange(cap, dtype=torch.int32, device=DEV),
        "_keys": torch.zeros(cap, engine.dim, dtype=torch.int32, device=DEV),
        "_indices": torch.zeros(cap, dtype=torch.int64, device=DEV),
        "_size": torch.tensor([n], dtype=torch.int32, device=DEV),
    }
    state["_keys"][:n] = keys
    state["_indices"][:n] = torch.arange(n, device=DEV)
    engine.load_state_dict(state)


def _standing_map(keys, capacity, g):
    """A HashMap that holds `keys` with a colour and the caller's own number of
    each (below 2^24: exact in float32)."""
    m = ash.HashMap(keys.shape[1], {"color": 3, "id": 1}, capacity, DEV)
    _restore(m.engine, keys)
    n = keys.shape[0]
    m.values["color"][:n] = _rand(g, n, 3)
    m.values["id"][:n] = torch.arange(n, device=DEV).float().unsqueeze(1)
    return m


def _surface_blocks(n, g, order):
    """n block coordinates around spheres, each surface block with its +1
    neighbours, in a random order by the generator `order`; the spheres' radii
    and centres (blocks)."""
    r_mean = min(math.sqrt(max(n, 64) / (256 * 4 * math.pi)) * 1.9, SPARSE * 0.22)
    have = torch.empty(0, dtype=torch.int64, device=DEV)
    corner = torch.tensor([[(c >> d) & 1 for d in range(3)] for c in range(8)], device=DEV)
    radii_all, centres_all = [], []
    while have.numel() < n:
        radii = (_rand(g, 8) * 0.8 + 0.6) * r_mean
        room = SPARSE - 2 * (radii.unsqueeze(1) + 2)
        centres = _rand(g, 8, 3) * room + radii.unsqueeze(1) + 2
        points = _on_spheres(radii, centres, int(480 * (1.4 * r_mean) ** 2) + 512, g)
        blocks = torch.floor(points).long().clamp_(0, SPARSE - 2)
        have = torch.unique(torch.cat([have, _pack((blocks.view(-1, 1, 3) + corner).view(-1, 3))]))
        radii_all.append(radii)
        centres_all.append(centres)
    have = have[:n]
    coords = _unpack(have[torch.randperm(n, generator=order, device=DEV)], 3).contiguous()
    return coords, torch.cat(radii_all), torch.cat(centres_all)


def _grid(case, g, e, geometry=None):
    """A bounded grid over the unit cube with the case's blocks active; the
    spheres its blocks surround, in world units."""
    coords, radii, centres = _surface_blocks(case["blocks"], geometry or g, g)
    grid = ash.BoundedSparseDenseGrid(
        3, case["blocks"], e, grid_dim=case.get("grid", 8), sparse_grid_dim=SPARSE,
        bbox_min=torch.zeros(3), bbox_max=torch.ones(3), device=DEV)
    _restore(grid.engine, coords)
    with torch.no_grad():
        grid.embeddings.normal_(std=0.01, generator=g)
    grid.construct_grid_neighbor_lut_(radius=1, bidirectional=False)
    unit = grid.grid_dim * grid.cell_size
    return grid, coords, radii * unit, centres * unit


def _ray_positions(grid, radii, centres, n, g):
    """n positions in ray order: 128 stratified samples per ray in a band of
    twelve cells around a sphere's surface."""
    rays = -(-n // 128)
    target, d = _on_spheres(radii, centres, rays, g), _unit(g, rays)
    t = (torch.arange(128, device=DEV) + _rand(g, rays, 128)) / 64 - 1
    x = target.view(-1, 1, 3) + (t * (12 * grid.cell_size)).unsqueeze(-1) * d.view(-1, 1, 3)
    return x.view(-1, 3)[:n].contiguous()


def _uniform_positions(grid, coords, n, g):
    """n positions in no order, ten in eleven inside active blocks."""
    inside = int(n / 1.1)
    pick = torch.randint(coords.shape[0], (inside,), generator=g, device=DEV)
    a = (coords[pick] + _rand(g, inside, 3)) * grid.grid_dim
    b = _rand(g, n - inside, 3) * (SPARSE * grid.grid_dim - 1)
    cells = torch.cat([a, b])[torch.randperm(n, generator=g, device=DEV)]
    return grid.transform_cell_to_world(cells).contiguous()


def _frame(case, radii, centres, turn, g):
    """A camera on an orbit of 3 m around the spheres: unprojected points in
    image order, depth, colour, extrinsic, intrinsic."""
    w, h = case["width"], case["height"]
    k = torch.tensor([[525.0 * w / 640, 0, (w - 1) / 2], [0, 525.0 * h / 480, (h - 1) / 2], [0, 0, 1]],
                     device=DEV)
    eye = torch.tensor([3 * math.cos(turn), 0.6 * math.sin(2 * turn), 3 * math.sin(turn)], device=DEV)
    fwd = -eye / eye.norm()
    right = torch.linalg.cross(torch.tensor([0.0, 1.0, 0.0], device=DEV), fwd)
    right = right / right.norm()
    rot = torch.stack([right, torch.linalg.cross(fwd, right), fwd])
    ext = torch.eye(4, device=DEV)
    ext[:3, :3], ext[:3, 3] = rot, -rot @ eye
    v, u = torch.meshgrid(torch.arange(h, device=DEV), torch.arange(w, device=DEV), indexing="ij")
    d = torch.stack([(u - k[0, 2]) / k[0, 0], (v - k[1, 2]) / k[1, 1], torch.ones_like(u).float()], -1)
    d = d.view(-1, 3) @ rot
    a, best = (d * d).sum(-1), torch.full((h * w,), float("inf"), device=DEV)
    for r, c in zip(radii, centres):
        oc = eye - c
        b = d @ oc
        disc = b * b - a * ((oc * oc).sum() - r * r)
        s = (-b - disc.clamp_min(0).sqrt()) / a
        best = torch.minimum(best, torch.where((disc > 0) & (s > 0), s, best))
    depth = torch.where(best < 6.0, best, torch.zeros_like(best))
    points = eye + depth.unsqueeze(1) * d
    return points[depth > 0].contiguous(), depth.view(h, w), _rand(g, h, w, 3), ext, k


# -------------------------------------------------------------------- prepare
def _prepare_find(case, g):
    keys = _distinct_keys(case["stored"], case["dim"], g)
    return {"map": _standing_map(keys, int(1.5 * case["stored"]), g),
            "queries": _queries(keys, case["n"], 0.7, g)}


def _prepare_set(case, g):
    n, dim = case["n"], case["dim"]
    base = _distinct_keys(max(1, int(n * case["unique"])), dim, g)
    keys = torch.cat([base, base[torch.randint(len(base), (n - len(base),), generator=g, device=DEV)]])
    return {"set": ash.HashSet(dim, 2 * n, DEV),
            "keys": keys[torch.randperm(n, generator=g, device=DEV)].contiguous(),
            "queries": _queries(base, n, 0.5, g)}


def _prepare_map(case, g):
    n = case["n"]
    keys = _distinct_keys(n, case["dim"], g)
    return {"map": ash.HashMap(case["dim"], {"color": 3, "id": 1}, int(1.5 * n), DEV), "keys": keys,
            "values": {"color": _rand(g, n, 3), "id": torch.arange(n, device=DEV).float().unsqueeze(1)},
            "queries": _queries(keys, n, 1.0, g)}


def _prepare_update(case, g):
    stored, n = case["stored"], case["n"]
    keys = _distinct_keys(stored + n, case["dim"], g)
    new = keys[stored:].contiguous()
    return {"map": _standing_map(keys[:stored], int(1.5 * (stored + n)), g), "new": new,
            "values": {"color": _rand(g, n, 3), "id": torch.arange(n, device=DEV).float().unsqueeze(1)},
            # half of the queries go to the newcomers, which are gone at the second asking
            "queries": torch.cat([_queries(new, n - n // 2, 1.0, g), _queries(keys[:stored], n // 2, 1.0, g)])}


def _prepare_embed(case, g):
    keys = _distinct_keys(case["stored"], case["dim"], g)
    table = ash.HashEmbedding(case["dim"], int(1.25 * case["stored"]), case["e"], DEV)
    _restore(table.engine, keys)
    with torch.no_grad():
        table.embedding.normal_(generator=g)
    return {"table": table, "queries": _queries(keys, case["n"], 0.9, g),
            "z": torch.randn(case["n"], case["e"], generator=g, device=DEV)}


def _prepare_forward(case, g):
    grid, coords, radii, centres = _grid(case, g, case["e"])
    x = (_ray_positions(grid, radii, centres, case["n"], g) if case["rays"]
         else _uniform_positions(grid, coords, case["n"], g))
    return {"grid": grid, "x": x, "interpolation": case["interpolation"]}


def _prepare_train(case, g):
    grid, _, radii, centres = _grid(case, g, case["e"])
    x = _ray_positions(grid, radii, centres, case["n"], g)
    return {"grid": grid, "x": x.requires_grad_(True), "interpolation": case["interpolation"],
            "dense": case["dense"]}


def _prepare_fuse(case, g):
    radii, centres = _rand(g, 48) * 0.35 + 0.1, (_rand(g, 48, 3) * 2 - 1) * 1.2
    turn = float(_rand(g, 1)) * 2 * math.pi
    points, depth, color, ext, k = _frame(case, radii, centres, turn, g)
    beside = _frame(case, radii, centres, turn + 0.5, g)[0]
    # the map stands already: the blocks of this view and of one beside it
    seen = ash.UnBoundedSparseDenseGrid(3, 1 << 18, 1, 1, cell_size=8 * case["cell"], device=DEV)
    blocks = seen.spatial_init_(torch.cat([points, beside]), dilation=1, bidirectional=True)[0]
    packed = torch.sort(_pack(blocks.view(-1, 3)))[0]
    coords = _unpack(packed[torch.randperm(packed.numel(), generator=g, device=DEV)], 3)
    grid = ash.UnBoundedSparseDenseGrid(3, max(80_000, int(1.25 * len(coords))), case["e"], 8,
                                        cell_size=case["cell"], device=DEV)
    _restore(grid.engine, coords)
    with torch.no_grad():
        e = grid.embeddings
        e[..., :-1].uniform_(0, 0.04, generator=g)
        e[..., -1:] = torch.randint(0, 9, e[..., -1:].shape, generator=g, device=DEV).float()
    return {"grid": grid, "points": points, "depth": depth, "color": color if case["e"] == 5 else None,
            "ext": ext, "k": k, "count": case["count"]}


def _prepare_rays(case, g):
    geometry, n = _gen(1), case["rays"]
    grid, _, radii, centres = _grid(case, g, 1, geometry)
    origin = 0.05 + 0.9 * _rand(geometry, n, 3)
    d = _on_spheres(radii, centres, n, geometry) - origin
    order = torch.randperm(n, generator=g, device=DEV)
    origin, d = origin[order], d[order]
    # a step of half a block for the coarse march; samples of about two cells
    return {"grid": grid, "o": origin, "d": (d / d.norm(dim=1, keepdim=True).clamp_min(1e-6)).contiguous(),
            "t_step": 4 * grid.cell_size, "samples": case["samples"]}


def _prepare_surface(case, g):
    grid, coords, radii, centres = _grid(case, g, case["e"], _gen(1))
    field = torch.full(grid.embeddings.shape[:2], float("inf"), device=DEV)
    for s in range(0, len(coords), 65_536):
        world = grid.cell_to_world(coords[s:s + 65_536].view(-1, 1, 3), grid.cell_coords.view(1, -1, 3))
        part = field[s:s + 65_536].view(-1)
        for r, c in zip(radii, centres):
            torch.minimum(part, (world - c).norm(dim=1) - r, out=part)
    with torch.no_grad():
        # row i belongs to coords[i] (see _restore)
        grid.embeddings.uniform_(0, 1, generator=g)
        grid.embeddings[..., 0] = field
        grid.embeddings[..., -1] += 1.0
    w = torch.exp(-torch.linspace(-1.5, 1.5, case["window"], device=DEV).square())
    w = (w.view(-1, 1, 1) * w.view(1, -1, 1) * w.view(1, 1, -1)).unsqueeze(-1)
    return {"grid": grid, "window": (w / w.sum()).repeat(1, 1, 1, case["e"]).contiguous()}


def prepare(case, seed):
    state = globals()["_prepare_" + case["op"]](case, _gen(seed))
    state["op"] = case["op"]
    return state


# ------------------------------------------------------------------------ run
def _run_find(s):
    return s["map"].find(s["queries"], return_values=True)


def _run_set(s):
    t = s["set"]
    t.clear()
    t.insert(s["keys"])
    return t.find(s["queries"]), t.size()


def _run_map(s):
    m = s["map"]
    m.clear()
    m.insert(s["keys"], s["values"])
    return m.find(s["queries"], return_indices=False, return_values=True), m.size()


def _run_update(s):
    m = s["map"]
    m.insert(s["new"], s["values"])
    read = m.find(s["queries"], return_indices=False, return_values=True)
    m.erase(s["new"])
    stays = m.find(s["queries"])[0]
    # the listing comes in an order of its own: filed by index
    keys, indices, values = m.items(return_indices=True, return_values=True)
    rows = torch.empty_like(keys), torch.empty_like(values["color"])
    rows[0][indices], rows[1][indices] = keys, values["color"]
    return read, stays, rows


def _run_embed(s):
    t = s["table"]
    t.embedding.grad = None
    y = t(s["queries"])
    y.backward(s["z"])
    return y, t.embedding.grad


def _run_forward(s):
    with torch.no_grad():
        return s["grid"](s["x"], s["interpolation"])


def _run_train(s):
    grid, x = s["grid"], s["x"]
    grid.embeddings.grad = None
    y, masks = grid(x, s["interpolation"])
    (gx,) = torch.autograd.grad(y[:, 0].sum(), x, create_graph=True)
    loss = (y**2).mean() + (gx.norm(dim=-1) - 1).abs().mean()
    x.grad = None
    if s["dense"]:
        with ash.dense_grad(grid):
            loss.backward()
    else:
        loss.backward()
    return y, masks, gx, loss, x.grad, grid.embeddings.grad


def _run_fuse(s):
    grid = s["grid"]
    count = ash.fusion.fuse_frame(grid, s["points"], s["depth"], s["k"], s["ext"], 0.04, 6.0, s["color"],
                                  count_blocks=s["count"])
    return count, grid.embeddings


def _run_rays(s):
    grid = s["grid"]
    near, far = grid.ray_find_near_far(s["o"], s["d"], 0.0, 2.0, s["t_step"])
    return near, far, grid.ray_sample(s["o"], s["d"], near, far, s["samples"])


def _run_surface(s):
    grid = s["grid"]
    # blocks were activated since the last export: the table is rebuilt
    grid.construct_grid_neighbor_lut_(radius=1, bidirectional=False)
    with torch.no_grad():
        smooth = grid.convolution(grid.embeddings, s["window"])
        return smooth, grid.surface_mesh(smooth[..., 0], smooth[..., -1], weight_thr=0.5)


def run(state):
    return globals()["_run_" + state["op"]](state)


# ----------------------------------------------------------------------- work
def _rows_met(case):
    """Cells whose rows the queries of a grid need: eight corners each, shared
    between neighbouring samples of a ray."""
    cells = case["blocks"] * case.get("grid", 8) ** 3
    met = case["n"] * (8 if not case.get("rays", True) else 0.9)
    return cells * -math.expm1(-met / cells)


def work(case):
    """Keys and positions in, results out, value and embedding rows that are
    needed once each; an entry of a table counts as its key and its index."""
    op, n = case["op"], case.get("n", 0)
    entry = 4 * case.get("dim", 3) + 4
    key = 4 * case.get("dim", 3)
    flops = 0
    if op == "find":
        size = n * (key + entry + 8 + 1) + n * 2 * 16
    elif op == "set":
        size = 2 * n * key + 2 * n * case["unique"] * entry + n
    elif op == "map":
        # rows into the map, and out of it
        size = n * (2 * key + 2 * entry + 1 + 4 * 16)
    elif op == "update":
        # the same, the erase, the second find, and the listing filed
        size = n * (4 * key + 4 * entry + 2 + 4 * 16) + case["stored"] * (2 * key + 8 + 16 + 12)
    elif op == "embed":
        size = n * (key + entry + 1 + 3 * 4 * case["e"]) + int(1.25 * case["stored"]) * 4 * case["e"]
    elif op == "forward":
        e = case["e"]
        size = n * (12 + 4 * e + 1) + _rows_met(case) * 4 * e
        flops = n * (16 * e + 40)
    elif op == "train":
        e = case["e"]
        size = n * (12 + 4 * e + 1 + 24) + _rows_met(case) * 4 * e + case["blocks"] * case["grid"] ** 3 * 4 * e
        flops = n * 4 * (16 * e + 60)
    elif op == "fuse":
        pixels = case["width"] * case["height"]
        blocks = 1.1 / case["cell"] ** 2
        size = pixels * (4 + 4 + (12 if case["e"] == 5 else 0)) + blocks * 512 * 8 * case["e"]
        flops = blocks * 512 * 40
    elif op == "rays":
        size = case["rays"] * (24 + 16 + 8 + 16 * case["samples"] / 4) + case["blocks"] * entry
    else:
        cells = case["blocks"] * 512
        size = cells * case["e"] * 8 + case["blocks"] * (entry + 8 * 8) + cells * 8
        flops = 2 * cells * case["e"] * case["window"] ** 3
    return {"bytes": float(size), "flops": float(flops)}


def tolerance(case):
    """Look-ups move bytes; everything else is float32 arithmetic whose sums
    may be taken in another order."""
    if case["op"] in ("find", "set", "map", "update"):
        return "exact"
    return {"rel": 1e-5}
