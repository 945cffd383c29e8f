"""Workloads of the PACK3D attention layer, through its public entry points.

Four kinds of work:

* ``infer``  -- ``PACK3DAttention`` without gradients,
* ``train``  -- the same layer, forward and backward to the input and to every
  parameter,
* ``graph``  -- ``pack3d_hip``, forward and backward, on the neighbour graph of
  a masked volume (an ellipsoid of occupied voxels), which is no complete grid,
* ``layout`` -- ``build_layout``, ``TokenLayout.repack`` to a random token order
  and ``prepare_geometry`` on the packed tables.

Grids are (z, y, x) voxels, blocks and radii (z, y, x) as well.
"""
from __future__ import annotations

import math
from contextlib import nullcontext

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import pack3d_amd as p3d

DEVICE = "cuda:0"
TYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16, "autocast": torch.float32}


def _layer_case(name, kind, grid, block, radius, *, order="raster", batch=1, dim, heads, kv_heads, head_dim,
                pool, dtype):
    case = {"kind": kind, "z": grid[0], "y": grid[1], "x": grid[2], "bz": block[0], "by": block[1], "bx": block[2],
            "rz": radius[0], "ry": radius[1], "rx": radius[2], "order": order, "batch": batch, "dim": dim,
            "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "pool": pool, "dtype": dtype}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest call: one 4,096-token block of a small model, where launches and host work count.
        _layer_case("infer_small", "infer", (16, 16, 16), (2, 2, 2), (1, 1, 1), order="morton", dim=64, heads=4,
                    kv_heads=2, head_dim=16, pool=4, dtype="bf16"),
        # Two volumes of 65,536 tokens served as one batch.
        _layer_case("infer_batch", "infer", (16, 64, 64), (4, 4, 4), (2, 2, 2), batch=2, dim=192, heads=4, kv_heads=4,
                    head_dim=48, pool=1, dtype="bf16"),
        # The largest volume served in one call: 64^3 tokens, radius 2.
        _layer_case("infer_large", "infer", (64, 64, 64), (4, 4, 4), (2, 2, 2), dim=192, heads=4, kv_heads=4,
                    head_dim=48, pool=1, dtype="bf16"),
        # A wide fp16 layer on tokens that the surrounding program keeps in an order of its own.
        _layer_case("infer_fp16_repacked", "infer", (16, 64, 64), (1, 4, 4), (1, 1, 1), order="random", dim=512,
                    heads=8, kv_heads=2, head_dim=64, pool=16, dtype="fp16"),
        # An fp32 model served under bf16 autocast.
        _layer_case("infer_autocast", "infer", (16, 64, 64), (1, 4, 4), (1, 1, 1), dim=512, heads=8, kv_heads=2,
                    head_dim=64, pool=16, dtype="autocast"),
        # The smallest training step.
        _layer_case("train_small", "train", (16, 16, 16), (2, 2, 2), (1, 1, 1), order="morton", dim=64, heads=4,
                    kv_heads=2, head_dim=16, pool=4, dtype="bf16"),
        # Training on a stack of image slices: a neighbourhood within the slice only.
        _layer_case("train_slices", "train", (1, 128, 128), (1, 4, 4), (0, 1, 1), batch=2, dim=512, heads=8,
                    kv_heads=2, head_dim=64, pool=16, dtype="bf16"),
        # Training with the widest heads.
        _layer_case("train_wide_heads", "train", (16, 32, 32), (4, 4, 4), (1, 1, 1), order="morton", dim=512, heads=4,
                    kv_heads=2, head_dim=128, pool=1, dtype="bf16"),
        # Training in full fp32 on a ragged volume (27-slot blocks, 693 summaries).
        _layer_case("train_fp32_ragged", "train", (21, 27, 33), (3, 3, 3), (2, 2, 2), dim=192, heads=4, kv_heads=4,
                    head_dim=48, pool=1, dtype="fp32"),
        # The largest training step: 262,144 tokens under bf16 autocast.
        _layer_case("train_large", "train", (32, 128, 64), (4, 4, 4), (2, 2, 2), dim=192, heads=4, kv_heads=4,
                    head_dim=48, pool=1, dtype="autocast"),
        # A masked volume: a custom graph of about 32,000 occupied voxels, forward and backward of the core.
        _layer_case("train_masked_graph", "graph", (32, 48, 40), (1, 4, 4), (1, 1, 1), dim=0, heads=8, kv_heads=2,
                    head_dim=64, pool=16, dtype="bf16"),
        # A program that sets its geometry up: a new volume shape, a token order of its own, a table from elsewhere.
        _layer_case("layout_setup", "layout", (32, 64, 64), (4, 4, 4), (2, 2, 2), order="morton", dim=0, heads=0,
                    kv_heads=0, head_dim=0, pool=1, dtype="int"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["infer", "infer", "infer", "train", "train", "train", "graph", "layout"])
    while True:
        block = rng.choice([(2, 2, 2), (1, 4, 4), (3, 3, 3), (4, 4, 4), (2, 4, 4), (1, 8, 8), (4, 2, 3)])
        tokens = _log_int(rng, 1024, 131072)
        # Block counts per axis: a volume of about `tokens` with sides up to a factor of 2 apart.
        side = (tokens / 3.0) ** (1.0 / 3.0)
        flat = block[0] == 1 and kind != "graph" and rng.random() < 0.25
        if flat:
            area = math.sqrt(tokens / 2)
            counts = (1, max(1, round(area * rng.uniform(0.7, 1.4) / block[1])), max(1, round(area / block[2])))
        else:
            counts = tuple(max(1, round(side * rng.uniform(0.8, 2.0) / b)) for b in block)
        grid = tuple(c * b for c, b in zip(counts, block))
        n = math.prod(grid)
        radius = (0, 1, 1) if flat else rng.choice([(1, 1, 1), (1, 1, 1), (2, 2, 2), (1, 2, 1)])
        pool = rng.choice([1, 2, 4, 16])
        order = rng.choice(["raster", "morton", "random"])
        batch = rng.choice([1, 1, 2, 3]) if n <= 32768 else 1
        heads, kv_heads = rng.choice([(4, 4), (4, 2), (8, 2), (2, 1)])
        head_dim = rng.choice([16, 32, 48, 64, 128])
        dim = rng.choice([64, 96, 128, 192, 256, 320, 384, 512])
        dtype = rng.choice(["bf16", "bf16", "fp16", "autocast", "fp32"])
        if kind == "graph":
            order, dim, batch = "raster", 0, 1
            dtype = "bf16" if dtype == "autocast" else dtype
        if kind == "layout":
            heads = kv_heads = head_dim = dim = 0
            order, batch, dtype = "morton", 1, "int"
            if n < 1000 or n > 140000:
                continue
        else:
            summaries = math.ceil(math.prod(counts) / pool)
            scores = batch * heads * n * summaries * head_dim
            limit = 1e11 / (12 if dtype == "fp32" else 1) / (3 if kind != "infer" else 1)
            wide = batch * heads * n * head_dim
            if n < 500 or n > 140000 or scores > limit or wide > 1.0e8:
                continue
            if summaries < 2:
                continue
        return _layer_case(None, kind, grid, block, radius, order=order, batch=batch, dim=dim, heads=heads,
                           kv_heads=kv_heads, head_dim=head_dim, pool=pool, dtype=dtype)


# ---------------------------------------------------------------- inputs

def _grid(case):
    return (case["z"], case["y"], case["x"])


def _block(case):
    return (case["bz"], case["by"], case["bx"])


def _radius(case):
    return (case["rz"], case["ry"], case["rx"])


def _volume(case):
    return math.prod(_block(case))


def _parameters(case, seed):
    """The layer's parameters by name, on the CPU in fp32: Xavier weights as a
    trained projection's scale, a learned scorer and bias, LayerNorm near one."""
    gen = torch.Generator().manual_seed(2 * seed + 1)
    dim, h, g, d = case["dim"], case["heads"], case["kv_heads"], case["head_dim"]

    def xavier(rows, cols):
        bound = math.sqrt(6.0 / (rows + cols))
        return (torch.rand(rows, cols, generator=gen) * 2 - 1) * bound

    def normal(count, scale, mean=0.0):
        return mean + scale * torch.randn(count, generator=gen)

    return {"pool_weight": normal(d, 0.5 / math.sqrt(d)), "slot_bias": normal(_volume(case), 0.1),
            "local_scale": normal(d, 0.1, 1.0), "global_scale": normal(d, 0.05, 0.25),
            "norm.weight": normal(dim, 0.1, 1.0), "norm.bias": normal(dim, 0.1), "to_q.weight": xavier(h * d, dim),
            "to_kv.weight": xavier(4 * g * d, dim), "gate.weight": xavier(2 * h, dim), "gate.bias": normal(2 * h, 0.1),
            "to_out.weight": xavier(dim, h * d)}


def _activations(case, seed):
    """x and the upstream gradient, [batch, tokens, dim] in the model's type."""
    gen = torch.Generator(device=DEVICE).manual_seed(2 * seed)
    shape = (case["batch"], math.prod(_grid(case)), case["dim"])
    dt = TYPES[case["dtype"]]
    x = torch.randn(shape, generator=gen, device=DEVICE).to(dt)
    dy = torch.randn(shape, generator=gen, device=DEVICE).to(dt) if case["kind"] == "train" else None
    return x, dy


def _permutation(case, seed):
    n = math.prod(_grid(case))
    return torch.from_numpy(np.random.default_rng(seed).permutation(n))


def _build_layout(case):
    kind = "raster_block" if case["order"] == "raster" else "native_block_morton"
    return p3d.build_layout(_grid(case), _block(case), radius=_radius(case), pool_size=case["pool"], layout=kind,
                            device=DEVICE)


def _masked_tables(case):
    """(neighbours [N, W], blocks [F, V]) of the voxels inside the ellipsoid
    that fills the grid, numbered in raster order; absent entries are -1."""
    grid, block, radius = _grid(case), _block(case), _radius(case)
    axes = [(np.arange(s) + 0.5) / s * 2 - 1 for s in grid]
    inside = axes[0][:, None, None] ** 2 + axes[1][None, :, None] ** 2 + axes[2][None, None, :] ** 2 <= 1.0
    index = np.full(grid, -1, np.int64)
    index[inside] = np.arange(int(inside.sum()))
    coords = np.argwhere(inside)
    pad = np.full([s + 2 * r for s, r in zip(grid, radius)], -1, np.int64)
    pad[tuple(slice(r, r + s) for s, r in zip(grid, radius))] = index
    offsets = np.stack(np.meshgrid(*[np.arange(2 * r + 1) for r in radius], indexing="ij"), -1).reshape(-1, 3)
    neighbors = np.stack([pad[tuple((coords + off).T)] for off in offsets], 1)
    cells = [s // b for s, b in zip(grid, block)]
    blocks = index.reshape(cells[0], block[0], cells[1], block[1], cells[2], block[2])
    blocks = blocks.transpose(0, 2, 4, 1, 3, 5).reshape(math.prod(cells), -1)
    blocks = blocks[(blocks >= 0).any(1)]
    return torch.from_numpy(neighbors), torch.from_numpy(np.ascontiguousarray(blocks))


def _graph_inputs(case, n, seed):
    """q, kl, vl, kg, vg (rotated keys as a caller has them), scorer weight,
    slot bias, gate, and the two branch scales; and the upstream gradient."""
    gen = torch.Generator(device=DEVICE).manual_seed(2 * seed)
    b, h, g, d, dt = case["batch"], case["heads"], case["kv_heads"], case["head_dim"], TYPES[case["dtype"]]

    def normal(*shape, scale=1.0, mean=0.0):
        return mean + scale * torch.randn(shape, generator=gen, device=DEVICE)

    inputs = [normal(b, h, n, d)] + [normal(b, g, n, d) for _ in range(4)]
    inputs = [t.to(dt) for t in inputs]
    inputs += [normal(d, scale=0.5 / math.sqrt(d)), normal(_volume(case), scale=0.1), normal(b, h, n).sigmoid(),
               normal(d, scale=0.1, mean=1.0).to(dt), normal(d, scale=0.05, mean=0.25).to(dt)]
    return inputs, normal(b, h, n, d).to(dt)


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case, "kind": kind}
    if kind == "layout":
        state["permutation"] = _permutation(case, seed).to(DEVICE)
        return state
    if kind == "graph":
        neighbors, blocks = _masked_tables(case)
        state["geometry"] = p3d.prepare_geometry(neighbors.to(DEVICE), blocks.to(DEVICE), case["pool"])
        inputs, dy = _graph_inputs(case, neighbors.shape[0], seed)
        state["inputs"], state["dy"] = [t.requires_grad_() for t in inputs], dy
        return state
    layout = _build_layout(case)
    if case["order"] == "random":
        layout = layout.repack(_permutation(case, seed))
    layer = p3d.PACK3DAttention(case["dim"], heads=case["heads"], kv_heads=case["kv_heads"],
                                head_dim=case["head_dim"], block_volume=_volume(case))
    layer.load_state_dict(_parameters(case, seed))
    state["layer"] = layer.to(DEVICE, TYPES[case["dtype"]])
    state["layout"] = layout
    x, state["dy"] = _activations(case, seed)
    state["x"] = x.requires_grad_(kind == "train")
    return state


def _layer_call(state):
    amp = torch.autocast("cuda", torch.bfloat16) if state["case"]["dtype"] == "autocast" else nullcontext()
    with amp:
        return state["layer"](state["x"], state["layout"])


def _tables(geometry):
    return {"neighbors": geometry.neighbors, "reverse_neighbors": geometry.reverse_neighbors,
            "blocks": geometry.blocks}


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            return _layer_call(state)
    if kind == "train":
        layer, x = state["layer"], state["x"]
        layer.zero_grad(set_to_none=True)
        x.grad = None
        y = _layer_call(state)
        y.backward(state["dy"])
        return {"y": y.detach(), "dx": x.grad, **{name: p.grad for name, p in layer.named_parameters()}}
    if kind == "graph":
        inputs = state["inputs"]
        y = p3d.pack3d_hip(*inputs, state["geometry"])
        grads = torch.autograd.grad(y, inputs, state["dy"])
        return [y.detach(), *grads]
    layout = _build_layout(state["case"])
    moved = layout.repack(state["permutation"])
    checked = p3d.prepare_geometry(moved.geometry.neighbors, moved.geometry.blocks, state["case"]["pool"])
    return {"built": {"order": layout.order, "coords": layout.coords, **_tables(layout.geometry)},
            "moved": {"order": moved.order, "coords": moved.coords, **_tables(moved.geometry)},
            "checked": _tables(checked)}


# ------------------------------------------------------------------ work

def _edges(case):
    """Valid neighbour entries of one volume."""
    total = 1
    for s, r in zip(_grid(case), _radius(case)):
        total *= sum(min(s - 1, i + r) - max(0, i - r) + 1 for i in range(s))
    return total


def work(case):
    n = math.prod(_grid(case))
    width = math.prod(2 * r + 1 for r in _radius(case))
    if case["kind"] == "layout":
        degree = math.prod(min(2 * r + 1, s) for s, r in zip(_grid(case), _radius(case)))
        tables = 4 * n * (width + degree + 1)
        # Built, moved (its permutation read) and checked: each output written once; order and coordinates twice.
        return {"bytes": 3 * tables + 2 * 32 * n + 8 * n, "flops": 0}
    b, h, g, d, dim = case["batch"], case["heads"], case["kv_heads"], case["head_dim"], case["dim"]
    size = torch.empty((), dtype=TYPES[case["dtype"]]).element_size()
    edges = _edges(case)
    if case["kind"] == "graph":
        neighbors, blocks = _masked_tables(case)
        n, fine = neighbors.shape[0], blocks.shape[0]
        edges = int((neighbors >= 0).sum())
    else:
        fine = n // _volume(case)
    m = math.ceil(fine / case["pool"])
    core = 4 * b * h * d * (n * m + edges)
    if case["kind"] == "graph":
        tensors = b * n * d * (h + 4 * g)
        moved = 2 * size * tensors + 2 * size * b * h * n * d + 2 * 4 * b * h * n + 4 * n * width * 2 + 4 * n
        # The backward recomputes the scores: five products of the forward's two.
        return {"bytes": moved, "flops": core * 7 // 2}
    weights = dim * (2 * h * d + 4 * g * d + 2 * h)
    linear = 2 * b * n * weights
    if case["kind"] == "infer":
        return {"bytes": size * (2 * b * n * dim + weights), "flops": linear + core}
    return {"bytes": size * (4 * b * n * dim + 2 * weights), "flops": 3 * linear + core * 7 // 2}


def tolerance(case):
    # About four times the distance from 64-bit results: a layer's output (with its residual) lies 2e-3 (bf16),
    # 2.8e-4 (fp16) and 2e-7 (fp32) from them, gradients of the parameters, which sum over all tokens, up to
    # 1e-2, 1e-3 and 2e-6.
    if case["kind"] == "layout":
        return "exact"
    kind = "bf16" if case["dtype"] == "autocast" else case["dtype"]
    if case["kind"] == "infer":
        return {"rel": {"fp32": 1e-6, "bf16": 8e-3, "fp16": 1.2e-3}[kind]}
    return {"rel": {"fp32": 1e-5, "bf16": 3e-2, "fp16": 4e-3}[kind]}


# ----------------------------------------------------------------- exact

def _morton(coords):
    code = torch.zeros(coords.shape[:-1], dtype=torch.int64)
    for bit in range(int(coords.max()).bit_length()):
        for axis in range(3):
            code |= ((coords[..., axis] >> bit) & 1) << (3 * bit + axis)
    return code


def _grid_order(case):
    """(raster index of each row, blocks [F, V] of rows) of the built layout."""
    grid, block = torch.tensor(_grid(case)), torch.tensor(_block(case))
    n = math.prod(_grid(case))
    order = torch.arange(n)
    if case["order"] != "raster":
        coords = _coordinates(case)
        slot = _morton(coords % block)
        order = (_morton(coords // block) * (int(slot.max()) + 1) + slot).argsort()
    return order, torch.arange(n).view(-1, _volume(case))


def _coordinates(case):
    return torch.stack(torch.meshgrid(*[torch.arange(s) for s in _grid(case)], indexing="ij"), -1).reshape(-1, 3)


def _stencil(case, order):
    """Neighbour rows [N, W] of each row, -1 outside the grid."""
    grid, radius = _grid(case), _radius(case)
    row_of = torch.empty_like(order)
    row_of[order] = torch.arange(order.numel(), device=order.device)
    raster = torch.full([s + 2 * r for s, r in zip(grid, radius)], -1, dtype=torch.int64, device=order.device)
    raster[tuple(slice(r, r + s) for s, r in zip(grid, radius))] = row_of.view(grid)
    coords = _coordinates(case).to(order.device)[order]
    columns = []
    for dz in range(2 * radius[0] + 1):
        for dy in range(2 * radius[1] + 1):
            for dx in range(2 * radius[2] + 1):
                columns.append(raster[coords[:, 0] + dz, coords[:, 1] + dy, coords[:, 2] + dx])
    return torch.stack(columns, 1), coords


def _reverse(neighbors):
    """Rows that list row j, ascending, padded with -1."""
    n, width = neighbors.shape
    valid = neighbors >= 0
    source = torch.arange(n, device=neighbors.device)[:, None].expand(n, width)[valid]
    target, by_target = torch.sort(neighbors[valid], stable=True)
    degree = torch.bincount(target, minlength=n)
    out = torch.full((n, max(1, int(degree.max()))), -1, dtype=torch.int32, device=neighbors.device)
    slot = torch.arange(target.numel(), device=neighbors.device) - (degree.cumsum(0) - degree)[target]
    out[target, slot] = source[by_target].int()
    return out


def _rotate(t, coords):
    """Axial rotation of [B, heads, N, d] at integer coordinates [N, 3]: d / 2
    pairs split over (z, y, x), the remainder first."""
    pairs = t.shape[-1] // 2
    out, start = [], 0
    for axis in range(3):
        count = pairs // 3 + (axis < pairs % 3)
        freq = 10000.0 ** (-torch.arange(count, dtype=torch.float64, device=t.device) / max(count, 1))
        angle = coords[:, axis, None].double() * freq
        even, odd = t[..., start:start + 2 * count:2], t[..., start + 1:start + 2 * count:2]
        c, s = angle.cos(), angle.sin()
        out.append(torch.stack((even * c - odd * s, even * s + odd * c), -1).flatten(-2))
        start += 2 * count
    return torch.cat(out, -1)


def _pool(keys, values, weight, bias, blocks, pool):
    """Slot softmax over each fine block, then the mean over each group of
    `pool` blocks that hold a token."""
    valid = blocks >= 0
    k, v = keys[:, :, blocks.clamp_min(0)], values[:, :, blocks.clamp_min(0)]
    logit = (k @ weight + bias).masked_fill(~valid, -torch.inf)
    a = logit.softmax(-1)[..., None]
    fine_k, fine_v = (a * k).sum(-2), (a * v).sum(-2)
    groups = math.ceil(blocks.shape[0] / pool)
    owner = torch.arange(blocks.shape[0], device=blocks.device) // pool
    count = torch.bincount(owner, minlength=groups).double()[:, None]
    zero = fine_k.new_zeros(*fine_k.shape[:2], groups, fine_k.shape[-1])
    return zero.index_add(2, owner, fine_k) / count, zero.index_add(2, owner, fine_v) / count


def _attend(q, kl, vl, sk, sv, neighbors, gate, sl, sg):
    """One chunk of query rows q [B, H, c, d] with neighbour rows [c, W]."""
    b, h, c, d = q.shape
    g = kl.shape[1]
    valid = neighbors >= 0
    index = neighbors.clamp_min(0).reshape(-1)
    k = kl.index_select(2, index).view(b, g, c, -1, d)
    v = vl.index_select(2, index).view(b, g, c, -1, d)
    qg = q.view(b, g, h // g, c, d) / math.sqrt(d)
    local = torch.einsum("bgrcd,bgcwd->bgrcw", qg, k).masked_fill(~valid, -torch.inf)
    local = torch.where(valid.any(-1, keepdim=True), local, torch.zeros_like(local)).softmax(-1) * valid
    ol = torch.einsum("bgrcw,bgcwd->bgrcd", local, v)
    p = (qg.reshape(b, g, -1, d) @ sk.transpose(-1, -2)).softmax(-1)
    og = (p @ sv).view(b, g, h // g, c, d)
    return (sl * ol + gate.view(b, g, h // g, c, 1) * sg * og).reshape(b, h, c, d)


def _core(q, kl, vl, kg, vg, weight, bias, gate, sl, sg, neighbors, blocks, pool):
    sk, sv = _pool(kg, vg, weight, bias, blocks, pool)
    b, h, n, d = q.shape
    widest = max(neighbors.shape[1] * d, sk.shape[2]) * b * h
    step = max(256, min(n, int(5e8 // widest)))
    parts = [checkpoint(_attend, q[:, :, i:i + step], kl, vl, sk, sv, neighbors[i:i + step], gate[:, :, i:i + step],
                        sl, sg, use_reentrant=False) for i in range(0, n, step)]
    return torch.cat(parts, 2)


def exact(case, seed):
    kind = case["kind"]
    if kind == "layout":
        order, blocks = _grid_order(case)
        order, blocks = order.to(DEVICE), blocks.to(DEVICE)
        neighbors, coords = _stencil(case, order)
        perm = _permutation(case, seed).to(DEVICE)
        inverse = torch.empty_like(perm)
        inverse[perm] = torch.arange(perm.numel(), device=DEVICE)
        moved = torch.where(neighbors >= 0, inverse[neighbors.clamp_min(0)], -1)[perm]
        built = {"neighbors": neighbors.int(), "reverse_neighbors": _reverse(neighbors), "blocks": blocks.int()}
        after = {"neighbors": moved.int(), "reverse_neighbors": _reverse(moved), "blocks": inverse[blocks].int()}
        return {"built": {"order": order, "coords": coords, **built},
                "moved": {"order": order[perm], "coords": coords[perm], **after}, "checked": dict(after)}
    if kind == "graph":
        neighbors, blocks = (t.to(DEVICE) for t in _masked_tables(case))
        inputs, dy = _graph_inputs(case, neighbors.shape[0], seed)
        inputs = [t.double().requires_grad_() for t in inputs]
        y = _core(*inputs, neighbors, blocks, case["pool"])
        return [y.detach(), *torch.autograd.grad(y, inputs, dy.double())]
    train = kind == "train"
    order, blocks = _grid_order(case)
    if case["order"] == "random":
        perm = _permutation(case, seed)
        inverse = torch.empty_like(perm)
        inverse[perm] = torch.arange(perm.numel())
        order, blocks = order[perm], inverse[blocks]
    neighbors, coords = _stencil(case, order.to(DEVICE))
    dt = TYPES[case["dtype"]]
    p = {name: t.to(DEVICE, dt).double().requires_grad_(train) for name, t in _parameters(case, seed).items()}
    x, dy = _activations(case, seed)
    x = x.double().requires_grad_(train)
    b, n, h, g, d = case["batch"], x.shape[1], case["heads"], case["kv_heads"], case["head_dim"]
    with torch.set_grad_enabled(train):
        xn = torch.nn.functional.layer_norm(x, (case["dim"],), p["norm.weight"], p["norm.bias"])
        q = (xn @ p["to_q.weight"].t()).view(b, n, h, d).transpose(1, 2)
        kl, vl, kg, vg = (xn @ p["to_kv.weight"].t()).view(b, n, 4, g, d).permute(2, 0, 3, 1, 4)
        gate = (xn @ p["gate.weight"].t() + p["gate.bias"]).view(b, n, h, 2).softmax(-1)[..., 1].transpose(1, 2)
        q, kl, kg = (_rotate(t, coords) for t in (q, kl, kg))
        o = _core(q, kl, vl, kg, vg, p["pool_weight"], p["slot_bias"], gate, p["local_scale"], p["global_scale"],
                  neighbors, blocks.to(DEVICE), case["pool"])
        y = x + o.transpose(1, 2).reshape(b, n, h * d) @ p["to_out.weight"].t()
        if not train:
            return y
        y.backward(dy.double())
    return {"y": y.detach(), "dx": x.grad, **{name: t.grad for name, t in p.items()}}
