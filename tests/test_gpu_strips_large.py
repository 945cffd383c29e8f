"""One-plane grids that the brick kernels take in strips of 8 rows by their rule
(csrc/strips.hpp): the rule at measured sizes and at those of the GPU test, and
the forward and every gradient there against the oracle, with four strips to a
workgroup and a last one with three."""
import math

import pytest
import torch

import oracle.pack3d_oracle as ref
import pack3d_amd as p3d
from pack3d_amd.rope import axial_rope as hip_axial
from tests._cases import random_core_inputs, rel_l2
from tests._host_cpp import run_host_cpp

TOL = {torch.float32: 3e-5, torch.float16: 5e-3, torch.bfloat16: 3.5e-2}
NAMES = ["y", "q", "kl", "vl", "kg", "vg", "pool_weight", "slot_bias", "gate", "local_scale", "global_scale"]

CASES = [
    ((1, 116, 60), (1, 4, 4), (0, 1, 1), "raster_block", 2, 8, 4, 64, torch.bfloat16),
    ((1, 124, 60), (1, 4, 4), (0, 2, 2), "native_block_morton", 2, 8, 4, 64, torch.float16),
    ((1, 114, 60), (1, 6, 6), (0, 2, 1), "raster_block", 2, 8, 8, 48, torch.bfloat16),
    ((1, 126, 60), (1, 6, 6), (0, 1, 2), "native_block_morton", 4, 4, 4, 32, torch.float16),
    ((1, 120, 64), (1, 8, 8), (0, 1, 1), "raster_block", 4, 4, 4, 16, torch.bfloat16),
    ((1, 120, 64), (1, 8, 8), (1, 1, 1), "raster_block", 2, 8, 4, 128, torch.bfloat16),
    ((1, 124, 60), (1, 4, 4), (0, 1, 1), "native_block_morton", 2, 8, 4, 48, torch.float32),
]


def _bricks(shape):
    return -(-shape[1] // 8), -(-shape[2] // 8)


def test_rule(tmp_path):
    """(forward, backward, head_dim, 16-bit kind or fp32, bricks in y and x, query
    head planes, kv head planes): sizes where one tiling measured at least a tenth
    faster, and every case of the GPU test."""
    points = [
        (True, True, 64, "bf16", 16, 16, 16, 4), (True, True, 128, "fp16", 16, 16, 16, 4), (True, True, 48, "fp32", 16, 16, 16, 4),
        (False, False, 64, "bf16", 8, 8, 16, 8), (True, False, 32, "bf16", 8, 8, 16, 8), (True, True, 128, "bf16", 8, 8, 16, 8),
        (False, True, 16, "bf16", 6, 7, 16, 16), (True, True, 32, "fp16", 6, 7, 16, 16), (False, True, 64, "bf16", 6, 7, 16, 16),
        (False, False, 16, "fp32", 9, 11, 8, 4), (False, False, 48, "bf16", 9, 11, 16, 10), (False, True, 64, "bf16", 9, 11, 16, 16),
        (False, False, 64, "bf16", 1, 4, 1, 1),
    ]
    kinds = {torch.float32: "fp32", torch.float16: "fp16", torch.bfloat16: "bf16"}
    points += [(True, True, 16, "fp32", 15, 8, 16, 8)]  # the packed rotation's layer
    points += [(True, True, d, kinds[t], *_bricks(shape), b * h, b * g) for shape, _, _, _, b, h, g, d, t in CASES]
    body = "".join(
        f'printf("%d %d\\n", p3d::strips_forward({d}, {int(kind == "bf16")}, {by}, {bx}, {h}), '
        f'p3d::strips_backward({d}, {int(kind == "fp32")}, {by}, {bx}, {g}));\n' for _, _, d, kind, by, bx, h, g in points)
    for point, line in zip(points, run_host_cpp(tmp_path, ["strips.hpp"], body)):
        assert line == f"{int(point[0])} {int(point[1])}", point


@pytest.mark.gpu
@pytest.mark.parametrize("shape,block,radius,kind,b,heads,kv_heads,d,dtype", CASES)
def test_strips_match_oracle(gpu, shape, block, radius, kind, b, heads, kv_heads, d, dtype):
    print(f"strips {shape} {radius} {kind} b{b} h{heads} g{kv_heads} d{d} {dtype}", flush=True)
    kw = dict(radius=radius, pool_size=16, layout=kind)
    lay_h, lay_r = p3d.build_layout(shape, block, **kw), ref.build_layout(shape, block, **kw)
    inputs = random_core_inputs(b, heads, kv_heads, math.prod(shape), d, math.prod(block), dtype, seed=d)
    xs = [t.to(gpu).requires_grad_() for t in inputs]
    rs = [t.clone().requires_grad_() for t in inputs]
    y = p3d.pack3d_hip_rope(*xs, lay_h.geometry, hip_axial(d, shape, lay_h.coords))
    up = torch.randn(y.shape, generator=torch.Generator().manual_seed(3)).to(dtype)
    got = [y, *torch.autograd.grad(y, xs, up.to(gpu))]
    q, kl, vl, kg, vg = rs[:5]
    q, kl, kg = (ref.axial_rope(t, lay_r.coords) for t in (q, kl, kg))
    e = ref.pack3d_reference(q, kl, vl, kg, vg, *rs[5:], lay_r.geometry)
    print("  oracle forward", flush=True)
    exp = [e, *torch.autograd.grad(e, rs, up)]
    for name, a, x in zip(NAMES, got, exp):
        err = rel_l2(a.float(), x.float())
        print(f"  {name}: rel_l2={err:.3g}", flush=True)
        assert torch.isfinite(a).all() and err < TOL[dtype], (name, err)


@pytest.mark.gpu
def test_strips_packed_rotation_layer(gpu):
    """The rotation by packed row (the layer's "packed" positions) in strips, with
    every gradient of the layer."""
    print("strips packed rotation layer", flush=True)
    torch.manual_seed(0)
    shape, b = (1, 120, 64), 2
    kw = dict(heads=8, kv_heads=4, head_dim=16, block_volume=64, position_encoding="packed")
    oracle, layer = ref.PACK3DAttention(64, **kw), p3d.PACK3DAttention(64, **kw)
    layer.load_state_dict(oracle.state_dict())
    layer = layer.to(gpu)
    kw = dict(radius=(0, 1, 1), pool_size=4, layout="native_block_morton")
    x, dy = torch.randn(2, b, math.prod(shape), 64)
    out = []
    for m, lay, dev in ((layer, p3d.build_layout(shape, (1, 8, 8), **kw), gpu), (oracle, ref.build_layout(shape, (1, 8, 8), **kw), "cpu")):
        xs = x.to(dev).requires_grad_()
        y = m(xs, lay)
        out.append([y, *torch.autograd.grad(y, [xs, *m.parameters()], dy.to(dev))])
    for a, e in zip(*out):
        assert rel_l2(a, e) < TOL[torch.float32]
