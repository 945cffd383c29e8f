"""One-plane grids of 670 to 1,200 bricks, on either side of the line where the
brick kernels take them in strips of 8 rows (test_gpu_strips_large.py is well past
it).  Forward and every gradient against the oracle, with the rotation fused
(axial and by packed row), on ragged rows and columns, every head_dim and type,
and both plane widths of head_dim 64."""
import math

import pytest
import torch

import oracle.pack3d_oracle as ref
import pack3d_amd as p3d
from pack3d_amd.rope import axial_rope as hip_axial
from tests._cases import random_core_inputs, rel_l2

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 3e-5, torch.float16: 5e-3, torch.bfloat16: 3.5e-2}
NAMES = ["y", "q", "kl", "vl", "kg", "vg", "pool_weight", "slot_bias", "gate", "local_scale", "global_scale"]


@pytest.mark.parametrize("shape,block,radius,kind,b,heads,kv_heads,d,dtype", [
    ((1, 44, 52), (1, 4, 4), (0, 1, 1), "raster_block", 2, 8, 4, 64, torch.bfloat16),
    ((1, 44, 52), (1, 4, 4), (0, 2, 2), "native_block_morton", 2, 8, 4, 64, torch.float16),
    ((1, 36, 60), (1, 6, 6), (0, 2, 1), "raster_block", 2, 8, 8, 48, torch.bfloat16),
    ((1, 132, 18), (1, 6, 6), (0, 1, 2), "native_block_morton", 3, 4, 4, 32, torch.float16),
    ((1, 18, 132), (1, 6, 6), (0, 1, 1), "raster_block", 3, 4, 4, 16, torch.bfloat16),
    ((1, 40, 56), (1, 8, 8), (1, 1, 1), "raster_block", 2, 8, 4, 128, torch.bfloat16),
    ((1, 44, 52), (1, 4, 4), (0, 2, 2), "native_block_morton", 2, 8, 4, 48, torch.float32),
])
def test_strips_match_oracle(gpu, shape, block, radius, kind, b, heads, kv_heads, d, dtype):
    print(f"strips {shape} {radius} {kind} b{b} h{heads} g{kv_heads} d{d} {dtype}", flush=True)
    bricks = -(-shape[1] // 8) * -(-shape[2] // 8) * b
    assert bricks * heads > 512 and bricks * kv_heads > 256
    kw = dict(radius=radius, pool_size=2, layout=kind)
    lay_h, lay_r = p3d.build_layout(shape, block, **kw), ref.build_layout(shape, block, **kw)
    inputs = random_core_inputs(b, heads, kv_heads, math.prod(shape), d, math.prod(block), dtype, seed=d)
    xs = [t.to(gpu).requires_grad_() for t in inputs]
    rs = [t.clone().requires_grad_() for t in inputs]
    y = p3d.pack3d_hip_rope(*xs, lay_h.geometry, hip_axial(d, shape, lay_h.coords))
    q, kl, vl, kg, vg = rs[:5]
    q, kl, kg = (ref.axial_rope(t, lay_r.coords) for t in (q, kl, kg))
    e = ref.pack3d_reference(q, kl, vl, kg, vg, *rs[5:], lay_r.geometry)
    up = torch.randn(e.shape, generator=torch.Generator().manual_seed(3)).to(dtype)
    got = [y, *torch.autograd.grad(y, xs, up.to(gpu))]
    exp = [e, *torch.autograd.grad(e, rs, up)]
    for name, a, x in zip(NAMES, got, exp):
        err = rel_l2(a.float(), x.float())
        print(f"  {name}: rel_l2={err:.3g}", flush=True)
        assert torch.isfinite(a).all() and err < TOL[dtype], (name, err)


def test_strips_packed_rotation(gpu):
    """The rotation by packed row (the layer's "packed" positions) in strips."""
    print("strips packed rotation", flush=True)
    torch.manual_seed(0)
    shape, b = (1, 44, 52), 2
    oracle = ref.PACK3DAttention(64, heads=8, kv_heads=4, head_dim=16, block_volume=16, position_encoding="packed")
    layer = p3d.PACK3DAttention(64, heads=8, kv_heads=4, head_dim=16, block_volume=16, position_encoding="packed")
    layer.load_state_dict(oracle.state_dict())
    layer = layer.to(gpu)
    kw = dict(radius=(0, 1, 1), pool_size=1, layout="native_block_morton")
    x = torch.randn(b, math.prod(shape), 64)
    with torch.no_grad():
        got = layer(x.to(gpu), p3d.build_layout(shape, (1, 4, 4), **kw)).cpu()
        exp = oracle(x, ref.build_layout(shape, (1, 4, 4), **kw))
    assert float((got - exp).abs().max()) < 2e-5
