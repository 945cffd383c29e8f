"""Weight gradients stage by stage, and fp32 training's linear maps: p3d_weight_grad / p3d_weight_grad3 on fp32
operands against the product in 64 bits, and InputProjections / OutputResidual
in fp32 against torch's linear maps, through the layer and differentiated twice.

The kernel's sum of r products is a chain of roundings of its partial sums;
random roundings leave a relative error near sqrt(r) units of 2^-24 at most."""
import math

import pytest
import torch
import torch.nn.functional as F

import pack3d_amd as p3d
from pack3d_amd import _lib, linear
from tests._cases import rel_l2

pytestmark = pytest.mark.gpu


def _bound(rows):
    return 2.0 ** -24 * math.sqrt(rows)


@pytest.mark.parametrize("rows,out_f,in_f", [(1, 8, 32), (31, 8, 64), (33, 264, 96), (64, 256, 128), (1000, 40, 160),
                                             (4099, 136, 192), (5003, 328, 224), (3001, 264, 256), (2049, 24, 512),
                                             (18711, 768, 192)])
def test_weight_grad_fp32(gpu, rows, out_f, in_f):
    """Every tile width; row counts around a stage of 32 tokens; output counts
    around a block of 256; column ranges of wider tensors."""
    print(f"weight grad fp32 {rows}x{out_f}x{in_f}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(rows + out_f)
    dy = torch.randn(rows, out_f + 16, device=gpu, generator=gen)[:, 8:8 + out_f]
    x = torch.randn(rows, in_f + 8, device=gpu, generator=gen)[:, :in_f]
    dw = linear.weight_grad(dy, x)
    err = rel_l2(dw.double(), torch.mm(dy.double().t(), x.double()))
    print(f"  rel_l2={err:.3g}", flush=True)
    assert err <= _bound(rows)


@pytest.mark.parametrize("rows,in_f,outs", [(37, 192, (192, 768, 8)), (4099, 96, (96, 384, 16)), (3000, 512, (64, 128, 8))])
def test_weight_grads3_fp32(gpu, rows, in_f, outs):
    print(f"weight grads3 fp32 {rows}x{in_f} {outs}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(rows + in_f)
    dys = [torch.randn(rows, o, device=gpu, generator=gen) for o in outs]
    x = torch.randn(rows, in_f, device=gpu, generator=gen)
    got = linear.weight_grads3(dys, x)
    assert got is not None
    for dy, dw in zip(dys, got):
        assert rel_l2(dw.double(), torch.mm(dy.double().t(), x.double())) <= _bound(rows)


def test_fp32_layer_matches_torch_linear(gpu, monkeypatch):
    """Output and every gradient against the same layer with a forward hook on
    to_q, which keeps the torch modules."""
    print("fp32 layer linear maps", flush=True)
    torch.manual_seed(0)
    shape = (4, 12, 20)
    layer = p3d.PACK3DAttention(96, heads=4, kv_heads=2, head_dim=32, block_volume=64).to(gpu)
    lay = p3d.build_layout(shape, (4, 4, 4), radius=1, pool_size=1, layout="raster_block", device=gpu)
    x = torch.randn(1, math.prod(shape), 96, device=gpu)
    dy = torch.randn_like(x)
    names, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (names.append(name), call(name, *a))[1])

    def run():
        names.clear()
        xs = x.clone().requires_grad_()
        y = layer(xs, lay)
        grads = torch.autograd.grad(y, [xs, *layer.parameters()], dy)
        return [y.detach(), *grads], [n for n in names if n.startswith("p3d_weight_grad")]

    got, used = run()
    assert sorted(used) == ["p3d_weight_grad", "p3d_weight_grad3"], used
    seen = []
    layer.to_q.register_forward_hook(lambda m, i, o: seen.append(1))
    exp, used = run()
    assert seen and not used, used
    for a, b in zip(got, exp):
        assert rel_l2(a, b) < 2e-6


def test_fp32_maps_differentiated_twice(gpu):
    """create_graph: the gradients are differentiable and equal torch's."""
    print("fp32 maps twice", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(1)

    def normal(*shape):
        return torch.randn(*shape, device=gpu, generator=gen).requires_grad_()

    x, wq, wkv, wg, bg, wo = normal(2, 50, 32), normal(32, 32), normal(64, 32), normal(8, 32), normal(8), normal(32, 32)

    def second(maps):
        q, kv, gl, out = maps
        first = torch.autograd.grad((q * kv[..., :32]).sum() + gl.square().sum() + out.square().sum(),
                                    [x, wq, wkv, wg, bg, wo], create_graph=True)
        return torch.autograd.grad(sum(g.square().sum() for g in first), [x, wq, wkv, wg, bg, wo])

    q, kv, gl = linear.InputProjections.apply(x, wq, wkv, wg, bg, torch.float32)
    out = linear.OutputResidual.apply(x.reshape(-1, 32), q.reshape(-1, 32), wo, torch.float32)
    q2, kv2, gl2 = F.linear(x, wq), F.linear(x, wkv), F.linear(x, wg, bg)
    out2 = x.reshape(-1, 32) + F.linear(q2.reshape(-1, 32), wo)
    for a, b in zip(second((q, kv, gl, out)), second((q2, kv2, gl2, out2))):
        assert rel_l2(a, b) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,out_f,in_f,splits", [(1, 8, 32, 1), (31, 40, 128, 1), (32, 264, 160, 1), (33, 8, 256, 1),
                                                    (95, 520, 96, 2), (96, 256, 512, 2), (97, 24, 192, 2),
                                                    (641, 300 * 8, 64, 9), (1100, 520, 256, 17)])
def test_weight_grad_stages(gpu, dtype, rows, out_f, in_f, splits):
    """Ranges of less than a stage, of one, two and three, their partial last
    stages beside rows of NaN, and several tiles to a range below, at and above
    eight ranges.  16-bit products are exact in fp32."""
    print(f"weight grad stages {rows}x{out_f}x{in_f} s{splits} {dtype}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(rows + out_f)
    dy, x = (torch.full((rows + 64, c), float("nan"), device=gpu, dtype=dtype) for c in (out_f, in_f))
    dy[:rows] = torch.randn(rows, out_f, device=gpu, generator=gen).to(dtype)
    x[:rows] = torch.randn(rows, in_f, device=gpu, generator=gen).to(dtype)
    dw, work = torch.empty(out_f, in_f, device=gpu), torch.empty(splits, out_f, in_f, device=gpu)
    _lib.call("p3d_weight_grad", dy.data_ptr(), out_f, x.data_ptr(), in_f, dw.data_ptr(), work.data_ptr(), rows, out_f,
              in_f, splits, _lib.DTYPES[dtype], _lib.stream_of(gpu))
    exp = torch.mm(dy[:rows].double().t(), x[:rows].double())
    assert rel_l2(dw.double(), exp) <= _bound(rows)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_frozen_weights(gpu, dtype):
    """Only what requires a gradient gets one, with the value it has when all do."""
    gen = torch.Generator(device=gpu).manual_seed(2)

    def normal(*shape):
        return torch.randn(*shape, device=gpu, generator=gen).to(dtype)

    args = [normal(100, 64), normal(64, 64), normal(128, 64), normal(8, 64), normal(8)]

    def grads(mask):
        leaves = [t.clone().requires_grad_(m) for t, m in zip(args, mask)]
        q, kv, gl = linear.InputProjections.apply(*leaves, dtype)
        (q.square().sum() + kv.square().sum() + gl.square().sum()).backward()
        return [t.grad for t in leaves]

    every = grads([True] * 5)
    for mask in ([False, True, False, False, False], [True, False, True, False, True], [False, False, False, True, False]):
        for got, exp, m in zip(grads(mask), every, mask):
            assert (got is None) != m
            # one rounding to the type: the sums may take another order
            assert not m or rel_l2(got.float(), exp.float()) < (1e-5 if dtype == torch.float32 else 2.0 ** -7)
