"""Upstream gradients as reductions of the output leave them: rows that all lie
at one address (y.sum(1), y.sum((0, 1)): a row stride of 0), a single row of any
stride, overlapping rows.  What the weight and input gradients hand to their
kernels covers its rows, and the layer's gradients are those of a dense one."""
import math

import pytest
import torch

import pack3d_amd as p3d
from pack3d_amd import _lib, linear
from tests._cases import rel_l2


def _operands(rows, cols, dtype):
    base = torch.arange(rows * (cols + 8) + 8, dtype=torch.float32).to(dtype)
    return {"dense": base[:rows * cols].view(rows, cols), "columns": base[:rows * (cols + 8)].view(rows, cols + 8)[:, 8:],
            "one row": base[:cols].expand(rows, cols), "one value": base[0].expand(rows, cols),
            "overlapping": base.as_strided((rows, cols), (8, 1)), "transposed": base[:rows * cols].view(cols, rows).t(),
            "misaligned": base[1:1 + rows * cols].view(rows, cols)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 5])
def test_weight_grad_operands_cover_their_rows(monkeypatch, rows, dtype):
    """Every form of either operand reaches the kernel as 16-byte aligned rows
    at a stride of at least their length, with its values."""
    seen = []

    def call(name, dy, ldy, x, ldx, *rest):
        seen.append((name, dy % 16, ldy, x % 16, ldx))

    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)
    out_f, in_f = 24, 32
    for dy in _operands(rows, out_f, dtype).values():
        for x in _operands(rows, in_f, dtype).values():
            linear.weight_grad(dy, x)
            name, dy_off, ldy, x_off, ldx = seen.pop()
            assert name == "p3d_weight_grad" and dy_off == 0 and x_off == 0
            assert ldy >= out_f and ldy % 8 == 0 and ldx >= in_f and ldx % 8 == 0


@pytest.mark.parametrize("rows", [1, 5])
def test_shared_passes_take_dense_rows_only(monkeypatch, rows):
    """weight_grads3 and input_grad run their kernels on rows that the strides
    cover, and leave the others to the caller's separate products."""
    seen = []
    monkeypatch.setattr(_lib, "call", lambda name, *args: seen.append((name, args)))
    monkeypatch.setattr(_lib, "stream_of", lambda device: 0)
    forms = _operands(rows, 64, torch.bfloat16)
    dense, w = forms["dense"], torch.zeros(64, 64, dtype=torch.bfloat16)
    for name, dy in forms.items():
        for made in (linear.weight_grads3([dense, dy, dense], dense), linear.weight_grads3([dense] * 3, dy),
                     linear.input_grad([dense, dy, dense], [w] * 3)):
            if rows > 1:
                assert (made is None) == (name not in ("dense", "columns")), name
    assert seen
    for name, args in seen:
        # (address, row stride, columns) of each gradient, then x's address and stride
        operands = {"p3d_weight_grad3": [args[0:2], args[3:5], args[6:8], args[9:11]],
                    "p3d_input_grad": [args[0:2], args[3:5], args[6:8]]}.get(name, [])
        assert all(at % 16 == 0 and ld >= 64 and ld % 8 == 0 for at, ld in operands), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,dims", [(1, (1,)), (2, (0, 1)), (2, (1,)), (1, (0, 1, 2))])
def test_layer_backward_of_reduced_output(gpu, dtype, b, dims):
    """The gradients of a reduced output are those of the same dense gradient, bit
    for bit: the kernels see the same values."""
    print(f"reduced output b{b} {dims} {dtype}", flush=True)
    torch.manual_seed(0)
    layer = p3d.PACK3DAttention(64, heads=4, kv_heads=2, head_dim=16, block_volume=64).to(gpu, dtype)
    lay = p3d.build_layout((4, 8, 8), (4, 4, 4), radius=1, pool_size=1, layout="raster_block", device=gpu)
    x = torch.randn(b, 256, 64, device=gpu).to(dtype).requires_grad_()
    params = [x, *layer.parameters()]
    y = layer(x, lay)
    up = torch.randn(y.sum(dims).shape, device=gpu).to(dtype)
    got = torch.autograd.grad(y.sum(dims), params, up)
    for d in sorted(dims):
        up = up.unsqueeze(d)
    exp = torch.autograd.grad(layer(x, lay), params, up.expand(y.shape).contiguous())
    for a, e in zip(got, exp):
        assert torch.equal(a, e)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_maps_backward_of_expanded_gradients(gpu, dtype):
    """InputProjections and OutputResidual on gradients of row stride 0, against
    the sums in 64 bits."""
    print(f"expanded gradients {dtype}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(3)

    def normal(*shape):
        return torch.randn(*shape, device=gpu, generator=gen).to(dtype)

    rows = 300
    leaves = [t.requires_grad_() for t in (normal(rows, 64), normal(64, 64), normal(128, 64), normal(8, 64), normal(8))]
    made = linear.InputProjections.apply(*leaves, dtype)
    ups = [normal(t.shape[1]).expand(t.shape) for t in made]
    got = torch.autograd.grad(made, leaves, ups)
    x, *ws, _ = (t.detach().double() for t in leaves)
    ups = [u.double() for u in ups]
    exp = [sum(u @ w for u, w in zip(ups, ws)), *(u.t() @ x for u in ups), ups[2].sum(0)]
    wo, y = normal(64, 64).requires_grad_(), normal(rows, 64).requires_grad_()
    up = normal(64).expand(rows, 64)
    got += torch.autograd.grad(linear.OutputResidual.apply(leaves[0], y, wo, dtype), (y, wo), up)
    exp += [up.double() @ wo.detach().double(), up.double().t() @ y.detach().double()]
    # Sums of at most 300 products in fp32 (2^-24 sqrt(300)); in bf16 the input
    # gradient may be rounded three times on its way (three products in one buffer).
    tol = 2.0 ** -24 * math.sqrt(rows) if dtype == torch.float32 else 3 * 2.0 ** -8
    for a, e in zip(got, exp):
        assert rel_l2(a.double(), e) < tol
