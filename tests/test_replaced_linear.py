"""fp32 training with linear modules that are more than nn.Linear's product: a
forward replaced on the object, a module of another class (with no bias
attribute).  The layer calls them, as it does in every other mode."""
import types

import pytest
import torch
import torch.nn.functional as F
from torch import nn

import pack3d_amd as p3d
from pack3d_amd.attention import _plain_linear
from tests._cases import rel_l2


class _Weighted(nn.Module):
    def __init__(self, linear):
        super().__init__()
        self.weight = linear.weight

    def forward(self, x):
        return F.linear(x, self.weight)


def _replace_forward(m, scale):
    m.forward = types.MethodType(lambda self, x: scale * nn.Linear.forward(self, x), m)
    return m


def test_plain_linear():
    assert _plain_linear(nn.Linear(4, 4)) and _plain_linear(nn.Linear(4, 4, bias=False))
    hooked = nn.Linear(4, 4)
    hooked.register_forward_hook(lambda m, i, o: None)
    backward = nn.Linear(4, 4)
    backward.register_full_backward_hook(lambda m, i, o: None)
    weighted = nn.utils.parametrizations.weight_norm(nn.Linear(4, 4))
    for m in (hooked, backward, weighted, _replace_forward(nn.Linear(4, 4), 2), _Weighted(nn.Linear(4, 4)), nn.Identity()):
        assert not _plain_linear(m)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["to_q", "to_kv"])
@pytest.mark.parametrize("how", ["forward", "class"])
def test_fp32_layer_calls_replaced_modules(gpu, name, how):
    """Against a layer of plain modules with the same function."""
    print(f"replaced {name} {how}", flush=True)
    torch.manual_seed(0)
    lay = p3d.build_layout((4, 8, 8), (4, 4, 4), radius=1, pool_size=1, layout="raster_block", device=gpu)
    layers = [p3d.PACK3DAttention(64, heads=4, kv_heads=2, head_dim=16, block_volume=64).to(gpu) for _ in range(2)]
    layers[1].load_state_dict(layers[0].state_dict())
    if how == "forward":
        _replace_forward(getattr(layers[0], name), 2.0)
        with torch.no_grad():
            getattr(layers[1], name).weight.mul_(2.0)
    else:
        setattr(layers[0], name, _Weighted(getattr(layers[0], name)))
    x, dy = torch.randn(2, 1, 256, 64, device=gpu)
    out = []
    for layer in layers:
        xs = x.clone().requires_grad_()
        y = layer(xs, lay)
        y.backward(dy)
        out.append([y, xs.grad, *(p.grad * (2.0 if how == "forward" and layer is layers[1] and n == f"{name}.weight" else 1.0)
                                  for n, p in layer.named_parameters())])
    for a, b in zip(*out):
        assert rel_l2(a, b) < 2e-6  # two orders of the same fp32 sums
