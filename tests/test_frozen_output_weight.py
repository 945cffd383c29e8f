"""The output product with a frozen weight or an input without gradient: no pass
is made for what nothing asks for, and the other gradients are those of the
whole backward."""
import pytest
import torch

from pack3d_amd import _lib, linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", ["narrow", "wide"])
@pytest.mark.parametrize("mask", [(True, False), (False, True), (False, False)])
def test_output_product_frozen(gpu, monkeypatch, which, mask):
    print(f"frozen output {which} {mask}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(0)
    wide, dt = which == "wide", torch.bfloat16
    fn = linear.OutputResidualWide if wide else linear.OutputResidual
    x, y, wo = (torch.randn(*s, device=gpu, generator=gen).to(t)
                for s, t in (((100, 64), torch.float32 if wide else dt), ((100, 64), dt), ((64, 64), torch.float32)))
    up = torch.randn_like(x)
    calls, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])

    def grads(need):
        leaves = [t.clone().requires_grad_(n) for t, n in zip((x, y, wo), (True, *need))]
        calls.clear()
        out = fn.apply(*leaves, dt)
        out.backward(up)
        return [t.grad for t in leaves], [n for n in calls if n == "p3d_weight_grad"]

    every, used = grads((True, True))
    assert used
    got, used = grads(mask)
    assert bool(used) == mask[1]
    for a, e, need in zip(got, every, (True, *mask)):
        assert torch.equal(a, e) if need else a is None
