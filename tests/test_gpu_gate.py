"""The gate's backward past the heads of one launch row, and both directions of
the gate on infinite and NaN logits and gradients."""
import math

import pytest
import torch

from pack3d_amd import linear

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,n,h", [(1, 3, 2048), (2, 130, 2049), (1, 257, 4100)])
def test_gate_backward_many_heads(gpu, dtype, b, n, h):
    """Any count of heads, as torch's softmax takes: the logit gradients are one
    rounding and four fp32 operations from those in 64 bits, the bias gradient an
    fp32 sum of b n terms."""
    print(f"gate heads b{b} n{n} h{h} {dtype}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(h)
    gl = torch.randn(b, n, 2 * h, generator=gen, device=gpu).to(dtype).requires_grad_()
    bias = torch.zeros(2 * h, device=gpu, requires_grad=True)
    dgate = torch.randn(b, h, n, generator=gen, device=gpu)
    got, dbias = torch.autograd.grad(linear.GateProbability.apply(gl, bias, h, torch.float32), (gl, bias), dgate)
    exact_gl = gl.detach().double().requires_grad_()
    exact = exact_gl.view(b, n, h, 2).softmax(-1)[..., 1].transpose(1, 2)
    (exp,) = torch.autograd.grad(exact, exact_gl, dgate.double())
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0  # half a subnormal step
    assert bool(((got.double() - exp).abs() <= (16 * EPS[torch.float32] + EPS[dtype]) * exp.abs() + tiny).all())
    bound = (b * n + 16) * EPS[torch.float32] * exp.abs().sum((0, 1))
    assert bool(((dbias.double() - exp.sum((0, 1))).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("upstream", [1.0, -2.0, 0.0, math.inf, -math.inf, math.nan])
def test_gate_of_infinite_and_nan_logits(gpu, dtype, upstream):
    """As an overflowed step leaves them: the gate is NaN where torch's softmax is,
    a logit gradient is finite where torch's is, and the bias gradient of a head
    shows what any of its tokens does not hold finite."""
    print(f"gate specials {dtype} {upstream}", flush=True)
    inf, nan = math.inf, math.nan
    values = [nan, inf, -inf, 0.0, 3.0, -200.0, 200.0]
    pairs = torch.tensor([[a, b] for a in values for b in values])
    gl = pairs.view(1, 1, -1).to(gpu, dtype).requires_grad_()  # one token, one head per pair
    heads = len(pairs)
    bias = torch.zeros(2 * heads, device=gpu, requires_grad=True)
    gate = linear.GateProbability.apply(gl, bias, heads, torch.float32)
    dgate = torch.full_like(gate, upstream)
    got, dbias = torch.autograd.grad(gate, (gl, bias), dgate)
    ref = gl.detach().float().requires_grad_()
    exact = ref.view(1, 1, heads, 2).softmax(-1)[..., 1].transpose(1, 2)
    (exp,) = torch.autograd.grad(exact, ref, dgate)
    assert torch.equal(gate.isnan(), exact.isnan())
    assert torch.equal(gate.nan_to_num(), exact.nan_to_num()) or torch.allclose(gate.nan_to_num(), exact.nan_to_num(), rtol=1e-6, atol=0)
    finite = exp.view(heads, 2).isfinite().all(-1)
    assert torch.equal(got.view(heads, 2).isfinite().all(-1), finite)
    assert torch.equal(dbias.view(heads, 2).isfinite().all(-1), finite)
