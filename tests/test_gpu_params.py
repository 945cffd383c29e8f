"""The small passes of the 16-bit training step (csrc/params.hip) against fp64:
sums of partial gradients, column sums, the gate's pair softmax in both
directions, casts, and the transposed concatenation of weights."""
import pytest
import torch

from pack3d_amd import _lib, linear

pytestmark = pytest.mark.gpu

EPS = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 7, 512, 513, 2048, 2049])
def test_sum_rows(gpu, rows, dtype):
    """Every job shape (1 to 129 columns, strided rows) on both sides of the
    column split; an fp32 sum of r terms is within r ulps of the sum of
    magnitudes, and the result is rounded once."""
    print(f"sum_rows {rows} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(rows)
    jobs = []
    for cols, extra in ((1, 0), (5, 3), (64, 0), (129, 7)):
        src = torch.randn(rows, cols + extra, generator=gen).to(gpu)
        jobs.append((src[:, :cols], torch.full((cols,), float("nan"), dtype=dtype, device=gpu)))
    _lib.sum_rows(jobs, gpu)
    for src, out in jobs:
        exact = src.double().sum(0)
        bound = rows * EPS[torch.float32] * src.double().abs().sum(0) + EPS[dtype] * (exact.abs() + 1e-6)
        assert bool(((out.double() - exact).abs() <= bound).all()), (src.shape, dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(1, 8), (127, 8), (128, 16), (1000, 24), (4097, 256)])
def test_column_sums(gpu, rows, cols, dtype):
    print(f"column_sums {rows}x{cols} {dtype}", flush=True)
    x = torch.randn(rows, cols + 8, generator=torch.Generator().manual_seed(cols)).to(gpu, dtype)[:, :cols]
    got = linear.column_sums(x, torch.float32)
    exact = x.double().sum(0)
    assert bool(((got.double() - exact).abs() <= rows * EPS[torch.float32] * x.double().abs().sum(0)).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,n,h", [(1, 1, 1), (2, 255, 4), (3, 257, 8)])
@pytest.mark.parametrize("wide", [True, False])
def test_gate_probability(gpu, dtype, b, n, h, wide):
    """The gate and its gradient from wide logit gaps (saturated pairs), and a
    gradient with permuted strides, against fp64: four fp32 operations and one
    rounding to the output's type."""
    print(f"gate b{b} n{n} h{h} {dtype} wide={wide}", flush=True)
    gen = torch.Generator().manual_seed(n + h)
    gl = (torch.randn(b, n, 2 * h, generator=gen) * 8).to(gpu, dtype).requires_grad_()
    out_dtype = torch.float32 if wide else dtype
    bias = torch.zeros(2 * h, device=gpu, requires_grad=True)
    gate = linear.GateProbability.apply(gl, bias, h, out_dtype)
    dgate = torch.randn(n, b, h, generator=gen).to(gpu, out_dtype).permute(1, 2, 0)
    exact_gl = gl.detach().double().requires_grad_()
    exact = exact_gl.view(b, n, h, 2).softmax(-1)[..., 1].transpose(1, 2)
    got, dbias = torch.autograd.grad(gate, (gl, bias), dgate)
    (exp,) = torch.autograd.grad(exact, exact_gl, dgate.double())
    # The bias gradient sums the unrounded gradients: fp32 sums of b n terms.
    err = (dbias.double() - exp.sum((0, 1))).abs()
    assert bool((err <= (b * n + 16) * EPS[torch.float32] * exp.abs().sum((0, 1))).all())
    assert gate.dtype == out_dtype and gate.shape == (b, h, n)
    # Half a subnormal step of fp16; else the fp64 reference's own error where it
    # forms y1 - y1 y1 of a saturated pair (2^-53 of |dgate| < 8, with margin).
    tiny = 2.0 ** -24 if dtype == torch.float16 else 2.0 ** -48
    for a, e, t in ((gate, exact, out_dtype), (got, exp, dtype)):
        err = (a.double() - e).abs()
        assert bool((err <= (16 * EPS[torch.float32] + EPS[t]) * e.abs() + tiny).all()), float(err.max())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_cast_all(gpu, dtype):
    print(f"cast_all {dtype}", flush=True)
    gen = torch.Generator().manual_seed(0)
    tensors = [torch.randn(3, 5, generator=gen), torch.randn(2048, generator=gen), torch.randn(129, 33, generator=gen).t(),
               torch.randn(7, generator=gen).to(dtype)]
    tensors = [t.to(gpu) for t in tensors]
    for got, t in zip(linear.cast_all(tensors, dtype), tensors):
        assert got.is_contiguous() and torch.equal(got, t.to(dtype))


@pytest.mark.parametrize("outs,dim,k_pad", [((8, 8, 8), 64, 64), ((192, 768, 8), 192, 1024), ((33, 65, 31), 96, 192)])
def test_concat_transpose(gpu, outs, dim, k_pad):
    print(f"concat_transpose {outs} {dim}", flush=True)
    gen = torch.Generator().manual_seed(dim)
    ws = [torch.randn(o, dim, generator=gen).to(gpu, torch.bfloat16) for o in outs]
    wt = torch.full((dim, k_pad), float("nan"), dtype=torch.bfloat16, device=gpu)
    args = [v for w, o in zip(ws, outs) for v in (w.data_ptr(), o)]
    _lib.call("p3d_concat_transpose", *args, dim, wt.data_ptr(), k_pad, _lib.stream_of(gpu))
    exp = torch.zeros_like(wt)
    exp[:, :sum(outs)] = torch.cat(ws, 0).t()
    assert torch.equal(wt, exp)
