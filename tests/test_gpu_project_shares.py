"""Few row tiles: the output blocks of the projections (and of the output product) and the channels of their
input gradient are shared by several workgroups.  Every output is formed alike, so
the first rows of a call with row tiles for every compute unit equal those of a
small call, bit for bit."""
import pytest
import torch

from pack3d_amd import _lib, linear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,outs", [(64, (64, 256, 8)), (96, (48, 64, 8)), (128, (16, 16, 8)), (192, (192, 768, 8)),
                                      (256, (128, 512, 16)), (384, (96, 384, 24)), (512, (512, 1024, 8))])
@pytest.mark.parametrize("rows", [1, 257, 8192, 16640, 32769])
def test_shared_outputs_equal_whole(gpu, dim, outs, rows):
    print(f"project shares dim{dim} {outs} rows{rows}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(dim + rows)
    dt, many = torch.bfloat16, 66000
    x = torch.randn(many, dim, device=gpu, generator=gen).to(dt)
    ws = [(torch.randn(o, dim, device=gpu, generator=gen) / dim ** 0.5).to(dt) for o in outs]
    bg = torch.randn(outs[2], device=gpu, generator=gen).to(dt)
    dys = [torch.randn(many, o, device=gpu, generator=gen).to(dt) for o in outs]
    whole = (*linear.project_linear(x, ws, bg), linear.input_grad(dys, ws))
    part = (*linear.project_linear(x[:rows], ws, bg), linear.input_grad([dy[:rows] for dy in dys], ws))
    for a, b in zip(whole, part):
        assert torch.equal(a[:rows].view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("k,dim,residual", [(64, 64, torch.bfloat16), (96, 96, torch.float32), (192, 192, torch.bfloat16),
                                            (512, 512, torch.float32), (256, 32, torch.bfloat16)])
@pytest.mark.parametrize("rows", [1, 257, 8192, 16640])
def test_shared_output_product_equals_whole(gpu, k, dim, residual, rows):
    print(f"output product shares k{k} dim{dim} {residual} rows{rows}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(k + rows)
    dt, many = torch.bfloat16, 66000
    y = torch.randn(many, k, device=gpu, generator=gen).to(dt)
    wo = (torch.randn(dim, k, device=gpu, generator=gen) / k ** 0.5).to(dt)
    x = torch.randn(many, dim, device=gpu, generator=gen).to(residual)

    def product(n):
        out = torch.full((n, dim), float("nan"), device=gpu, dtype=residual)
        _lib.call("p3d_out_residual", y.data_ptr(), wo.data_ptr(), x.data_ptr(), out.data_ptr(), n, k, dim,
                  _lib.DTYPES[dt], _lib.DTYPES[residual], _lib.stream_of(gpu))
        return out

    whole, part = product(many), product(rows)
    assert torch.isfinite(whole).all() and torch.equal(whole[:rows], part)
