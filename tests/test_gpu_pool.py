"""Summaries whose steps are shared by several pooling waves: more steps than
waves, a last summary with fewer steps than waves (the rest of its waves have
none), blocks taken whole and packed, empty slots, and summaries enough for a
wave each.  Forward and every gradient against the oracle."""
import pytest
import torch

import oracle.pack3d_oracle as ref
import pack3d_amd as p3d
from tests._cases import make_case, rel_l2

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 3e-5, torch.float16: 5e-3, torch.bfloat16: 3.5e-2}
NAMES = ["y", "q", "kl", "vl", "kg", "vg", "pool_weight", "slot_bias", "gate", "local_scale", "global_scale"]


@pytest.mark.parametrize("n,d,b,heads,kv_heads,volume,pool,dtype", [
    (2112, 64, 1, 2, 1, 64, 32, torch.bfloat16),    # 32 steps, then 1
    (1900, 48, 2, 2, 2, 64, 12, torch.float16),     # 12 steps, a partial last block
    (1000, 128, 1, 2, 1, 27, 7, torch.bfloat16),    # 7 steps of one 27-slot block
    (1040, 16, 1, 2, 2, 16, 24, torch.float32),     # four blocks a step: 6 steps, then 5
    (1300, 32, 2, 2, 1, 8, 32, torch.float16),      # eight blocks a step: 4 steps, then 1
    (900, 128, 1, 2, 1, 64, 3, torch.float32),      # 3 steps: two waves
    (4200, 16, 4, 4, 4, 16, 8, torch.bfloat16),     # 1,024 summaries with padding, 2 waves each
    (4200, 16, 8, 4, 4, 16, 8, torch.bfloat16),     # 2,048: one wave each
])
def test_shared_summaries_match_oracle(gpu, n, d, b, heads, kv_heads, volume, pool, dtype):
    print(f"shared summaries n{n} d{d} b{b} g{kv_heads} v{volume} pool{pool} {dtype}", flush=True)
    inputs, nb, blocks, pool = make_case(n=n, d=d, b=b, h=heads, g=kv_heads, volume=volume, pool=pool, dtype=dtype,
                                         seed=n)
    hg, og = p3d.prepare_geometry(nb.to(gpu), blocks.to(gpu), pool), ref.prepare_geometry(nb, blocks, pool)
    xs = [t.to(gpu).requires_grad_() for t in inputs]
    rs = [t.detach().clone().requires_grad_() for t in inputs]
    y, e = p3d.pack3d_hip(*xs, hg, temperature=0.8), ref.pack3d_reference(*rs, og, temperature=0.8)
    up = torch.randn(e.shape, generator=torch.Generator().manual_seed(3)).to(dtype)
    got, exp = [y, *torch.autograd.grad(y, xs, up.to(gpu))], [e, *torch.autograd.grad(e, rs, up)]
    for name, a, x in zip(NAMES, got, exp):
        err = rel_l2(a.float().cpu(), x.float())
        print(f"  {name}: rel_l2={err:.3g}", flush=True)
        assert torch.isfinite(a).all() and err < TOL[dtype], (name, err)
