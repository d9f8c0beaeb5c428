"""Launches around the sizes at which the attention kernels change at head dim 128: 144 pairs of 64-row query blocks in
the forward, 320 query blocks in dQ."""
import pytest
import torch

from conftest import cos_sim, max_abs
from oracle import sla_oracle as O
from sla_amd import _attention

pytestmark = pytest.mark.gpu

TOL_ABS = 2e-2
TOL_COS = 0.999


@pytest.mark.parametrize("H,L,ratio,dtype", [(9, 1985, 0.1, torch.bfloat16),     # 144 pairs, 288 blocks, one row in the last block
                                              (11, 1600, 0.1, torch.float16),     # 143 pairs
                                              (10, 2048, 0.2, torch.bfloat16),    # 160 pairs, 320 blocks
                                              (29, 650, 0.2, torch.bfloat16)])    # odd block count per head, 319 blocks
def test_lines_between_the_kernels(dev, H, L, ratio, dtype):
    g = torch.Generator().manual_seed(H * L)
    q, k, v, do = (torch.randn(1, H, L, 128, generator=g).to(dtype) for _ in range(4))
    m, lut, T = O.get_block_map(q, k, ratio, 64, 64)
    o_ref, lse_ref = O.sparse_attn_fwd_dense(q, k, v, m, 64, 64)
    refs = O.sparse_attn_bwd_dense(q, k, v, o_ref, do, lse_ref, m, 64, 64)
    qd, kd, vd = (t.to(dev).requires_grad_(True) for t in (q, k, v))
    o = _attention.apply(qd, kd, vd, m.to(dev), lut.to(dev), T, 64, 64)
    o.backward(do.to(dev))
    assert max_abs(o.detach().cpu(), o_ref) <= TOL_ABS and cos_sim(o.detach().cpu(), o_ref) >= TOL_COS
    for name, t, r in zip(("dq", "dk", "dv"), (qd, kd, vd), refs):
        assert max_abs(t.grad.cpu(), r) <= TOL_ABS and cos_sim(t.grad.cpu(), r) >= TOL_COS, name
