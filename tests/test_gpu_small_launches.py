"""Launches around the sizes at which the attention kernels change: 144 pairs of 64-row query blocks in the forward (either
head dim), 320 query blocks in dQ (head dim 128)."""
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


@pytest.mark.parametrize("H,L,T,BLKQ,dtype", [(9, 1985, 3, 64, torch.bfloat16),      # 144 pairs, one row in the last block
                                               (29, 650, 4, 64, torch.float16),       # no partner for a head's last block
                                               (20, 1000, 1, 64, torch.bfloat16),     # one step
                                               (20, 1024, 16, 64, torch.bfloat16),    # every key block
                                               (19, 1000, 5, 128, torch.float16),     # 128-row blocks, ragged second half
                                               (23, 832, 4, 128, torch.bfloat16)])    # last 128-row block without a second half
@pytest.mark.parametrize("lut_dtype", [torch.int32, torch.int64])
def test_head_dim_64_pairs(dev, H, L, T, BLKQ, dtype, lut_dtype):
    """Head dim 64 through the kernel that walks two query blocks: rows with shared and with own key blocks, in any order."""
    from sla_amd.sparse_attn import sparse_attn_fwd
    g = torch.Generator().manual_seed(L + T)
    q, k, v = (torch.randn(1, H, L, 64, generator=g).to(dtype) for _ in range(3))
    M, N = -(-L // BLKQ), -(-L // 64)
    lut = torch.stack([torch.randperm(N, generator=g)[:T] for _ in range(H * M)]).view(1, H, M, T)
    o_ref, lse_ref = O.sparse_attn_fwd_gather(q, k, v, lut, BLKQ, 64)
    o, lse = sparse_attn_fwd(*(t.to(dev) for t in (q, k, v)), lut.to(lut_dtype).to(dev), T, BLKQ, 64, 64 ** -0.5)
    assert max_abs(o.cpu(), o_ref) <= TOL_ABS and cos_sim(o.cpu(), o_ref) >= TOL_COS
    assert max_abs(lse.cpu(), lse_ref) <= 2e-3          # fp32 sums of 16-bit products, base-2 units


def test_head_dim_64_growing_scores_and_repeated_entries(dev):
    """The reference maximum of the online softmax has to move (later key blocks score far higher), and a table row that
    names a key block twice is walked as given."""
    from sla_amd.sparse_attn import sparse_attn_fwd
    H, L, T = 20, 1024, 8
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, H, L, 64, generator=g).to(torch.bfloat16) for _ in range(3))
    k = (k.float() * (1 + 6 * torch.arange(L).view(1, 1, L, 1) / L)).to(torch.bfloat16)
    lut = torch.stack([torch.randperm(16, generator=g)[:T].sort().values for _ in range(H * 16)]).view(1, H, 16, T)
    lut[:, :, 3, 1] = lut[:, :, 3, 0]
    o_ref, _ = O.sparse_attn_fwd_gather(q, k, v, lut, 64, 64)
    o, _ = sparse_attn_fwd(*(t.to(dev) for t in (q, k, v)), lut.to(dev), T, 64, 64, 64 ** -0.5)
    assert max_abs(o.cpu(), o_ref) <= TOL_ABS and cos_sim(o.cpu(), o_ref) >= TOL_COS
