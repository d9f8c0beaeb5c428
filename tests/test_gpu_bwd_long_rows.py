"""Look-up rows of more than 2048 key blocks: dQ by its general kernel (delta and the short jobs in launches of their own), dK/dV by the
stream kernel over numbered work items, every list cut into segments: against dense attention in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,BLKQ", [(64, 64), (64, 128), (128, 64)])
def test_rows_longer_than_the_stream_kernel_keeps(dev, D, BLKQ):
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    N, T = 2050, 2049
    L = 64 * N - 27
    M = -(-L // BLKQ)
    g = torch.Generator(device=dev).manual_seed(D + BLKQ)
    q, k, v, do = (torch.randn(1, 1, L, D, device=dev, generator=g).bfloat16() for _ in range(4))
    # row m selects every key block but 7 m + 5 (mod N)
    left_out = (7 * torch.arange(M, device=dev) + 5) % N
    lut = torch.arange(T, device=dev).expand(M, T)
    lut = (lut + (lut >= left_out[:, None])).int()[None, None].contiguous()
    smap = torch.ones(1, 1, M, N, dtype=torch.int8, device=dev)
    smap[0, 0, torch.arange(M, device=dev), left_out] = 0
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, T, BLKQ, 64, scale)
    got = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, T, BLKQ, 64, scale)
    qf, kf, vf, dof = (t[0, 0].float() for t in (q, k, v, do))
    kt, vt = kf.T.contiguous(), vf.T.contiguous()
    dq, dk, dv = (torch.zeros_like(qf) for _ in range(3))
    for r in range(0, L, 2048):
        rows = slice(r, min(L, r + 2048))
        mask = smap[0, 0, r // BLKQ:-(-rows.stop // BLKQ)].bool().repeat_interleave(BLKQ, 0).repeat_interleave(64, 1)
        s = (qf[rows] @ kt).mul_(scale).masked_fill_(~mask[:rows.stop - r, :L], float("-inf"))
        p = torch.softmax(s, -1)
        del s, mask
        dp = dof[rows] @ vt
        ds = p * (dp - (p * dp).sum(-1, keepdim=True))
        dv += p.T.contiguous() @ dof[rows]
        dq[rows] = ds @ kf * scale
        dk += ds.T.contiguous() @ qf[rows] * scale
        del p, dp, ds
    for name, a, r in zip(("dq", "dk", "dv"), got, (dq, dk, dv)):
        # (probabilities, dS and the result are rounded to bf16, u = 2^-9 each: within 4 u of the 2-norm)
        err = float((a[0, 0].float() - r).norm() / r.norm())
        assert err <= 4 * 2.0 ** -9, (name, err)
