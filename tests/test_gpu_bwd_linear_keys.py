"""Backward launches that form the linear branch's dk, dv, too (up to 2048 key blocks), and the first ones that do not: a whole
backward equals the attention's gradients with the linear branch's added, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,D,BLKQ,dtype,fmap", [
    (3, 63, 128, 64, torch.bfloat16, "softmax"),           # one ragged block per head
    (2, 65, 64, 64, torch.float16, "softmax"),             # one row in the second block
    (5, 801, 128, 128, torch.float16, "softmax"),          # 128-row query blocks, the last without a second half
    (7, 831, 64, 64, torch.bfloat16, "relu"),
    (16, 4096, 128, 64, torch.bfloat16, "relu"),           # 1024 key blocks
    (16, 4097, 128, 64, torch.bfloat16, "elu"),            # 1040: two rounds of workgroups and a little more
    (32, 4090, 64, 128, torch.float16, "softmax"),         # 2048
    (33, 3970, 64, 64, torch.bfloat16, "elu"),             # 2079
    (32, 4090, 128, 128, torch.float16, "softmax"),        # 2048
    (33, 3970, 128, 128, torch.bfloat16, "relu"),          # 2079
    (1, 6400, 64, 64, torch.bfloat16, "softmax"),          # one list in segments
])
def test_one_launch_equals_two(H, L, D, BLKQ, dtype, fmap):
    from sla_amd.inputs import make_proj
    from sla_amd.linear import linear_bwd
    from sla_amd.module import module_bwd
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    dev = torch.device("cuda:0")
    M, N = -(-L // BLKQ), -(-L // 64)
    T = min(2, N)
    g = torch.Generator(device=dev).manual_seed(L + D)
    q, k, v, do = (torch.randn(1, H, L, D, device=dev, generator=g).to(dtype) for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    # every row selects key block 0 and one more; some key blocks are selected by nobody
    lut = torch.stack([torch.zeros(M, dtype=torch.long), 1 + torch.arange(M) % max(N // 2, 1)][:T], 1).to(dev)
    lut = lut.expand(1, H, M, T).contiguous()
    smap = torch.zeros(1, H, M, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    lut = lut.int()
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, T, BLKQ, 64, scale)
    grads = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, T, BLKQ, 64, scale)
    ref = linear_bwd(q, k, v, w, b, do, fmap, accumulate_into=grads)
    got = module_bwd(q, k, v, o, do, lse, smap, lut, T, BLKQ, 64, scale, w, b, fmap)
    for name, a, r in zip(("dq", "dk", "dv", "dw", "db"), got, ref):
        assert torch.equal(a, r), name
