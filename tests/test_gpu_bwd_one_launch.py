"""dQ and dK/dV in one launch, with delta formed beforehand: against dense attention in fp32, lists cut into segments in several
strips of 64 key blocks among them, and bit for bit against the launches of their own that larger calls of head dim 128 take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _case(dev, H, L, D, BLKQ, lut, dtype, seed):
    M, N = -(-L // BLKQ), -(-L // 64)
    g = torch.Generator(device=dev).manual_seed(seed)
    q, k, v, do = (torch.randn(1, H, L, D, device=dev, generator=g).to(dtype) for _ in range(4))
    lut = lut.to(dev).expand(1, H, M, lut.shape[-1]).contiguous()
    smap = torch.zeros(1, H, M, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    return q, k, v, do, lut.int(), smap


@pytest.mark.parametrize("H,L,D,BLKQ,dtype,sinks", [
    (1, 40, 128, 64, torch.bfloat16, ()),                       # one ragged block: an odd number of query blocks, one wave idle
    (3, 65, 128, 64, torch.float16, (0,)),
    (5, 321, 128, 128, torch.bfloat16, (0,)),                   # 128-row blocks, the last without a second half
    (2, 64 * 65 - 3, 128, 64, torch.bfloat16, (0, 63, 64)),     # lists of 65 entries: two segments, on both sides of a strip's edge
    (2, 64 * 131 - 60, 128, 64, torch.float16, (5, 70, 130)),   # 131 entries: three segments, three strips per head
    (2, 128 * 67 + 9, 128, 128, torch.bfloat16, (1, 2, 134)),   # 68 entries of two halves each
    (40, 64 * 66, 128, 64, torch.bfloat16, (0, 65)),            # 80 strips: more than a wave's lanes
    (1, 33, 64, 64, torch.float16, ()),                         # head dim 64: two waves per query block, one row in the second
    (3, 97, 64, 64, torch.bfloat16, (0, 1)),                    # one row in the last 32 keys
    (3, 64 * 7 + 32, 64, 128, torch.float16, (2, 7)),
    (2, 64 * 131 - 60, 64, 64, torch.bfloat16, (5, 70, 130)),
    (40, 64 * 66, 64, 128, torch.bfloat16, (0, 65)),
])
def test_gradients(dev, H, L, D, BLKQ, dtype, sinks):
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    M, N = -(-L // BLKQ), -(-L // 64)
    rows = [sorted(set(sinks) | {(7 * m) % N}) for m in range(M)]
    T = min(len(r) for r in rows)
    if T < max(len(r) for r in rows):                           # (rows whose own block is a sink get another one)
        T += 1
        rows = [r if len(r) == T else sorted(set(r) | {next(x for x in range(N) if x not in r)}) for r in rows]
    q, k, v, do, lut, smap = _case(dev, H, L, D, BLKQ, torch.tensor(rows), dtype, L + H)
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, T, BLKQ, 64, scale)
    got = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, T, BLKQ, 64, scale)
    mask = smap[0, 0].bool().repeat_interleave(BLKQ, 0).repeat_interleave(64, 1)[:L, :L]
    for h in range(H) if H < 8 else (0, H // 2, H - 1):
        qf, kf, vf = (t[0, h].float().requires_grad_(True) for t in (q, k, v))
        s = ((qf @ kf.T.contiguous()) * scale).masked_fill(~mask, float("-inf"))
        ref = torch.autograd.grad(torch.softmax(s, -1) @ vf, (qf, kf, vf), do[0, h].float())
        for name, a, r in zip("qkv", got, ref):
            # (probabilities, dS and the result are rounded to 16 bit, at most u = 2^-9 each, within 4 u of the 2-norm)
            err = float((a[0, h].float() - r).norm())
            assert err <= 4 * 2.0 ** -9 * max(float(r.norm()), 1e-3) + 1e-3, (name, h, err)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,BLKQ,sink", [
    (128, 64, False), (64, 128, False),
    (64, 64, True),                                             # lists of 256 entries: four segments, in four strips per head
    (64, 128, True),                                            # 128 entries of two halves each: two segments
])
def test_one_launch_equals_two(dev, H, BLKQ, sink, dtype):
    """The largest call of head dim 128 with one launch (16384 key blocks) and a call with a head more, which has two (work items
    numbered beforehand, delta formed on dQ's way): the same bits per head; and a whole backward with two launches equals the attention's
    gradients with the linear branch's added."""
    from sla_amd.inputs import make_proj
    from sla_amd.linear import linear_bwd
    from sla_amd.module import module_bwd
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    D, N = 128, 16384 // H
    L, M = 64 * N - 7, N // (BLKQ // 64)
    i = torch.arange(M)
    rows = torch.stack([0 * i, 1 + i % (N - 1)] if sink else [i * 5 % N, (i * 5 + 3) % N], 1).sort(1).values
    q, k, v, do, lut, smap = _case(dev, H + 1, L, D, BLKQ, rows, dtype, 1)
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, 2, BLKQ, 64, scale)
    two = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, 2, BLKQ, 64, scale)
    first = [t[:, :H].contiguous() for t in (q, k, v, o, do, lse, smap, lut)]
    one = sparse_attn_bwd(*first, 2, BLKQ, 64, scale)
    for name, a, b in zip("qkv", one, two):
        assert torch.equal(a, b[:, :H]), name
    w, b = (t.to(dev) for t in make_proj(D))
    ref = linear_bwd(q, k, v, w, b, do, "softmax", accumulate_into=two)
    got = module_bwd(q, k, v, o, do, lse, smap, lut, 2, BLKQ, 64, scale, w, b, "softmax")
    for name, a, r in zip(("dq", "dk", "dv", "dw", "db"), got, ref):
        assert torch.equal(a, r), name


@pytest.mark.parametrize("H,L,D", [(32, 4090, 128), (33, 3970, 128)])
def test_linear_keys_on_either_side(dev, H, L, D):
    """2048 key blocks (dK/dV forms the linear branch's dk, dv, too) and 2079: the attention's gradients and the linear branch's added."""
    from sla_amd.inputs import make_proj
    from sla_amd.linear import linear_bwd
    from sla_amd.module import module_bwd
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    N = -(-L // 64)
    rows = torch.stack([torch.zeros(N, dtype=torch.long), 1 + torch.arange(N) % (N - 1)], 1)
    q, k, v, do, lut, smap = _case(dev, H, L, D, 64, rows, torch.bfloat16, H)
    w, b = (t.to(dev) for t in make_proj(D))
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, 2, 64, 64, scale)
    grads = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, 2, 64, 64, scale)
    ref = linear_bwd(q, k, v, w, b, do, "elu", accumulate_into=grads)
    got = module_bwd(q, k, v, o, do, lse, smap, lut, 2, 64, 64, scale, w, b, "elu")
    for name, a, r in zip(("dq", "dk", "dv", "dw", "db"), got, ref):
        assert torch.equal(a, r), name
