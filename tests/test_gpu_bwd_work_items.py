"""Work items of dK/dV: counts of (head, key block) pairs around 512, and key blocks that every query block selects, whose lists are
cut into segments that the last workgroup to finish adds up; alone and added to what the gradients hold.  Calls of these sizes find
their items in the launch that dQ shares (from the sums over strips of 64 key blocks); those of rows too far apart have them numbered
beforehand, 512 pairs to a wave, as have the larger calls of test_gpu_bwd_one_launch and the longer rows of test_gpu_bwd_long_rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


@pytest.mark.parametrize("H,N,T", [(511, 1, 1), (512, 1, 1), (171, 3, 2), (342, 3, 2), (8, 130, 3), (3, 171, 4)])
def test_gradients_over_all_pairs(dev, H, N, T):
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    D, L = 64, 64 * N - 5
    g = torch.Generator(device=dev).manual_seed(H)
    q, k, v, do = (torch.randn(1, H, L, D, device=dev, generator=g).bfloat16() for _ in range(4))
    # every row selects key block 0 (a list of N entries, several segments from 65 on) and T - 1 blocks after it
    i = torch.arange(N, device=dev)[:, None]
    lut = torch.cat([torch.zeros(N, 1, dtype=torch.long, device=dev), 1 + (i + torch.arange(T - 1, device=dev)) % max(N - 1, 1)], 1)
    lut = lut.sort(1).values.expand(1, H, N, T).contiguous()
    smap = torch.zeros(1, H, N, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    lut = lut.int()
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, T, 64, 64, scale)
    got = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, T, 64, 64, scale)
    mask = smap[0, 0].bool().repeat_interleave(64, 0).repeat_interleave(64, 1)[:L, :L]
    for h0 in range(0, H, 64 if N < 8 else 1):
        hs = slice(h0, h0 + (64 if N < 8 else 1))
        qf, kf, vf = (t[0, hs].float().requires_grad_(True) for t in (q, k, v))
        s = (torch.bmm(qf, kf.transpose(1, 2).contiguous()) * scale).masked_fill(~mask, float("-inf"))
        ref = torch.autograd.grad(torch.bmm(torch.softmax(s, -1), vf), (qf, kf, vf), do[0, hs].float())
        for name, a, r in zip("qkv", got, ref):
            # (probabilities, dS and the result are rounded to bf16, u = 2^-9 each: within 4 u of the largest 2-norm of a head)
            err = (a[0, hs].float() - r).flatten(1).norm(dim=1)
            assert bool((err <= 4 * 2.0 ** -9 * r.flatten(1).norm(dim=1).clamp_min(1e-3) + 1e-3).all()), (name, h0, err.max().item())


@pytest.mark.parametrize("N", [15, 16, 17, 33, 63, 65, 79, 81, 127])
def test_lists_of_maps_of_any_width(dev, N):
    """Key-block counts around the 16 bytes and the 64 columns the lists are read in, and maps that start at any byte."""
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    H, D, L, T = 2, 64, 64 * N - 9, 5
    g = torch.Generator(device=dev).manual_seed(N)
    q, k, v, do = (torch.randn(1, H, L, D, device=dev, generator=g).bfloat16() for _ in range(4))
    lut = torch.rand(1, H, N, N, device=dev, generator=g).argsort(-1)[..., :T].sort(-1).values.contiguous()
    smap = torch.zeros(1, H, N, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    lut = lut.int()
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, T, 64, 64, scale)
    got = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, T, 64, 64, scale)
    mask = smap[0].bool().repeat_interleave(64, 1).repeat_interleave(64, 2)[:, :L, :L]
    qf, kf, vf = (t[0].float().requires_grad_(True) for t in (q, k, v))
    s = (torch.bmm(qf, kf.transpose(1, 2).contiguous()) * scale).masked_fill(~mask, float("-inf"))
    ref = torch.autograd.grad(torch.bmm(torch.softmax(s, -1), vf), (qf, kf, vf), do[0].float())
    for name, a, r in zip("qkv", got, ref):
        # (as above)
        err = (a[0].float() - r).flatten(1).norm(dim=1)
        assert bool((err <= 4 * 2.0 ** -9 * r.flatten(1).norm(dim=1).clamp_min(1e-3) + 1e-3).all()), (name, err.max().item())
    for first in (1, 6, 15):
        moved = torch.ones(smap.numel() + 16, dtype=torch.int8, device=dev)[first:first + smap.numel()].view_as(smap)
        moved.copy_(smap)
        for a, r in zip(sparse_attn_bwd(q, k, v, o, do, lse, moved, lut, T, 64, 64, scale), got):
            assert torch.equal(a, r), first


@pytest.mark.parametrize("H,L", [(2, 8320), (1, 4161)])
def test_added_to_what_the_gradients_hold(dev, H, L):
    """A whole backward over lists in segments equals the attention's gradients plus the linear branch's, bit for bit."""
    from sla_amd.inputs import make_proj
    from sla_amd.linear import linear_bwd
    from sla_amd.module import module_bwd
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    D, T, N = 128, 2, -(-L // 64)
    g = torch.Generator(device=dev).manual_seed(L)
    q, k, v, do = (torch.randn(1, H, L, D, device=dev, generator=g).bfloat16() for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    lut = torch.stack([torch.zeros(N, dtype=torch.long), 1 + torch.arange(N) % (N - 1)], 1).to(dev).expand(1, H, N, T).contiguous()
    smap = torch.zeros(1, H, N, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    lut = lut.int()
    o, lse = sparse_attn_fwd(q, k, v, lut, T, 64, 64, D ** -0.5)
    grads = sparse_attn_bwd(q, k, v, o, do, lse, smap, lut, T, 64, 64, D ** -0.5)
    ref = linear_bwd(q, k, v, w, b, do, "elu", accumulate_into=grads)
    for _ in range(2):
        got = module_bwd(q, k, v, o, do, lse, smap, lut, T, 64, 64, D ** -0.5, w, b, "elu")
        for a, r in zip(got, ref):
            assert torch.equal(a, r)


@pytest.mark.parametrize("D,BLKQ", [(64, 64), (128, 64), (64, 128)])
def test_rows_too_far_apart_for_the_stream_kernels(dev, D, BLKQ):
    """Heads that span 2 GiB (one buffer of very long rows) go through the general dQ and dK/dV kernels and the sums behind them:
    against dense attention, and a whole backward against the attention's gradients plus the linear branch's, bit for bit.  Every
    row selects key block 0, so that with 64-row blocks its list is cut."""
    from sla_amd.inputs import make_proj
    from sla_amd.linear import linear_bwd
    from sla_amd.module import module_bwd
    from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_fwd
    H, L, T = 2, 4161, 2
    M, N, R = -(-L // BLKQ), -(-L // 64), (2 ** 30 // L + 8) // 8 * 8
    assert 2 * L * R >= 2 ** 31

    def views(buf):
        return [buf.as_strided((1, H, L, D), (L * R, D, R, 1), i * H * D) for i in range(3)]

    g = torch.Generator(device=dev).manual_seed(D + BLKQ)
    q, k, v, do = (torch.randn(1, H, L, D, device=dev, generator=g).bfloat16() for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    lut = torch.stack([torch.zeros(M, dtype=torch.long), 1 + torch.arange(M) % (N - 1)], 1).to(dev).expand(1, H, M, T).contiguous()
    smap = torch.zeros(1, H, M, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    lut = lut.int()
    scale = D ** -0.5
    o, lse = sparse_attn_fwd(q, k, v, lut, T, BLKQ, 64, scale)
    wide = views(torch.empty(L * R, dtype=torch.bfloat16, device=dev))
    for x, t in zip(wide, (q, k, v)):
        x.copy_(t)
    grads = views(torch.full((L * R,), float("nan"), dtype=torch.bfloat16, device=dev))
    sparse_attn_bwd(*wide, o, do, lse, smap, lut, T, BLKQ, 64, scale, grads=grads)
    mask = smap[0].bool().repeat_interleave(BLKQ, 1).repeat_interleave(64, 2)[:, :L, :L]
    qf, kf, vf = (t[0].float().requires_grad_(True) for t in (q, k, v))
    s = (torch.bmm(qf, kf.transpose(1, 2).contiguous()) * scale).masked_fill(~mask, float("-inf"))
    ref = torch.autograd.grad(torch.bmm(torch.softmax(s, -1), vf), (qf, kf, vf), do[0].float())
    for name, a, r in zip("qkv", grads, ref):
        # (as above)
        err = (a[0].float() - r).flatten(1).norm(dim=1)
        assert bool((err <= 4 * 2.0 ** -9 * r.flatten(1).norm(dim=1).clamp_min(1e-3) + 1e-3).all()), (name, err.max().item())
    ref = [t.contiguous() for t in linear_bwd(*wide, w, b, do, "elu", accumulate_into=grads)]
    for t in grads:
        t.fill_(float("nan"))
    got = module_bwd(*wide, o, do, lse, smap, lut, T, BLKQ, 64, scale, w, b, "elu", grads=grads)
    for a, r in zip(got, ref):
        assert torch.equal(a, r)


@pytest.mark.parametrize("H,D,T,whole", [(1, 128, 1, True), (2, 64, 1, True), (33, 64, 1, True), (2, 128, 3, False), (1, 64, 0, False)])
def test_map_with_more_ones_than_topk(dev, H, D, T, whole):
    """A map that contradicts topk (the C entry points accept it): every key block's gradients are written, from the first 64 of its
    query blocks and as many further segments as there is room for, H M T / 64 in the order of the key blocks; nothing else is
    touched.  The whole module's backward, with the linear branch formed in dK/dV (two sizes) and beside it (33 heads), and the attention's."""
    from sla_amd.inputs import make_proj
    from sla_amd.module import module_bwd
    from sla_amd.sparse_attn import sparse_attn_bwd
    M, L = 128, 128 * 64 - 3
    g = torch.Generator(device=dev).manual_seed(D + T)
    q, k, v, o, do = (torch.randn(1, H, L, D, device=dev, generator=g).bfloat16() for _ in range(5))
    lse = 6 + torch.rand(1, H, L, device=dev, generator=g)
    w, b = (t.to(dev) for t in make_proj(D))
    lut = torch.arange(M, device=dev, dtype=torch.int32).expand(1, H, M, M).contiguous()

    def run(smap):
        table = lut[..., :T].contiguous()
        grads = tuple(torch.full((1, H, L, D), float("nan"), dtype=torch.bfloat16, device=dev) for _ in range(3))
        if whole:
            return module_bwd(q, k, v, o, do, lse, smap, table, T, 64, 64, D ** -0.5, w, b, "elu", grads=grads)[1:3]
        return sparse_attn_bwd(q, k, v, o, do, lse, smap, table, T, 64, 64, D ** -0.5)[1:3]

    ones = torch.ones(1, H, M, M, dtype=torch.int8, device=dev)
    got = run(ones)
    kept = torch.ones(H * M, dtype=torch.long, device=dev)
    kept[:H * M * T // 64] = 2                                # (each list of 128 has one segment beyond its first)
    rows = torch.arange(M, device=dev)[:, None]
    ref = run((rows < 64 * kept.view(1, H, 1, M)).to(torch.int8))         # (fills the room and no more)
    for name, a, r in zip(("dk", "dv"), got, ref):
        assert torch.isfinite(a).all() and torch.equal(a, r), name
