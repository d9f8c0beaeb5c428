"""Complement-mode linear branch (linear attention over the non-selected key blocks) vs the brute-force oracle."""
import pytest
import torch

from conftest import cos_sim, max_abs
from oracle import sla_oracle as O
from sla_amd import SparseLinearAttention, _lib
from sla_amd.inputs import CONFIGS, make_inputs, make_proj
from sla_amd.linear import linear_bwd, linear_complement_bwd, linear_complement_fwd, linear_fwd

pytestmark = pytest.mark.gpu

TOL_ABS = 2e-2
TOL_COS = 0.999


@pytest.mark.parametrize("fmap", ["elu", "relu", "softmax"])
@pytest.mark.parametrize("L,D,BLKQ,ratio", [(512, 128, 64, 0.25), (1000, 128, 128, 0.3), (333, 64, 64, 0.5), (700, 64, 128, 0.2)])
def test_complement_vs_oracle(dev, fmap, L, D, BLKQ, ratio):
    g = torch.Generator().manual_seed(L + D)
    q, k, v, res = (torch.randn(1, 2, L, D, generator=g).to(torch.bfloat16) for _ in range(4))
    w, b = make_proj(D)
    m, lut, T = O.get_block_map(q, k, ratio, BLKQ, 64)
    ref = O.linear_branch_complement(q, k, v, lut, w, b, fmap, BLKQ, 64, torch.float32).float() + res.float()
    out = linear_complement_fwd(q.to(dev), k.to(dev), v.to(dev), lut.to(dev), T, w.to(dev), b.to(dev), res.to(dev), fmap,
                                BLKQ, 64).cpu()
    assert out.dtype == torch.bfloat16
    assert max_abs(out, ref) <= TOL_ABS and cos_sim(out, ref) >= TOL_COS


def test_empty_selection_equals_global_branch(dev):
    """With nothing selected the complement is everything: same result as the global linear branch up to the
    16-bit rounding of the per-block states and of the unfolded projection."""
    g = torch.Generator().manual_seed(11)
    q, k, v = (torch.randn(1, 2, 640, 128, generator=g).to(torch.bfloat16).to(dev) for _ in range(3))
    w, b = (t.to(dev) for t in make_proj(128))
    lut = torch.zeros((1, 2, 10, 0), dtype=torch.int64, device=dev)
    out = linear_complement_fwd(q, k, v, lut, 0, w, b, None, "elu")
    ref = linear_fwd(q, k, v, w, b, None, "elu")
    assert max_abs(out.cpu(), ref.cpu()) <= TOL_ABS and cos_sim(out.cpu(), ref.cpu()) >= TOL_COS


def test_int32_lut_and_module_option(dev):
    cfg = CONFIGS["cfg2"]
    d = make_inputs(cfg, H=2)
    q, k, v = (d[x] for x in "qkv")
    w, b = make_proj(cfg.D)
    mod = SparseLinearAttention(cfg.D, cfg.topk, "relu", cfg.BLKQ, cfg.BLKK, linear_mode="complement").to(dev)
    with torch.no_grad():
        mod.proj_l.weight.copy_(w)
        mod.proj_l.bias.copy_(b)
        o = mod(q.to(dev), k.to(dev), v.to(dev)).cpu()
    m, lut, T = O.get_block_map(q, k, cfg.topk, cfg.BLKQ, cfg.BLKK)
    o_s, _ = O.sparse_attn_fwd_gather(q, k, v, lut, cfg.BLKQ, cfg.BLKK)
    ref = o_s.float() + O.linear_branch_complement(q, k, v, lut, w, b, "relu", cfg.BLKQ, cfg.BLKK, torch.float32).float()
    assert max_abs(o, ref) <= TOL_ABS and cos_sim(o, ref) >= TOL_COS
    out32 = linear_complement_fwd(q.to(dev), k.to(dev), v.to(dev), lut.to(dev).int(), T, w.to(dev), b.to(dev), None, "relu")
    out64 = linear_complement_fwd(q.to(dev), k.to(dev), v.to(dev), lut.to(dev), T, w.to(dev), b.to(dev), None, "relu")
    assert torch.equal(out32, out64)
    with pytest.raises(NotImplementedError):
        SparseLinearAttention(cfg.D, cfg.topk, "relu", linear_mode="selected")


def _oracle_grads(q, k, v, lut, w, b, g, fmap, BLKQ):
    leaves = [t.float().clone().requires_grad_(True) for t in (q, k, v, w, b)]
    O.linear_branch_complement(*leaves[:3], lut, *leaves[3:], fmap, BLKQ, 64, torch.float32).backward(g.float())
    return [t.grad for t in leaves]


def _check_grads(got, refs):
    for name, a, r in zip(("dq", "dk", "dv", "dW", "db"), got, refs):
        a = a.cpu()
        scale = max(1.0, float(r.abs().max()))          # dW/db are sums over B*H*L rows
        assert max_abs(a, r) <= TOL_ABS * scale, (name, max_abs(a, r), scale)
        assert cos_sim(a, r) >= TOL_COS, (name, cos_sim(a, r))


@pytest.mark.parametrize("fmap", ["elu", "relu", "softmax"])
@pytest.mark.parametrize("L,D,BLKQ,ratio", [(512, 128, 64, 0.25), (1000, 128, 128, 0.3), (333, 64, 64, 0.5), (700, 64, 128, 0.2),
                                            (150, 128, 64, 0.4)])
def test_complement_backward_vs_autograd_oracle(dev, fmap, L, D, BLKQ, ratio):
    gen = torch.Generator().manual_seed(L + D + 1)
    q, k, v, g = (torch.randn(2, 2, L, D, generator=gen).to(torch.bfloat16) for _ in range(4))
    w, b = make_proj(D)
    m, lut, T = O.get_block_map(q, k, ratio, BLKQ, 64)
    refs = _oracle_grads(q, k, v, lut, w, b, g, fmap, BLKQ)
    args = [t.to(dev) for t in (q, k, v, m, lut)]
    got = linear_complement_bwd(*args, T, w.to(dev), b.to(dev), g.to(dev), fmap, BLKQ, 64)
    _check_grads(got, refs)
    # adding into existing gradients: one more 16-bit rounding of the sum
    base = [torch.randn(2, 2, L, D, generator=gen).to(torch.bfloat16).to(dev) for _ in range(3)]
    acc = linear_complement_bwd(*args, T, w.to(dev), b.to(dev), g.to(dev), fmap, BLKQ, 64,
                                accumulate_into=tuple(t.clone() for t in base))
    for a, x, y in zip(acc[:3], base, got[:3]):
        assert torch.equal(a, (x.float() + y.float()).to(torch.bfloat16))
    assert torch.equal(acc[3], got[3]) and torch.equal(acc[4], got[4])


def test_backward_with_nothing_selected_equals_the_global_backward(dev):
    gen = torch.Generator().manual_seed(13)
    q, k, v, g = (torch.randn(1, 2, 640, 128, generator=gen).to(torch.bfloat16).to(dev) for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(128))
    lut = torch.zeros((1, 2, 10, 0), dtype=torch.int64, device=dev)
    m = torch.zeros((1, 2, 10, 10), dtype=torch.int8, device=dev)
    got = linear_complement_bwd(q, k, v, m, lut, 0, w, b, g, "elu")
    ref = linear_bwd(q, k, v, w, b, g, "elu")
    _check_grads(got, [t.cpu().float() for t in ref])


def test_module_trains_in_complement_mode(dev):
    cfg = CONFIGS["cfg2"]
    d = make_inputs(cfg, H=2)
    q, k, v, do = (d[x] for x in ("q", "k", "v", "do"))
    w, b = make_proj(cfg.D)
    mod = SparseLinearAttention(cfg.D, cfg.topk, "softmax", cfg.BLKQ, cfg.BLKK, linear_mode="complement").to(dev)
    with torch.no_grad():
        mod.proj_l.weight.copy_(w)
        mod.proj_l.bias.copy_(b)
    qd, kd, vd = (t.to(dev).requires_grad_(True) for t in (q, k, v))
    mod(qd, kd, vd).backward(do.to(dev))
    m, lut, T = O.get_block_map(q, k, cfg.topk, cfg.BLKQ, cfg.BLKK)
    o_s, lse = O.sparse_attn_fwd_gather(q, k, v, lut, cfg.BLKQ, cfg.BLKK)
    sp = O.sparse_attn_bwd_gather(q, k, v, o_s, do, lse, lut, cfg.BLKQ, cfg.BLKK)
    lin = _oracle_grads(q, k, v, lut, w, b, do, "softmax", cfg.BLKQ)
    refs = [a + c for a, c in zip(sp, lin[:3])] + lin[3:]
    _check_grads((qd.grad, kd.grad, vd.grad, mod.proj_l.weight.grad, mod.proj_l.bias.grad), refs)


def test_everything_selected_leaves_the_bias_and_no_gradient(dev):
    """topk = 1: the complement is empty.  The difference of the two state sums is then exactly zero (not their
    rounding residue, which the 1e-5 of the divisor would amplify): the branch is the bias, and only the bias has a gradient."""
    from sla_amd import _attention
    gen = torch.Generator().manual_seed(17)
    q, k, v, g = (torch.randn(1, 2, 333, 128, generator=gen).to(torch.bfloat16).to(dev) for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(128))
    for BLKQ in (64, 128):
        M, N = -(-333 // BLKQ), 6
        lut = torch.arange(N, device=dev).expand(1, 2, M, N).contiguous()
        m = torch.ones(1, 2, M, N, dtype=torch.int8, device=dev)
        out = linear_complement_fwd(q, k, v, lut, N, w, b, None, "elu", BLKQ, 64)
        assert torch.equal(out, b.to(torch.bfloat16).expand_as(out))
        dq, dk, dv, dw, db = linear_complement_bwd(q, k, v, m, lut, N, w, b, g, "elu", BLKQ, 64)
        for t in (dq, dk, dv, dw):
            assert int(torch.count_nonzero(t)) == 0
        assert max_abs(db.cpu(), g.float().sum((0, 1, 2)).cpu()) <= 1e-2 * float(g.float().sum((0, 1, 2)).abs().max())


def _dense(q, k, v, lut, w, b, BLKQ):
    """The definition in fp32 with the block states as matrices: H = (all - selected) @ h."""
    L, D = q.shape[-2:]
    M, N = lut.shape[2], -(-L // 64)
    pad = lambda t, n: torch.nn.functional.pad(t, (0, 0, 0, n - L))  # noqa: E731
    phi = lambda t: torch.nn.functional.elu(t) + 1  # noqa: E731
    fk, vv = (pad(t, N * 64).unflatten(2, (N, 64)) for t in (phi(k), v))
    fq = pad(phi(q), M * BLKQ).unflatten(2, (M, BLKQ))
    rest = 1 - torch.zeros(*lut.shape[:2], M, N).scatter_(3, lut, 1.0)
    H = (rest @ (fk.transpose(-1, -2) @ vv).flatten(3)).unflatten(3, (D, D))
    z = rest @ fk.sum(3)
    o = (fq @ H) / (1e-5 + fq @ z.unsqueeze(-1))
    return o.flatten(2, 3)[:, :, :L] @ w.T + b


@pytest.mark.parametrize("L,D,BLKQ,T", [
    (300 * 64 - 17, 64, 64, 257),       # lists too long for the union of neighbouring lists
    (263 * 64, 64, 128, 256),           # the longest it takes
    (9 * 64 + 1, 128, 64, 1), (33 * 64 - 5, 128, 64, 7), (40 * 64, 128, 128, 30), (64, 128, 64, 0)])
def test_gather_over_groups_of_lists(dev, L, D, BLKQ, T):
    """Lists of random entries (every one names block 0, so that block's list of query blocks names all of them), groups of
    fewer than eight rows at the end; the states handed to the backward give the same bits as those it forms."""
    gen = torch.Generator().manual_seed(L + T)
    q, k, v, g = (torch.randn(1, 2, L, D, generator=gen).to(torch.bfloat16) for _ in range(4))
    w, b = make_proj(D)
    M, N = -(-L // BLKQ), -(-L // 64)
    order = torch.rand(1, 2, M, N, generator=gen)
    order[..., 0] = -1.0
    lut = order.argsort(-1)[..., :T].sort(-1).values.contiguous()
    m = torch.zeros(1, 2, M, N, dtype=torch.int8).scatter_(3, lut, 1)
    leaves = [t.float().clone().requires_grad_(True) for t in (q, k, v, w, b)]
    ref = _dense(*leaves[:3], lut, *leaves[3:], BLKQ)
    ref.backward(g.float())
    q, k, v, g, w, b, m, lut = (t.to(dev) for t in (q, k, v, g, w, b, m, lut))
    out, states = linear_complement_fwd(q, k, v, lut, T, w, b, None, "elu", BLKQ, 64, keep_states=True)
    assert torch.equal(out, linear_complement_fwd(q, k, v, lut.int(), T, w, b, None, "elu", BLKQ, 64))
    assert max_abs(out.cpu(), ref.detach()) <= TOL_ABS and cos_sim(out.cpu(), ref.detach()) >= TOL_COS
    got = linear_complement_bwd(q, k, v, m, lut, T, w, b, g, "elu", BLKQ, 64, states=states)
    for a, c in zip(got, linear_complement_bwd(q, k, v, m, lut, T, w, b, g, "elu", BLKQ, 64)):
        assert torch.equal(a, c)
    _check_grads(got, [t.grad for t in leaves])


@pytest.mark.parametrize("H,L,D,BLKQ,T", [
    (20, 16333, 128, 64, 3),            # two groups of heads in a place of their own
    (36, 65000, 128, 64, 2),            # ten groups, in the place of the groups' sums
    (19, 66000, 64, 64, 4), (7, 75600, 128, 128, 2)])
def test_states_of_a_few_heads_at_a_time(dev, H, L, D, BLKQ, T):
    """Forward and backward that do not keep the query blocks' states form them for a group of heads at a time: the bits of
    the calls that hold all of them."""
    g = torch.Generator(device=dev).manual_seed(L)
    q, k, v, do = (torch.randn(1, H, L, D, generator=g, device=dev).bfloat16() for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    M, N = -(-L // BLKQ), -(-L // 64)
    lut = torch.rand(1, H, M, N, generator=g, device=dev).topk(T, -1).indices.sort(-1).values.contiguous()
    m = torch.zeros(1, H, M, N, dtype=torch.int8, device=dev).scatter_(3, lut, 1)
    out, states = linear_complement_fwd(q, k, v, lut, T, w, b, v, "softmax", BLKQ, 64, keep_states=True)
    for table in (lut, lut.int()):
        assert torch.equal(out, linear_complement_fwd(q, k, v, table, T, w, b, v, "softmax", BLKQ, 64))
    ref = linear_complement_bwd(q, k, v, m, lut, T, w, b, do, "softmax", BLKQ, 64, states=states)
    for a, c in zip(linear_complement_bwd(q, k, v, m, lut, T, w, b, do, "softmax", BLKQ, 64), ref):
        assert torch.equal(a, c)


def test_inference_does_not_keep_the_states(dev):
    """Under no_grad, with parameters that could have a gradient, a forward takes no memory for the query blocks' states
    beyond what it holds at a time."""
    H, L, D = 16, 32760, 128
    q, k, v = (torch.randn(1, H, L, D, device=dev).bfloat16() for _ in range(3))
    mod = SparseLinearAttention(D, 0.02, "elu", linear_mode="complement").to(dev)
    size = lambda op: _lib.workspace_bytes(op, _lib.SLA_BF16, 1, H, L, D, 64, 64, 10)  # noqa: E731
    with torch.no_grad():
        ref = mod(q, k, v)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        assert torch.equal(mod(q, k, v), ref)
    used = torch.cuda.max_memory_allocated() - before
    tensors = 2 * q.numel() * 2 + H * L * 4 + (H * 512 * (512 + 10 * 8))          # attention output and result, lse, map, table
    assert used <= tensors + size(_lib.WS_LINEAR_COMPLEMENT) + (16 << 20), used
    assert size(_lib.WS_LINEAR_COMPLEMENT_STATES) > (128 << 20)


@pytest.mark.parametrize("L,D,BLKQ,T", [
    (129 * 64 - 3, 128, 64, 5),         # one row, and one step of 64 block states, past a tile of 128 rows
    (128 * 64, 64, 64, 127), (65 * 64, 128, 128, 64),
    (31 * 64 + 1, 64, 128, 2), (191 * 64, 128, 64, 190)])
def test_states_at_the_edges_of_their_tiles(dev, L, D, BLKQ, T):
    """The states H_i, z_i that a forward keeps, against the sums over the non-selected blocks in 64 bits.  Integers throughout
    (relu, small k and v): the block states are exact in 16 bits, z and the sums exact in 32, so H is the one rounding of the
    exact sum and z exact."""
    gen = torch.Generator().manual_seed(L + T)
    q, k, v = (torch.randint(lo, 2, (1, 2, L, D), generator=gen).to(torch.bfloat16) for lo in (0, 0, -1))
    w, b = make_proj(D)
    M, N = -(-L // BLKQ), -(-L // 64)
    lut = torch.rand(1, 2, M, N, generator=gen).argsort(-1)[..., :T].sort(-1).values.contiguous()
    _, states = linear_complement_fwd(*(t.to(dev) for t in (q, k, v, lut)), T, w.to(dev), b.to(dev), None, "relu", BLKQ, 64,
                                      keep_states=True)
    raw, n = states.cpu().view(torch.uint8).flatten(), 2 * M * D * D * 2
    H = raw[:n].view(torch.bfloat16).view(2, M, D, D)
    at = -(-n // 256) * 256
    z = raw[at:at + 2 * M * D * 4].view(torch.float32).view(2, M, D)
    kb, vb = (torch.nn.functional.pad(t[0].double(), (0, 0, 0, N * 64 - L)).unflatten(1, (N, 64)) for t in (k, v))
    rest = 1 - torch.zeros(2, M, N, dtype=torch.float64).scatter_(2, lut[0], 1.0)
    want_h = (rest @ (vb.transpose(-1, -2) @ kb).flatten(2)).unflatten(2, (D, D))          # (transposed: [d2][d1])
    assert torch.equal(H, want_h.to(torch.bfloat16))
    assert torch.equal(z.double(), rest @ kb.sum(2))
