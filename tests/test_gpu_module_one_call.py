"""sla_module_fwd / sla_module_bwd_states (what SparseLinearAttention runs) against the single-step entry points they string
together: the same bits, with few and many heads, short and long sequences; a second stream that is handed over stays idle."""
import pytest
import torch

from sla_amd import SageSparseLinearAttention, SparseLinearAttention, _lib, get_block_map
from sla_amd.inputs import make_proj
from sla_amd.linear import linear_bwd, linear_state_fwd
from sla_amd.sparse_attn import sparse_attn_bwd, sparse_attn_linear_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,D,BLKQ,in_dtype,half", [
    (3, 2100, 128, 64, torch.bfloat16, False), (2, 1000, 64, 128, torch.float32, False), (2, 777, 128, 64, torch.float32, True),
    (2, 640, 64, 64, torch.float16, False),          # a mask from half precision, bf16 compute
    (12, 6001, 128, 64, torch.bfloat16, False), (24, 6001, 64, 64, torch.float32, True),
    (2, 30001, 64, 64, torch.bfloat16, False)])
def test_one_call_equals_the_steps(dev, H, L, D, BLKQ, in_dtype, half):
    ratio, fmap, dtype = 0.1, "elu" if not half else "softmax", torch.float16 if half else torch.bfloat16
    g = torch.Generator().manual_seed(L + D)
    q, k, v, do = (torch.randn(1, H, L, D, generator=g).to(in_dtype).to(dev) for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    mod = SparseLinearAttention(D, ratio, fmap, BLKQ, 64, use_bf16=not half).to(dev)
    with torch.no_grad():
        mod.proj_l.weight.copy_(w)
        mod.proj_l.bias.copy_(b)
    # the steps, on one stream
    sparse_map, lut, T = get_block_map(q, k, ratio, BLKQ, 64)
    qc, kc, vc, dc = (t.to(dtype) for t in (q, k, v, do))
    state = linear_state_fwd(kc, vc, w, fmap)
    out, o_s, lse = sparse_attn_linear_fwd(qc, kc, vc, lut, T, BLKQ, 64, D ** -0.5, state, b, fmap, want_o_s=True)
    ref = sparse_attn_bwd(qc, kc, vc, o_s, dc, lse, sparse_map, lut, T, BLKQ, 64, D ** -0.5)
    _, _, _, dw, db = linear_bwd(qc, kc, vc, w, b, dc, fmap, accumulate_into=ref)
    for _ in range(2):                               # (twice: memory of the first call is used again)
        qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
        mod.zero_grad()
        o = mod(qg, kg, vg)
        o.backward(do)
        assert o.dtype == in_dtype and torch.equal(o.detach(), out.to(in_dtype))
        with torch.no_grad():
            assert torch.equal(mod(q, k, v), out.to(in_dtype))
        for name, t, r in zip(("dq", "dk", "dv"), (qg, kg, vg), ref):
            assert torch.equal(t.grad, r.to(in_dtype)), name
        assert torch.equal(mod.proj_l.weight.grad, dw) and torch.equal(mod.proj_l.bias.grad, db)


@pytest.mark.parametrize("in_dtype", [torch.bfloat16, torch.float32])
def test_gradients_own_their_memory(dev, in_dtype):
    """What the backward returns can be detached in place and kept one without the others."""
    mod = SparseLinearAttention(64, 0.5).to(dev)
    x = [torch.randn(1, 2, 256, 64, device=dev, dtype=in_dtype, requires_grad=True) for _ in range(3)]
    inputs = [*x, mod.proj_l.weight, mod.proj_l.bias]
    for t, grad in zip(inputs, torch.autograd.grad(mod(*x).sum(), inputs)):
        assert grad.shape == t.shape and not grad._is_view()
        assert grad.untyped_storage().nbytes() == t.numel() * t.element_size()


def test_fp32_v_off_alignment(dev):
    """An fp32 v that does not lie on 16 bytes is converted by the copy, as any other."""
    q, k, v, do = (torch.randn(1, 2, 300, 64, device=dev) for _ in range(4))
    mod = SparseLinearAttention(64, 0.5).to(dev)
    off = torch.empty(v.numel() + 1, device=dev)[1:].view_as(v).copy_(v)
    assert off.is_contiguous() and off.data_ptr() % 16
    with torch.no_grad():
        assert torch.equal(mod(q, k, off), mod(q, k, v))
    grads = []
    for t in (v, off):
        x = [q.clone().requires_grad_(True), k.clone().requires_grad_(True), t.detach().requires_grad_(True)]
        grads.append(torch.autograd.grad(mod(*x), x, do))
    assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("H,L,D,BLKQ,half", [(3, 2100, 128, 64, False), (2, 1000, 64, 128, True), (12, 6001, 128, 128, True),
                                             (24, 6001, 64, 64, False)])
def test_packed_one_call_equals_the_steps(dev, H, L, D, BLKQ, half):
    """forward_packed, whose calls read q, k, v and write their gradients where the packed tensors hold them, against the
    single-step entry points on the views: the same bits, call after call."""
    ratio, fmap, dtype = 0.1, "elu" if not half else "softmax", torch.float16 if half else torch.bfloat16
    g = torch.Generator().manual_seed(L + D)
    qkv = torch.randn(1, L, 3, H, D, generator=g).to(dtype).to(dev)
    do = torch.randn(1, L, H, D, generator=g).to(dtype).to(dev)
    w, b = (t.to(dev) for t in make_proj(D))
    mod = SparseLinearAttention(D, ratio, fmap, BLKQ, 64, use_bf16=not half).to(dev)
    with torch.no_grad():
        mod.proj_l.weight.copy_(w)
        mod.proj_l.bias.copy_(b)
    q, k, v = (qkv[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    dv = do.permute(0, 2, 1, 3)
    sparse_map, lut, T = get_block_map(q, k, ratio, BLKQ, 64)
    state = linear_state_fwd(k, v, w, fmap)
    out, o_s, lse = sparse_attn_linear_fwd(q, k, v, lut, T, BLKQ, 64, D ** -0.5, state, b, fmap, want_o_s=True)
    ref = torch.empty_like(qkv)
    grads = tuple(ref[:, :, i].permute(0, 2, 1, 3) for i in range(3))
    sparse_attn_bwd(q, k, v, o_s, dv, lse, sparse_map, lut, T, BLKQ, 64, D ** -0.5, grads=grads)
    _, _, _, dw, db = linear_bwd(q, k, v, w, b, dv, fmap, accumulate_into=grads)
    for call in range(2):
        x = qkv.clone().requires_grad_(True)
        mod.zero_grad()
        o = mod.forward_packed(x)
        o.backward(do)
        assert torch.equal(o.detach(), out.permute(0, 2, 1, 3)) and torch.equal(x.grad, ref), call
        assert torch.equal(mod.proj_l.weight.grad, dw) and torch.equal(mod.proj_l.bias.grad, db)
        with torch.no_grad():
            assert torch.equal(mod.forward_packed(qkv), o)


@pytest.mark.parametrize("H,L,D", [(2, 1000, 64), (82, 2001, 128)])          # few launches, and those of large inputs
def test_a_second_stream_stays_idle(dev, monkeypatch, H, L, D):
    """sla_module_fwd, sage_module_fwd and sla_module_bwd_states take the handle of a second stream and put nothing on it: it is idle
    while the calling stream still holds the call back, and the results are those without one."""
    side, lib = torch.cuda.Stream(device=dev), _lib.load()

    class WithSide:
        def __getattr__(self, name):
            entry = getattr(lib, name)
            if not name.endswith(("module_fwd", "module_bwd_states")):
                return entry
            used.add(name)
            return lambda *args: entry(*args[:-1], side.cuda_stream)

    used = set()
    x = [torch.randn(1, H, L, D, device=dev).bfloat16().requires_grad_(True) for _ in range(3)]
    do = torch.randn(1, H, L, D, device=dev).bfloat16()
    mods = [SparseLinearAttention(D, 0.1).to(dev), SageSparseLinearAttention(D, 0.1).to(dev)]
    w, b = (t.to(dev) for t in make_proj(D))
    with torch.no_grad():
        for mod in mods:
            mod.proj_l.weight.copy_(w)
            mod.proj_l.bias.copy_(b)

    def calls():
        out = mods[0](*x)
        return [out.detach(), mods[1](*x), *torch.autograd.grad(out, x, do)]

    ref = calls()
    monkeypatch.setattr(_lib, "load", lambda: WithSide())
    torch.cuda.synchronize()
    torch.cuda._sleep(40_000_000)
    got = calls()
    busy, idle = not torch.cuda.current_stream(dev).query(), side.query()
    torch.cuda.synchronize()
    assert used == {"sla_module_fwd", "sage_module_fwd", "sla_module_bwd_states"} and busy and idle
    for a, r in zip(got, ref):
        assert torch.equal(a, r)
