"""The module forward's shared launches (pooling with the 16-bit copies, partial states with the column mean, finished states with
the block means of k) against the single-step entry points: the same bits, at lengths around a block, a batch of rows in flight,
a group of chunk sums (2048 rows) and a slice, and on either side of the size at which the pooling passes widen their loads."""
import pytest
import torch

from sla_amd import SparseLinearAttention, get_block_map
from sla_amd.inputs import make_proj
from sla_amd.linear import linear_state_fwd
from sla_amd.sparse_attn import sparse_attn_linear_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,L,D,BLKQ,in_dtype,fmap,half", [
    (1, 1, 1, 64, 64, torch.float32, "softmax", False), (1, 2, 63, 128, 128, torch.float32, "elu", True),
    (2, 1, 65, 64, 64, torch.bfloat16, "relu", False), (1, 3, 129, 128, 64, torch.float16, "softmax", True),
    (1, 2, 191, 64, 128, torch.float32, "relu", False), (1, 5, 2049, 128, 128, torch.bfloat16, "softmax", False),
    (1, 2, 4097, 64, 64, torch.float16, "softmax", True), (3, 7, 1023, 128, 64, torch.float32, "elu", False),
    (1, 16, 4160, 64, 64, torch.bfloat16, "elu", False), (1, 8, 8191, 128, 64, torch.bfloat16, "relu", False),
    (2, 40, 321, 64, 64, torch.float32, "softmax", True), (1, 1, 10500, 64, 64, torch.float32, "elu", False),
    (1, 40, 6601, 128, 128, torch.bfloat16, "elu", False), (1, 40, 6601, 128, 64, torch.float32, "softmax", True)])   # (from 64 MiB on)
def test_forward_equals_the_steps(dev, B, H, L, D, BLKQ, in_dtype, fmap, half):
    dtype = torch.float16 if half else torch.bfloat16
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(B, H, L, D, generator=g).to(in_dtype).to(dev) for _ in range(3))
    w, b = (t.to(dev) for t in make_proj(D))
    ratio = 1.0 if L < 256 else 0.3            # (at least one block selected)
    mod = SparseLinearAttention(D, ratio, fmap, BLKQ, 64, use_bf16=not half).to(dev)
    with torch.no_grad():
        mod.proj_l.weight.copy_(w)
        mod.proj_l.bias.copy_(b)
        _, lut, T = get_block_map(q, k, ratio, BLKQ, 64)
        qc, kc, vc = (t.to(dtype) for t in (q, k, v))
        state = linear_state_fwd(kc, vc, w, fmap)
        out, _, _ = sparse_attn_linear_fwd(qc, kc, vc, lut, T, BLKQ, 64, D ** -0.5, state, b, fmap, want_o_s=True)
        assert torch.equal(mod(q, k, v), out.to(in_dtype))
        if in_dtype == dtype:                  # (B, L, H, D) activations read where they lie
            rows = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
            assert torch.equal(mod(*rows), out)


@pytest.mark.parametrize("H,L,D,fmap,half", [(1, 1, 64, "softmax", False), (2, 63, 128, "elu", True), (3, 129, 64, "relu", False),
                                             (5, 2049, 128, "softmax", False), (1, 10500, 64, "elu", False)])
def test_quantised_forward_equals_the_steps(dev, H, L, D, fmap, half):
    """The quantised module's preparation likewise: an odd number of key blocks, less than a block, a state build of many slices."""
    from sla_amd import SageSparseLinearAttention
    from sla_amd.linear import linear_out_fwd, linear_state_quant_v_fwd
    from sla_amd.sage import sage_attn_fwd, sage_prepare
    dtype, ratio = torch.float16 if half else torch.bfloat16, 1.0 if L < 256 else 0.2
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, generator=g).to(dtype).to(dev) for _ in range(3))
    mod = SageSparseLinearAttention(D, ratio, fmap, use_bf16=not half).to(dev)
    with torch.no_grad():
        for p, t in zip((mod.proj_l.weight, mod.proj_l.bias), make_proj(D)):
            p.copy_(t)
        _, lut, T, q8, qs, k8, ks, _, _ = sage_prepare(q, k, None, ratio)
        ws, v8, vs = linear_state_quant_v_fwd(k, v, mod.proj_l.weight, fmap)
        o_s = sage_attn_fwd(q8, qs, k8, ks, v8, vs, lut, T, dtype)
        assert torch.equal(mod(q, k, v), linear_out_fwd(q, mod.proj_l.bias, o_s, ws, fmap))


@pytest.mark.parametrize("H,L,D,fmap,half", [(12, 12287, 128, "elu", False), (12, 12288, 128, "softmax", False), (24, 12289, 64, "relu", True)])
def test_quantised_forward_on_one_stream_equals_the_steps(dev, H, L, D, fmap, half):
    """On either side of the size (36 MiB per tensor) from which the preparation on one stream, here a capturing one, is the separate
    calls' again; replayed several times with eager work between."""
    from sla_amd import SageSparseLinearAttention
    dtype = torch.float16 if half else torch.bfloat16
    g = torch.Generator(device=dev).manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, device=dev, generator=g).to(dtype) for _ in range(3))
    mod = SageSparseLinearAttention(D, 0.05, fmap, use_bf16=not half).to(dev)
    with torch.no_grad():
        for p, t in zip((mod.proj_l.weight, mod.proj_l.bias), make_proj(D)):
            p.copy_(t)
        ref = mod(q, k, v)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = mod(q, k, v)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref)
            assert torch.equal(mod(q, k, v), ref)
            torch.cuda.synchronize()
