"""fp32 inputs: the attention kernels write the module's output as fp32 numbers themselves, the values of the 16-bit output."""
import pytest
import torch

from sla_amd import SparseLinearAttention, get_block_map
from sla_amd.inputs import make_proj
from sla_amd.linear import linear_state_fwd
from sla_amd.sparse_attn import sparse_attn_linear_fwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,D,BLKQ,half", [
    (1, 129, 64, 64, False), (2, 161, 128, 128, True), (3, 290, 128, 64, False),    # one query block per workgroup, partial rows
    (24, 801, 128, 64, True), (24, 833, 64, 128, False)])                            # two, the last one alone
def test_values_of_the_16_bit_output(dev, H, L, D, BLKQ, half):
    dtype = torch.float16 if half else torch.bfloat16
    g = torch.Generator().manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, generator=g).to(dev) for _ in range(3))
    w, b = (t.to(dev) for t in make_proj(D))
    mod = SparseLinearAttention(D, 0.5, "softmax", BLKQ, 64, use_bf16=not half).to(dev)
    with torch.no_grad():
        mod.proj_l.weight.copy_(w)
        mod.proj_l.bias.copy_(b)
        _, lut, T = get_block_map(q, k, 0.5, BLKQ, 64)
        qc, kc, vc = (t.to(dtype) for t in (q, k, v))
        state = linear_state_fwd(kc, vc, w, "softmax")
        ref = sparse_attn_linear_fwd(qc, kc, vc, lut, T, BLKQ, 64, D ** -0.5, state, b, "softmax", want_o_s=False)[0]
        out = mod(q, k, v)
    assert out.dtype == torch.float32 and out.is_contiguous() and torch.equal(out, ref.float())
    assert torch.equal(mod(q, k, v).detach(), out)                                   # through autograd


@pytest.mark.parametrize("H,L,D,BLKQ", [(2, 161, 128, 128), (24, 833, 64, 64)])
def test_16_bit_output_of_fp32_inputs(dev, monkeypatch, H, L, D, BLKQ):
    """The C entry point's other form (in_dtype fp32, output in the compute dtype), which the module does not ask for."""
    from sla_amd import _lib
    g = torch.Generator().manual_seed(L)
    q, k, v = (torch.randn(1, H, L, D, generator=g).to(dev) for _ in range(3))
    mod = SparseLinearAttention(D, 0.5, "elu", BLKQ, 64).to(dev)
    with torch.no_grad():
        for p, t in zip((mod.proj_l.weight, mod.proj_l.bias), make_proj(D)):
            p.copy_(t)
        out = mod(q, k, v)
        monkeypatch.setattr(_lib, "SLA_F32_BOTH", _lib.SLA_F32)      # (fills the first half of the fp32 tensor)
        half = mod(q, k, v).view(-1).view(torch.bfloat16)[:out.numel()].view_as(out)
    assert torch.equal(half.float(), out)
