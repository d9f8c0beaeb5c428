"""The quantised module's scales of v from the slices' maxima, at slice counts on either side of the sixteen loads it keeps in flight:
the same bits as the separate calls."""
import pytest
import torch

from sla_amd import SageSparseLinearAttention
from sla_amd.inputs import make_proj
from sla_amd.linear import linear_out_fwd, linear_state_quant_v_fwd
from sla_amd.sage import sage_attn_fwd, sage_prepare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,D", [(2, 64, 128), (3, 129, 64), (1, 960, 128), (2, 1024, 128), (1, 4352, 64), (1, 7900, 64), (3, 8192, 128),
                                   (1, 8200, 128), (129, 1300, 64)])      # 1, 2, 15, 16, 17, 31, 32, 33 and 3 slices
def test_module_equals_the_steps(dev, H, L, D):
    g = torch.Generator(device=dev).manual_seed(L + D)
    q, k, v = (torch.randn(1, H, L, D, device=dev, generator=g).bfloat16() for _ in range(3))
    v[:, :, -1] *= 3                           # (the last slice's maxima count)
    v[:, 0, 0, ::2] *= 5
    ratio = 1.0 if L < 256 else 0.5            # (at least one block selected)
    mod = SageSparseLinearAttention(D, ratio, "elu").to(dev)
    with torch.no_grad():
        for p, t in zip((mod.proj_l.weight, mod.proj_l.bias), make_proj(D)):
            p.copy_(t)
        _, lut, T, q8, qs, k8, ks, _, _ = sage_prepare(q, k, None, ratio)
        ws, v8, vs = linear_state_quant_v_fwd(k, v, mod.proj_l.weight, "elu")
        o_s = sage_attn_fwd(q8, qs, k8, ks, v8, vs, lut, T, torch.bfloat16)
        assert torch.equal(mod(q, k, v), linear_out_fwd(q, mod.proj_l.bias, o_s, ws, "elu"))
