"""Linear branch's backward at head dim 64 through its streaming kernels: lengths around the 16 rows of a wave, the 128 of a
step and the ends of slices, both layouts, both 16-bit types, against 64-bit autograd."""
import pytest
import torch

from sla_amd.inputs import make_proj

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return torch.device("cuda:0")


def _phi(x, fmap):
    if fmap == "elu":
        return torch.nn.functional.elu(x) + 1
    return torch.relu(x) if fmap == "relu" else torch.softmax(x, -1)


@pytest.mark.parametrize("L", [1, 15, 17, 127, 129, 1153])
@pytest.mark.parametrize("fmap,dtype", [("elu", torch.bfloat16), ("relu", torch.bfloat16), ("softmax", torch.bfloat16),
                                        ("softmax", torch.float16)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_against_float64(dev, L, fmap, dtype, accumulate):
    from sla_amd.linear import linear_bwd
    B, H, D = 2, 3, 64
    gen = torch.Generator(device=dev).manual_seed(L)
    q, k, v, do = (torch.randn(B, H, L, D, device=dev, generator=gen).to(dtype) for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    base = [torch.randn(B, H, L, D, device=dev, generator=gen).to(dtype) for _ in range(3)]
    into = tuple(t.clone() for t in base) if accumulate else None
    got = linear_bwd(q, k, v, w, b, do, fmap, accumulate_into=into)
    x = [t.double().requires_grad_(True) for t in (q, k, v, w)]
    a, c = _phi(x[0], fmap), _phi(x[1], fmap)
    den = 1e-5 + (a * c.sum(-2, keepdim=True)).sum(-1, keepdim=True)
    out = (a @ (c.transpose(-1, -2).contiguous() @ x[2]) / den) @ x[3].t().contiguous()
    ref = [*torch.autograd.grad(out, x, do.double()), do.double().sum((0, 1, 2))]
    # Each gradient is a few products of values rounded to the 16-bit type (half a unit in the last place each, u = 2^-9 or
    # 2^-12), and dq, dk take a difference of sums of the same size: within 8 u of the 2-norm of the terms, which for one or a
    # few rows is that of the summed magnitudes, not of the result.
    u = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    # |terms|: the gradients without the cancelling normalisation (the divisor held fixed)
    y = [t.detach().clone().requires_grad_(True) for t in x]
    a2, c2 = _phi(y[0], fmap), _phi(y[1], fmap)
    out2 = (a2 @ (c2.transpose(-1, -2).contiguous() @ y[2]) / den.detach()) @ y[3].t().contiguous()
    mag = [*torch.autograd.grad(out2, y, do.double()), ref[4]]
    for i, (g, r, m) in enumerate(zip(got, ref, mag)):
        assert torch.isfinite(g).all()
        if accumulate and i < 3:
            r = base[i].double() + r
        bound = 8 * u * (r.norm() + m.norm())
        assert (g.double() - r).norm() <= bound, (i, ((g.double() - r).norm() / bound).item())
