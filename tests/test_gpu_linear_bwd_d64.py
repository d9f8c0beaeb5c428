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


def _float64(q, k, v, w, do, fmap):
    """Gradients in 64 bits, and the 2-norms of the terms they are sums of (the divisor held fixed)."""
    x = [t.double().requires_grad_(True) for t in (q, k, v, w)]
    a, c = _phi(x[0], fmap), _phi(x[1], fmap)
    den = 1e-5 + (a * c.sum(-2, keepdim=True)).sum(-1, keepdim=True)
    out = (a @ (c.transpose(-1, -2).contiguous() @ x[2]) / den) @ x[3].t().contiguous()
    ref = [*torch.autograd.grad(out, x, do.double()), do.double().sum((0, 1, 2))]
    y = [t.detach().clone().requires_grad_(True) for t in x]
    a2, c2 = _phi(y[0], fmap), _phi(y[1], fmap)
    out2 = (a2 @ (c2.transpose(-1, -2).contiguous() @ y[2]) / den.detach()) @ y[3].t().contiguous()
    return ref, [*torch.autograd.grad(out2, y, do.double()), ref[4]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("projection", ["zero", "random"])
@pytest.mark.parametrize("fmap", ["relu", "elu", "softmax"])
@pytest.mark.parametrize("D", [64, 128])
def test_rows_without_weight(dev, D, fmap, projection, dtype):
    """Query rows of zeros (padding) and, with the relu map, of no positive value: their divisor is 1e-5 and d(out) over it is
    past half precision's range.  A component that is positive in no key but in such a row is past it in phi(q) / den as well."""
    from sla_amd.linear import linear_bwd
    B, H, L = 1, 2, 200
    gen = torch.Generator(device=dev).manual_seed(D)
    q, k, v = (torch.randn(B, H, L, D, device=dev, generator=gen).to(dtype) for _ in range(3))
    do = (8 * torch.randn(B, H, L, D, device=dev, generator=gen)).to(dtype)
    q[:, :, 3] = 0
    q[:, :, 17:40] = 0
    q[:, :, 130] = -q[:, :, 130].abs()
    w, b = (t.to(dev) for t in make_proj(D))
    if projection == "zero":
        w = torch.zeros_like(w)
    got = linear_bwd(q, k, v, w, b, do, fmap)
    ref, mag = _float64(q, k, v, w, do, fmap)
    u = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    for i, (g, r, m) in enumerate(zip(got, ref, mag)):
        assert torch.isfinite(g).all(), i
        # (as above)
        assert (g.double() - r).norm() <= 8 * u * (r.norm() + m.norm()), i
    # (with a projection the state's gradient of that component is past half precision's range itself)
    if D == 64 and fmap == "relu" and (projection == "zero" or dtype == torch.bfloat16):
        k[..., 5] = -k[..., 5].abs()
        q[:, :, 3, 5] = 3
        got = linear_bwd(q, k, v, w, b, do, fmap)
        ref, mag = _float64(q, k, v, w, do, fmap)
        for i in range(1, 5):              # (dq of that row is a number over 1e-5 in any arithmetic)
            assert torch.isfinite(got[i]).all(), i
            assert (got[i].double() - ref[i]).norm() <= 8 * u * (ref[i].norm() + mag[i].norm()), i


@pytest.mark.parametrize("scale", [2.0 ** -13, 1.0, 2.0 ** 12])
@pytest.mark.parametrize("fmap,L", [("softmax", 6001), ("elu", 500)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_weight_gradients_of_small_and_large_gradients(dev, dtype, fmap, L, scale):
    """d_weight and d_bias, which are 32-bit, keep their precision whatever the size of d(out) and of the divisor."""
    from sla_amd.linear import linear_bwd
    B, H, D = 1, 2, 64
    gen = torch.Generator(device=dev).manual_seed(L)
    q, k, v, do = (torch.randn(B, H, L, D, device=dev, generator=gen) for _ in range(4))
    # (values of d(out) that half precision holds exactly, so that their own rounding is no part of the comparison)
    do = scale * do.bfloat16().float().clamp(-8, 8)
    q, k, v, do = (t.to(dtype) for t in (q, k, v, do))
    w, b = (t.to(dev) for t in make_proj(D))
    got = linear_bwd(q, k, v, w, b, do, fmap)
    ref, mag = _float64(q, k, v, w, do, fmap)
    u = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    for i in (3, 4):
        # (as above)
        bound = 8 * u * (ref[i].norm() + mag[i].norm())
        assert (got[i].double() - ref[i]).norm() <= bound, (i, ((got[i].double() - ref[i]).norm() / bound).item())


@pytest.mark.parametrize("L", [4992, 4993, 9990])
@pytest.mark.parametrize("D,dtype", [(64, torch.float16), (128, torch.bfloat16)])
def test_sums_over_many_slices(dev, D, dtype, L):
    """39, 40 and 79 slices of 128 rows: from 40 on a launch of its own adds the slices' sums up."""
    from sla_amd.linear import linear_bwd
    B, H = 1, 2
    gen = torch.Generator(device=dev).manual_seed(L)
    q, k, v, do = (torch.randn(B, H, L, D, device=dev, generator=gen).to(dtype) for _ in range(4))
    w, b = (t.to(dev) for t in make_proj(D))
    got = linear_bwd(q, k, v, w, b, do, "softmax")
    ref, mag = _float64(q, k, v, w, do, "softmax")
    u = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)
    for i, (g, r, m) in enumerate(zip(got, ref, mag)):
        # (as above; the sums over the rows are in 32 bits)
        assert (g.double() - r).norm() <= 8 * u * (r.norm() + m.norm()), i
