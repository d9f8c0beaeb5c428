"""The backward kernels at the edges of their loops: table rows of one to three key blocks (the rotated loop's
prologue and tail meet), lists of none to many query blocks, last blocks whose halves of 32 rows are short, full or missing."""
import pytest
import torch

from oracle import sla_oracle as O
from sla_amd import _attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,L,T,BLKQ,dtype", [(27, 769, 1, 64, torch.bfloat16),     # one row in the last block
                                               (27, 800, 2, 64, torch.float16),      # its first half full, no second one
                                               (27, 801, 3, 64, torch.bfloat16),     # one row in the second half
                                               (28, 768, 12, 64, torch.bfloat16),    # every key block
                                               (80, 801, 1, 128, torch.bfloat16),    # 128-row blocks, the last without a second half
                                               (80, 831, 2, 128, torch.float16)])
@pytest.mark.parametrize("D", [128, 64])
def test_short_rows_and_lists(dev, H, L, T, BLKQ, dtype, D):
    g = torch.Generator().manual_seed(L + T)
    q, k, v, do = (torch.randn(1, H, L, D, generator=g).to(dtype) for _ in range(4))
    M, N = -(-L // BLKQ), -(-L // 64)
    # the last key block in every third row, the others drawn from the first half of the rest: some lists stay empty
    lut = torch.stack([torch.randperm(N if T == N else max(N // 2, T), generator=g)[:T] for _ in range(H * M)])
    if T < N:
        lut[::3, -1] = N - 1
    lut = lut.sort(-1).values.view(1, H, M, T)
    m = torch.zeros(1, H, M, N, dtype=torch.int8).scatter_(-1, lut, 1)
    o_ref, lse_ref = O.sparse_attn_fwd_dense(q, k, v, m, BLKQ, 64)
    refs = O.sparse_attn_bwd_dense(q, k, v, o_ref, do, lse_ref, m, BLKQ, 64)
    qd, kd, vd = (t.to(dev).requires_grad_(True) for t in (q, k, v))
    o = _attention.apply(qd, kd, vd, m.to(dev), lut.to(dev), T, BLKQ, 64)
    o.backward(do.to(dev))
    # P, dS, the forward's output behind delta and the result are rounded to 16 bit (at most 2^-8 each), everything else is
    # fp32: the errors of one product's terms are independent, so the 2-norm stays well under the sum of the four
    for name, t, ref in zip(("dq", "dk", "dv"), (qd, kd, vd), refs):
        err = (t.grad.cpu().double() - ref.double()).norm() / ref.double().norm()
        assert err <= 4 * 2.0 ** -8, (name, float(err))
