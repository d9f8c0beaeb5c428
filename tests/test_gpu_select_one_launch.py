"""Scores and selection in one launch: key-block counts around its tiles of 16 and 32 blocks and the lengths at which its rows take
one, two or four keys per lane, more (257 blocks of 16-bit inputs) or leave it (129 of fp32), against the CPU oracle, bit for bit."""
import pytest
import torch

from oracle import sla_oracle as O
from sla_amd import get_block_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 128), (torch.float16, 64), (torch.float32, 64), (torch.float32, 128)])
@pytest.mark.parametrize("N,ratio", [(1, 1.0), (15, 0.2), (16, 0.3), (17, 0.5), (32, 0.2), (33, 0.2), (63, 1.0), (65, 0.1), (127, 0.05),
                                     (128, 0.7), (129, 0.05), (200, 0.2), (255, 0.5), (256, 0.1), (257, 0.1)])
def test_rows_of_any_length(dev, dtype, D, N, ratio):
    g = torch.Generator().manual_seed(N + D)
    L = 8 * N - (3 if N % 2 else 0)
    q = torch.randn(1, 3, L, D, generator=g).to(dtype)
    k = (torch.randn(1, 3, L, D, generator=g) + 0.3).to(dtype)
    for BLKQ in (8, 16):
        m_ref, lut_ref, T = O.get_block_map(q, k, ratio, BLKQ, 8)
        m, lut, _ = get_block_map(q.to(dev), k.to(dev), ratio, BLKQ, 8)
        assert torch.equal(m.cpu(), m_ref) and torch.equal(lut.cpu(), lut_ref), BLKQ


@pytest.mark.parametrize("H", [16, 17])
def test_equal_scores(dev, H):
    """Small integers: many exact ties, 256 and 272 workgroups of 16 rows."""
    g = torch.Generator().manual_seed(H)
    q, k = (torch.randint(-1, 2, (1, H, 2048, 64), generator=g).bfloat16() for _ in range(2))
    m_ref, lut_ref, T = O.get_block_map(q, k, 0.2, 8, 8)
    m, lut, _ = get_block_map(q.to(dev), k.to(dev), 0.2, 8, 8)
    assert torch.equal(m.cpu(), m_ref) and torch.equal(lut.cpu(), lut_ref)
