"""How the state build cuts a head's rows into slices, read off the workspace it asks for (one fp32 state and two fp32 rows per slice)."""
import pytest

from sla_amd import _lib


def slices(BH, L, D):
    total, states = (_lib.load().sla_workspace_bytes(op, _lib.SLA_BF16, 1, BH, L, D, 64, 64, 0)
                     for op in (_lib.WS_LINEAR_FWD, _lib.WS_LINEAR_STATES))
    per_slice = BH * (D * D + 2 * D) * 4                   # (a multiple of 256 for either head dim)
    n, rest = divmod(total - states, per_slice)
    assert n >= 1 and rest == 0
    return n


def tiles(L, D, n):
    """Slices of the fewest whole tiles with which a head has at most n of them."""
    tile = 128 if D == 64 else 64
    rows = -(-(-(-L // n)) // tile) * tile
    return -(-L // rows)


@pytest.mark.parametrize("BH,D", [(16, 64), (12, 64), (8, 64), (12, 128), (20, 128)])
def test_neighbouring_lengths_follow_one_rule(BH, D):
    for L in [*range(4100, 9000, 113), 5003, 6001]:
        n = slices(BH, L, D)
        assert n * BH <= 256 and n == tiles(L, D, min(256 // BH, -(-L // 256))), (BH, L, D, n)


@pytest.mark.parametrize("D", [64, 128])
def test_many_heads_leave_no_compute_units_idle(D):
    """Long enough sequences come to a workgroup for most of the 256 compute units, and to two rounds of them at most."""
    for BH in range(1, 513):
        L = (64 << 20) // (BH * D)             # (the largest below the line of two per unit)
        if L >= 16 * 128:
            assert 208 <= BH * slices(BH, L, D) <= 512, BH
        assert 208 <= BH * slices(BH, 4 * (64 << 20) // (BH * D), D), BH
