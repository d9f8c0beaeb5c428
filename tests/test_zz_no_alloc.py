"""The block-mask builder's entry point that allocates nothing (``sla_block_map_fwd_static``: its workspace is a
fixed array in device memory) against ``sla_block_map_fwd`` with a caller-provided workspace: same map and
look-up table, bit for bit, on two calls in a row, the second on a smaller input."""
import pytest
import torch

from sla_amd import _lib, get_block_map
from sla_amd.block_map import topk_count
from sla_amd.inputs import CONFIGS, make_inputs


def _static_map(q, k, ratio, BLKQ, BLKK, lut_dtype=torch.int64):
    """Calls the entry point through the C ABI; the only device memory involved besides the library's own array is
    the inputs and outputs allocated here, before the call."""
    B, H, L, D = q.shape
    M, N = -(-L // BLKQ), -(-L // BLKK)
    T = topk_count(N, ratio)
    sparse_map = torch.full((B, H, M, N), -1, dtype=torch.int8, device=q.device)
    lut = torch.full((B, H, M, T), -1, dtype=lut_dtype, device=q.device)
    def call():
        rc = _lib.load().sla_block_map_fwd_static(q.data_ptr(), k.data_ptr(), _lib.dtype_code(q.dtype), B, H, L, D, BLKQ,
                                                  BLKK, T, sparse_map.data_ptr(), lut.data_ptr(), lut.element_size(),
                                                  _lib.stream_ptr(q.device))
        _lib.check(rc)
        torch.cuda.synchronize()

    call()                       # the first call on a device looks the array's address up and loads the kernels
    # The second one is watched at the driver's level: torch's own counters only see torch's allocator, and a
    # hipMalloc inside the library, made through ctypes, would pass them by.
    torch.cuda.synchronize()
    free_before, _ = torch.cuda.mem_get_info(q.device)
    torch_before = torch.cuda.memory_allocated(q.device)
    sparse_map.fill_(-1)
    lut.fill_(-1)
    call()
    free_after, _ = torch.cuda.mem_get_info(q.device)
    assert free_after == free_before, f"device memory in use changed by {free_before - free_after} bytes during the call"
    assert torch.cuda.memory_allocated(q.device) == torch_before
    return sparse_map, lut, T


@pytest.mark.gpu
def test_static_scratch_entry_point_matches_the_workspace_one(dev):
    g = torch.Generator().manual_seed(11)
    # first call: two heads of the headline shape (ragged last blocks); second call: a smaller input of another
    # dtype and block size, so that stale contents of the shared array would show
    cfg = CONFIGS["cfg3"]
    d = make_inputs(cfg, H=2)
    q1, k1 = d["q"].to(dev), d["k"].to(dev)
    q2 = torch.randn(2, 3, 777, 64, generator=g).to(torch.float16).to(dev)
    k2 = (torch.randn(2, 3, 777, 64, generator=g) + 0.7).to(torch.float16).to(dev)
    q3 = torch.randn(1, 2, 1024, 64, generator=g).to(dev)              # fp32 inputs, as the reference's own dtype order
    k3 = torch.randn(1, 2, 1024, 64, generator=g).to(dev)
    for q, k, ratio, BLKQ, lut_dtype in ((q1, k1, cfg.topk, 64, torch.int64), (q2, k2, 0.3, 128, torch.int32),
                                         (q3, k3, 0.2, 64, torch.int64), (q1, k1, cfg.topk, 64, torch.int64)):
        m_ref, lut_ref, T_ref = get_block_map(q, k, ratio, BLKQ, 64)
        m, lut, T = _static_map(q, k, ratio, BLKQ, 64, lut_dtype)
        assert T == T_ref
        assert torch.equal(m, m_ref), f"map differs in {(m != m_ref).sum().item()} cells"
        assert torch.equal(lut.long(), lut_ref)


@pytest.mark.gpu
def test_static_scratch_entry_point_refuses_what_does_not_fit(dev):
    # the whole headline shape fits (12.7 MB of 16 MiB) ...
    need = _lib.load().sla_workspace_bytes(_lib.WS_BLOCK_MAP, _lib.SLA_BF16, 1, 12, 32760, 128, 64, 64, 25)
    assert 0 < need <= _lib.STATIC_SCRATCH_BYTES
    # ... forty heads of it do not: a clear error before anything is launched, outputs untouched
    q = torch.zeros(1, 40, 32760, 128, dtype=torch.bfloat16, device=dev)
    sparse_map = torch.full((1, 40, 512, 512), -1, dtype=torch.int8, device=dev)
    lut = torch.full((1, 40, 512, 25), -1, dtype=torch.int64, device=dev)
    rc = _lib.load().sla_block_map_fwd_static(q.data_ptr(), q.data_ptr(), _lib.SLA_BF16, 1, 40, 32760, 128, 64, 64, 25,
                                              sparse_map.data_ptr(), lut.data_ptr(), 8, _lib.stream_ptr(dev))
    assert rc == _lib.ERR_WORKSPACE and "static buffer" in _lib.last_error()
    torch.cuda.synchronize()
    assert bool((sparse_map == -1).all()) and bool((lut == -1).all())


def test_size_limit_is_checked_before_any_device_work():
    """No GPU needed: a problem that does not fit the fixed array is refused from its sizes alone."""
    lib = _lib.load()
    FAKE = 0x1000
    assert lib.sla_block_map_fwd_static(FAKE, FAKE, _lib.SLA_BF16, 1, 40, 32760, 128, 64, 64, 25, FAKE, FAKE, 8,
                                        None) == _lib.ERR_WORKSPACE
    assert "static buffer" in _lib.last_error() and str(_lib.STATIC_SCRATCH_BYTES) in _lib.last_error()
    assert lib.sla_block_map_fwd_static(FAKE, FAKE, 7, 1, 1, 64, 64, 64, 64, 1, FAKE, FAKE, 8, None) == _lib.ERR_BAD_ARG
    assert lib.sla_block_map_fwd_static(None, FAKE, _lib.SLA_BF16, 1, 1, 64, 64, 64, 64, 1, FAKE, FAKE, 8,
                                        None) == _lib.ERR_BAD_ARG


def test_many_short_heads_fit_the_fixed_array():
    """No GPU needed: what the block means as rows, the chunk sums and the scores fit into 16 MiB is not refused for its size
    (whole tiles of 32 blocks per head, which the kernels prefer, would not fit).  The pointer that is off 16 bytes keeps the
    call from launching anything."""
    lib = _lib.load()
    FAKE = 0x1000
    up = lambda n: -(-n // 256) * 256  # noqa: E731
    tight = 0
    for dtype, eb in ((_lib.SLA_F32, 4), (_lib.SLA_BF16, 2), (_lib.SLA_F16, 2)):
        for BH in (1, 2, 3, 12, 40, 96, 256, 1024, 4096, 16384):
            for L in (1, 63, 64, 65, 640, 1000, 2048, 8192, 8257, 32760):
                for D in (32, 64, 72, 128):
                    for BLKQ in (64, 128):
                        M, N, C = -(-L // BLKQ), -(-L // 64), -(-L // 64)
                        need = (up(BH * C * D * 4) + up(BH * -(-C // 32) * D * 4) + up(BH * D * eb) + up(BH * M * D * eb)
                                + up(BH * N * D * eb) + up(BH * M * N * eb))
                        if need > _lib.STATIC_SCRATCH_BYTES:
                            continue
                        rc = lib.sla_block_map_fwd_static(FAKE + 2, FAKE, dtype, BH, 1, L, D, BLKQ, 64, 1, FAKE, FAKE, 8, None)
                        assert rc != _lib.ERR_WORKSPACE, (dtype, BH, L, D, BLKQ, need)
                        tight += lib.sla_workspace_bytes(_lib.WS_BLOCK_MAP, dtype, BH, 1, L, D, BLKQ, 64, 1) > _lib.STATIC_SCRATCH_BYTES
    assert tight                    # (sizes at which it makes a difference are among them)


@pytest.mark.gpu
@pytest.mark.parametrize("BH,L,D,BLKQ,dtype,ratio", [
    (1024, 640, 128, 64, torch.bfloat16, 0.3), (1000, 333, 128, 128, torch.float16, 0.5), (3000, 300, 64, 64, torch.float16, 0.4),
    (4096, 64, 64, 128, torch.bfloat16, 1.0)])
def test_static_scratch_entry_point_with_many_short_heads(dev, BH, L, D, BLKQ, dtype, ratio):
    """The block means as rows give the bits that they give in tiles."""
    g = torch.Generator(device=dev).manual_seed(L)
    q = torch.randn(1, BH, L, D, generator=g, device=dev).to(dtype)
    k = (torch.randn(1, BH, L, D, generator=g, device=dev) + 0.5).to(dtype)
    assert _lib.workspace_bytes(_lib.WS_BLOCK_MAP, _lib.dtype_code(dtype), 1, BH, L, D, BLKQ, 64, 1) > _lib.STATIC_SCRATCH_BYTES
    m_ref, lut_ref, T_ref = get_block_map(q, k, ratio, BLKQ, 64)
    m, lut, T = _static_map(q, k, ratio, BLKQ, 64)
    assert T == T_ref and torch.equal(m, m_ref) and torch.equal(lut, lut_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("L,D,BLKQ,dtype", [(8193, 128, 64, torch.bfloat16), (9000, 64, 128, torch.float16), (127 * 64, 128, 128, torch.float16),
                                            (70000, 64, 64, torch.bfloat16), (1, 128, 64, torch.bfloat16), (2111, 64, 64, torch.float16)])
def test_a_workspace_without_room_for_tiles(dev, L, D, BLKQ, dtype):
    """sla_block_map_fwd with the least workspace (block means as rows), with scores in memory and without, against the one
    sla_workspace_bytes names."""
    H = 3
    g = torch.Generator(device=dev).manual_seed(L)
    q = torch.randn(1, H, L, D, generator=g, device=dev).to(dtype)
    k = (torch.randn(1, H, L, D, generator=g, device=dev) + 0.5).to(dtype)
    m_ref, lut_ref, T = get_block_map(q, k, 0.4, BLKQ, 64)
    M, N, C = -(-L // BLKQ), -(-L // 64), -(-L // 64)
    up = lambda n: -(-n // 256) * 256  # noqa: E731
    n = (up(H * C * D * 4) + up(H * -(-C // 32) * D * 4) + up(H * D * 2) + up(H * M * D * 2) + up(H * N * D * 2)
         + (up(H * M * N * 2) if N > 128 else 0))
    lib = _lib.load()
    ws = torch.full((n + 512,), 0xA5, dtype=torch.uint8, device=dev)
    m, lut = torch.full_like(m_ref, -1), torch.full_like(lut_ref, -1)
    call = lambda size: lib.sla_block_map_fwd(q.data_ptr(), k.data_ptr(), _lib.dtype_code(dtype), 1, H, L, D, BLKQ, 64, T,  # noqa: E731
                                              ws.data_ptr(), size, m.data_ptr(), lut.data_ptr(), 8, _lib.stream_ptr(dev))
    assert call(n - 1) == _lib.ERR_WORKSPACE
    _lib.check(call(n))
    assert torch.equal(m, m_ref) and torch.equal(lut, lut_ref) and bool((ws[n:] == 0xA5).all())
