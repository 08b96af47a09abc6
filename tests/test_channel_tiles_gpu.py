"""Per-channel W4A8 products in 256 x 256 tiles (csrc/qgemm_group_tiles.h) against the oracle, bit for bit: the shortest K (the pipeline's ends only), each remainder of its three
buffers, rows that end inside a tile, one tile and several for a workgroup; with the unit against the product and silu_and_mul."""
import pytest
import torch

from oracle import w4a8
from tests.util import assert_f16_equal, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture
def tiles():
    from omniserve_amd import _lib
    _lib.lib().omni_gemm_set_plan_override(16, 0)
    yield
    _lib.lib().omni_gemm_set_plan_override(0, 0)


@pytest.mark.parametrize("M,N,K", [(256, 256, 512), (257, 256, 768), (511, 512, 1024), (512, 256, 1280), (2100, 8192, 512), (300, 256, 1536)])
def test_channel_tiles(tiles, M, N, K):
    _run(M, N, K)


def test_channel_tiles_by_the_rule():
    _run(1020, 16384, 4096)


def _run(M, N, K):
    import omniserve_backend.qgemm_w4a8_per_chn as mod
    from omniserve_amd import _lib
    assert _lib.lib().omni_gemm_prefill_channel_tiles(M, N, K) == 1
    u, z, s1 = w4a8.synth_per_channel(N, K, seed=M + K)
    qw, s1h, szh = w4a8.pack_per_channel(u, z, s1)
    g = torch.Generator().manual_seed(M)
    a = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int32).to(torch.int8).numpy()
    sa, sums = (torch.rand(M, generator=g) * 0.02 + 0.001).half().numpy(), torch.randn(M, generator=g).half().numpy()
    out = torch.full((M + 2, N), 7.0, dtype=torch.half, device=DEV)
    mod.gemm_forward_cuda(to_dev(a), to_dev(qw), to_dev(s1h), to_dev(sa), to_dev(szh), to_dev(sums), out[1:-1])
    assert (out[0] == 7).all() and (out[-1] == 7).all()
    assert_f16_equal(out[1:-1].cpu().numpy(), w4a8.gemm_per_chn(a, qw, s1h, sa, szh, sums), "product in tiles")


@pytest.mark.parametrize("M,N,K", [(256, 256, 512), (300, 512, 768), (1023, 4096, 1024)])
def test_unit_in_the_tiles(tiles, M, N, K):
    """... of the kernel of the other tile heights, whose products and unit are the oracle's"""
    from omniserve_amd import _lib
    from tests.test_silu_rows_gpu import CHN, _case
    h, (x, w, ops) = _lib.lib(), _case(M, N, K, CHN)
    assert h.omni_gemm_prefill_channel_tiles(M, N, K) == 1 and h.omni_gemm_silu_rows_ok(M, N, K, CHN) == 1
    out, gu, want = (torch.full((M + 2, n), 7.0, dtype=torch.half, device=DEV) for n in (N // 2, N, N // 2))
    args = [t.data_ptr() for t in (x, w) + ops]
    assert h.omni_w4a8_per_chn_gemm_silu_rows(*args, out[1].data_ptr(), M, N, K, _lib.current_stream()) == 0
    h.omni_gemm_set_plan_override(0, 0)
    ws = torch.empty((max(h.omni_gemm_workspace_bytes(M, N, K), 1),), dtype=torch.uint8, device=DEV)
    assert h.omni_gemm_prefill_channel_tiles(M, N, K) == 0
    assert h.omni_w4a8_per_chn_gemm(*args, gu[1].data_ptr(), M, N, K, N, ws.data_ptr(), ws.numel(), _lib.current_stream()) == 0
    from omniserve_amd.backend import activation_ops
    activation_ops.silu_and_mul(want[1:-1], gu[1:-1])
    assert torch.equal(out, want) and torch.isfinite(out).all() and out[1:-1].abs().sum() > 0
