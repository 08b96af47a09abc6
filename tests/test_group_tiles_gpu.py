"""Per-group W4A8 products in 256 x 256 tiles (csrc/qgemm_group_tiles.h) against the oracle, bit for bit: the shortest K (the pipeline's ends only), each remainder of its
three buffers, rows that end inside a tile, one tile and several for a workgroup, scales over the whole byte and sums that wrap, parameters that do not begin at a dword."""
import pytest
import torch

from oracle import w4a8
from tests.util import assert_f16_equal, dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def tiles():
    from omniserve_amd import _lib
    _lib.lib().omni_gemm_set_plan_override(16, 0)
    yield
    _lib.lib().omni_gemm_set_plan_override(0, 0)


@pytest.mark.parametrize("M,N,K,wrap,shift", [(256, 256, 512, False, 0), (257, 256, 768, True, 0), (511, 512, 1024, False, 0), (512, 256, 1280, True, 0), (2100, 8192, 512, False, 0),
                                              (300, 256, 1536, True, 1)])
def test_group_tiles(tiles, M, N, K, wrap, shift):
    _run(M, N, K, wrap, shift)


def test_group_tiles_by_the_rule():
    _run(511, 26624, 1536, True, 0)


def _run(M, N, K, wrap, shift):
    import omniserve_backend.qgemm_w4a8_per_group as mod
    from omniserve_amd import _lib
    assert _lib.lib().omni_gemm_prefill_group_tiles(M, N, K) == 1
    u, z, s2, s1 = w4a8.synth_per_group(N, K, seed=M + K, wrap=wrap)
    qw, s1h, s2s, s2z = w4a8.pack_per_group(u, z, s2, s1)
    g = torch.Generator().manual_seed(M)
    a = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int32).to(torch.int8).numpy()
    sa = (torch.rand(M, generator=g) * 0.02 + 0.001).half().numpy()

    def shifted(x):
        x = to_dev(x)
        buf = torch.empty(x.numel() + shift, dtype=x.dtype, device=dev())
        buf[shift:] = x.flatten()
        return buf[shift:].view(x.shape)

    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.gemm_forward_cuda(to_dev(a), to_dev(qw), shifted(s2z), shifted(s2s), to_dev(s1h), to_dev(sa), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, w4a8.gemm_per_group(a, qw, s2z, s2s, s1h, sa), "per_group M=%d N=%d K=%d" % (M, N, K))
