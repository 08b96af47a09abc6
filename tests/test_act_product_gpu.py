"""o_proj / down_proj of one or two rows in slices of their own (csrc/act_product.hip) against the GEMV that has up to 16 rows: the slabs' sums,
the scales and the rows' sums, bit for bit."""
import pytest
import torch

from tests.test_norm_product_gpu import _Layer
from tests.util import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [(1, 4096, 14336), (2, 4096, 14336), (1, 4096, 4096), (2, 4096, 4096), (1, 128, 1024), (2, 192, 3072), (1, 3072, 8192),
                                   (2, 2048, 5120), (1, 1024, 6144), (2, 128, 49152)])
def test_act_product_sums_what_the_gemv_sums(mode, M, N, K):
    from omniserve_amd.backend import fused_ext
    if mode == 2 and M == 2:
        pytest.skip("int8 weights: one row")
    g = torch.Generator(device=dev())
    g.manual_seed(M + N + K + mode)
    lin = _Layer(N, K, mode, g)
    x = (3 * torch.randn((M, K), generator=g, device=dev())).half()
    if M == 2:
        x[1] = 0                                                     # no maximum
    assert fused_ext.act_product_ok(M, N, K, mode)
    amax = fused_ext.new_amax_slots(M, dev())
    amax.view(torch.float32).view(8, 16, 8)[3, :M, 5] = x.float().abs().amax(dim=1)
    slab = torch.full((64 << 20,), 7, dtype=torch.uint8, device=dev())
    a, s = (torch.full((M,), 5.0, dtype=torch.float16, device=dev()) for _ in range(2))
    n = fused_ext.act_product(x, amax, lin, slab, s if mode == 0 else None, a)
    total = slab.view(torch.int32)[:n * M * N].view(n, M, N).sum(dim=0)
    slab2, a2, s2 = torch.zeros_like(slab), torch.empty_like(a), torch.empty_like(s)
    if K <= 16384:
        if mode == 0:
            n2 = fused_ext.gemm_partial_f16_per_chn(x, amax, lin.qweight, slab2, s2, a2)
        elif mode == 1:
            n2 = fused_ext.gemm_partial_f16_per_group(x, amax, lin.qweight, lin.s2_zeros, lin.s2_scales, slab2, s2, a2)
        else:
            n2 = fused_ext.gemm_partial_f16_w8a8(x, amax, lin.weight, slab2, a2)
    else:      # (the GEMV's rows end there)
        import omniserve_backend.fused_kernels as fk
        codes = torch.empty((M, K), dtype=torch.int8, device=dev())
        fk.invoke_quant_fuse_sum(codes, x, s2, a2)
        n2 = (fused_ext.gemm_partial_per_chn(codes, lin.qweight, slab2) if mode == 0 else
              fused_ext.gemm_partial_per_group(codes, lin.qweight, lin.s2_zeros, lin.s2_scales, slab2) if mode == 1 else
              fused_ext.gemm_partial_w8a8(codes, lin.weight, slab2))
    assert torch.equal(total, slab2.view(torch.int32)[:n2 * M * N].view(n2, M, N).sum(dim=0))
    assert torch.equal(a.view(torch.int16), a2.view(torch.int16))
    if mode == 0:
        assert torch.equal(s.view(torch.int16), s2.view(torch.int16))


def test_act_product_refuses_what_it_does_not_cover():
    from omniserve_amd.backend import fused_ext
    ok = fused_ext.act_product_ok
    assert not ok(3, 4096, 4096, 0) and not ok(2, 4096, 4096, 2) and not ok(1, 4096 + 32, 4096, 0) and not ok(1, 4096, 4096 + 512, 0)
    assert not ok(1, 4096, 1024 * 43, 0)                             # a slice of 4 would be 11008: no whole steps; of 1 too long


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_act_product_refuses_buffers_that_do_not_fit(mode):
    from omniserve_amd.backend import fused_ext
    g = torch.Generator(device=dev())
    g.manual_seed(mode)
    N, K = 128, 2048
    f16 = lambda *s: torch.zeros(s, dtype=torch.float16, device=dev())      # noqa: E731
    good = dict(act=f16(1, K), amax=fused_ext.new_amax_slots(1, dev()), lin=_Layer(N, K, mode, g), slab=torch.empty((64 << 10,), dtype=torch.uint8, device=dev()),
                sum_out=f16(1) if mode == 0 else None, scale_out=f16(1))
    fused_ext.act_product(**good)
    for change in (dict(act=f16(1, K).float()), dict(act=f16(1, 2 * K)[:, ::2]), dict(act=f16(1, K // 2)), dict(act=f16(1, 2 * K)), dict(act=f16(K)), dict(amax=good["amax"][:-1]),
                   dict(amax=good["amax"].float()), dict(slab=good["slab"][:64]), dict(slab=good["slab"].view(2, -1)[:, ::2]), dict(scale_out=f16(0)), dict(scale_out=f16(1).float()),
                   dict(sum_out=f16(0)), dict(sum_out=f16(1).float())):
        with pytest.raises(RuntimeError):
            fused_ext.act_product(**{**good, **change})
