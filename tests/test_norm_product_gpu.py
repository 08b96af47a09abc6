"""Norm and product of one or two rows as one launch (csrc/norm_product.hip) against the calls that it replaces, bit for bit: new residual,
projection or SiLU activation, row maxima; the residual that it reads stays as it was."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu


class _Layer:
    """A projection with random weights: mode 0 W4A8 per-channel, 1 per-group, 2 W8A8"""

    def __init__(self, n, k, mode, g):
        r = lambda lo, hi, *s: torch.randint(lo, hi, s, generator=g, device=dev())      # noqa: E731
        scale = ((0.5 + torch.rand(n, generator=g, device=dev())) * 2e-4).half()
        self.mode, self.group = mode, 128 if mode == 1 else -1
        if mode == 2:
            self.weight, self.dequant_scale = r(-128, 128, n, k).to(torch.int8), scale
            return
        self.qweight, self.s1_scales = r(0, 256, n, k // 2).to(torch.uint8).view(torch.int8), scale
        if mode == 0:
            self.s1_szeros = (r(0, 16, n).half() * scale).half()
        else:
            self.s2_scales, self.s2_zeros = r(1, 9, k // 128, n).to(torch.int8), r(-120, 1, k // 128, n).to(torch.int8)

    def scales(self):
        return self.dequant_scale if self.mode == 2 else self.s1_scales


def _two_calls(x, gamma, lin, out, silu, amax, prod, slab, sk, p_a, p_sum):
    import omniserve_backend.layernorm_ops as ln
    import omniserve_backend.qgemm_w4a8_per_chn as chn
    import omniserve_backend.qgemm_w4a8_per_group as grp
    import omniserve_backend.qgemm_w8a8 as w8
    from omniserve_amd.backend import fused_ext
    M, H = x.shape
    codes = torch.empty((M, H), dtype=torch.int8, device=dev())
    s, a = (torch.empty(M, dtype=torch.float16, device=dev()) for _ in range(2))
    if slab is None:
        ln.rms_norm_general_fuse_sum(codes, x, gamma, s, a, 1e-5, True) if lin.mode == 0 else ln.rms_norm_general(codes, x, gamma, a, 1e-5, True)
    elif lin.mode == 0:
        fused_ext.splitk_add_rms_norm_general_fuse_sum(codes, x, slab, sk, prod.scales(), p_a, prod.s1_szeros, p_sum, gamma, s, a, 1e-5)
    else:
        fused_ext.splitk_w8_add_rms_norm_general_fuse_sum(codes, x, slab, sk, prod.scales(), p_a, gamma, None, a, 1e-5)
    if lin.mode == 0:
        if silu:
            fused_ext.gemm_silu_per_chn(codes, lin.qweight, lin.s1_scales, a, lin.s1_szeros, s, out, amax)
        else:
            chn.gemm_forward_cuda(codes, lin.qweight, lin.s1_scales, a, lin.s1_szeros, s, out)
    elif lin.mode == 1:
        if silu:
            fused_ext.gemm_silu_per_group(codes, lin.qweight, lin.s2_zeros, lin.s2_scales, lin.s1_scales, a, out, amax)
        else:
            grp.gemm_forward_cuda(codes, lin.qweight, lin.s2_zeros, lin.s2_scales, lin.s1_scales, a, out)
    elif silu:
        fused_ext.gemm_silu_w8a8(codes, lin.weight, lin.dequant_scale, a, out, amax)
    else:
        w8.w8a8_gemm_forward_cuda(codes, lin.weight, lin.dequant_scale, a, out)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("M,N,H,sk,silu", [(1, 64, 4096, 0, False), (2, 6144, 4096, 0, False), (1, 6144, 4096, 7, False), (2, 192, 4096, 8, False),
                                           (1, 192, 4096, 14, False), (1, 64, 2048, 16, False), (2, 2560, 3072, 1, False), (1, 320, 2048, 5, False),
                                           (1, 12288, 4096, 1, False), (2, 192, 4096, 2, False), (1, 320, 3072, 3, False), (2, 6144, 2048, 4, False),
                                           (1, 28672, 4096, 2, True), (2, 28672, 4096, 4, True), (2, 128, 2048, 1, True), (1, 8448, 3072, 3, True),
                                           (1, 16512, 2048, 2, True), (2, 22016, 4096, 3, True)])
def test_norm_product_gives_the_bits_of_the_calls_it_replaces(mode, M, N, H, sk, silu):
    from omniserve_amd.backend import fused_ext
    if mode == 2 and M == 2:
        pytest.skip("int8 weights: one row")
    g = torch.Generator(device=dev())
    g.manual_seed(1000 * M + N + H + sk + mode)
    lin, prod = _Layer(N, H, mode, g), _Layer(H, 256, mode, g)
    x = torch.randn((M, H), generator=g, device=dev()).half()
    gamma = (1 + 0.1 * torch.randn(H, generator=g, device=dev())).half()
    slab = torch.randint(-8000, 8000, (max(sk, 1), M, H), generator=g, device=dev(), dtype=torch.int32) if sk else None
    p_a = (0.2 + torch.rand(M, generator=g, device=dev())).half()
    p_sum = torch.randn(M, generator=g, device=dev()).half()
    want_x, want = x.clone(), torch.empty((M, N // 2 if silu else N), dtype=torch.float16, device=dev())
    amax = [fused_ext.new_amax_slots(M, dev()) for _ in range(2)] if silu else [None, None]
    _two_calls(want_x, gamma, lin, want, silu, amax[0], prod, slab, sk, p_a, p_sum)
    got, before, new_x = torch.full_like(want, 3.0), x.clone(), torch.full_like(x, 5.0)
    fused_ext.norm_product(x, gamma, 1e-5, lin, got, new_x if sk else None, slab, sk, prod, p_a, p_sum, amax[1])
    assert torch.equal(x, before)
    if sk:
        assert torch.equal(new_x.view(torch.int16), want_x.view(torch.int16))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    if silu:
        rows = [t.view(torch.float32).view(8, 16, 8).amax(dim=(0, 2)) for t in amax]
        assert torch.equal(rows[0], rows[1])


def test_norm_product_refuses_what_it_does_not_cover():
    from omniserve_amd.backend import fused_ext
    ok = fused_ext.norm_product_ok
    assert ok(1, 6144, 4096, 0, False, 14336) and ok(2, 28672, 4096, 1, True, 4096) and ok(1, 6144, 4096, 2, False, 14336)
    assert not ok(3, 6144, 4096, 0)                       # three rows
    assert not ok(1, 6144, 8192, 0) and not ok(1, 6144, 4096 + 512, 0) and not ok(1, 6144, 1024, 0)
    assert not ok(1, 6144 + 32, 4096, 0) and not ok(1, 28672 + 64, 4096, 0, True, 4096)
    assert not ok(2, 6144, 4096, 2, False, 4096)          # two rows with int8 weights
    assert not ok(1, 28672, 4096, 0, True)                # gate_up always consumes slabs


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_norm_product_refuses_buffers_that_do_not_fit(mode):
    """wrong types, strides and sizes, which the kernel would read or write past"""
    from omniserve_amd.backend import fused_ext
    g = torch.Generator(device=dev())
    g.manual_seed(mode)
    H, N, sk = 2048, 256, 3
    f16 = lambda *s: torch.zeros(s, dtype=torch.float16, device=dev())      # noqa: E731
    x = f16(1, 2 * H)
    good = dict(residual=x[:, :H], gamma=f16(H), epsilon=1e-5, lin=_Layer(N, H, mode, g), out=f16(1, N), residual_out=f16(1, H), slab=torch.zeros((sk, 1, H), dtype=torch.int32, device=dev()),
                sk=sk, producer=_Layer(H, 256, mode, g), p_ascales=f16(1), p_asums=f16(1))
    fused_ext.norm_product(**good)
    silu = dict(out=f16(1, N // 2), amax=fused_ext.new_amax_slots(1, dev()))
    fused_ext.norm_product(**{**good, **silu})
    bad = [dict(residual=x[:, :H].float()), dict(residual=f16(1, H // 2)), dict(residual=f16(1, 2 * H)[:, ::2]), dict(gamma=f16(H - 1)), dict(gamma=f16(2 * H)[::2]), dict(out=f16(1, N - 1)),
           dict(out=f16(1, N // 2)), dict(out=f16(1, 2 * N)[:, ::2]), dict(out=f16(1, N).float()), dict(sk=sk + 1), dict(slab=good["slab"][:2]), dict(producer=_Layer(H // 2, 256, mode, g)),
           dict(producer=_Layer(H, 256, 0 if mode == 2 else 2, g)), dict(residual_out=None), dict(residual_out=x[:, :H]), dict(residual_out=x[:, 64:H + 64]), dict(residual_out=f16(1, H - 64)),
           dict(p_ascales=None), dict(p_ascales=f16(1).float()), {**silu, "out": f16(1, N)}, {**silu, "amax": silu["amax"][:-1]}, {**silu, "amax": silu["amax"].float()}]
    if mode == 0:
        bad += [dict(p_asums=None), dict(p_asums=f16(0))]
    for change in bad:
        with pytest.raises(RuntimeError):
            fused_ext.norm_product(**{**good, **change})
