"""gate_up of many rows with silu_and_mul in the product's tiles (csrc/qgemm_exact.h, qgemm_group_tiles.h, qgemm_tiles.h): every tile height and both 256 x 256
kernels, row counts at the edges of their tiles, one and several bands, the smallest widths.  The codes, scales and sums are bit for bit those of product,
silu_and_mul and quantiser; so they are where the tiles do not have the unit."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _plan(M, N, K, mode):
    from omniserve_amd import _lib
    h, mb, kw, sk = _lib.lib(), ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    h.omni_gemm_get_prefill_plan(M, N, K, mode, 0, ctypes.byref(mb), ctypes.byref(kw), ctypes.byref(sk))
    ok = h.omni_gemm_silu_rows_ok(M, N, K, mode)
    return (ok, "tiles" if mode == 1 and h.omni_gemm_prefill_group_tiles(M, N, K) else mb.value)


def _case(M, N, K, mode):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    half = lambda *s: torch.rand(s, device=DEV, generator=g).half()      # noqa: E731
    x = torch.randint(-127, 128, (M, K), device=DEV, generator=g, dtype=torch.int8)
    if mode == 2:
        return x, torch.randint(-127, 128, (N, K), device=DEV, generator=g, dtype=torch.int8), (half(N) * 2e-3 / K ** 0.5, half(M))
    w = torch.randint(-128, 128, (N, K // 2), device=DEV, generator=g, dtype=torch.int8)
    if mode == 0:
        return x, w, (half(N) * 0.02 / K ** 0.5, half(M), half(N) * 1e-2, half(M))
    s2 = torch.randint(1, 9, (K // 128, N), device=DEV, generator=g, dtype=torch.int8)
    z2 = (-(torch.randint(0, 16, (K // 128, N), device=DEV, generator=g) * s2)).to(torch.int8)
    return x, w, (z2, s2, half(N) * 0.004 / K ** 0.5, half(M))


CHN, GRP, W8 = 0, 1, 2
SIZES = [(CHN, 1501, 28672, 4096, 8), (CHN, 1100, 24576, 512, True), (CHN, 700, 16384, 256, 6), (CHN, 449, 16384, 256, 8), (CHN, 2049, 512, 256, True), (CHN, 324, 12288, 256, 5),
         (CHN, 404, 12288, 256, 7), (CHN, 129, 1024, 256, True), (CHN, 4099, 1024, 768, True),
         (CHN, 1024, 57344, 512, True), (CHN, 1500, 57344, 8192, 8), (GRP, 1500, 57344, 8192, "tiles"), (W8, 1500, 57344, 8192, 16),
         (GRP, 2331, 28672, 4096, "tiles"), (GRP, 2049, 14336, 2048, "tiles"), (GRP, 512, 28672, 4096, "tiles"), (GRP, 700, 16384, 256, 6), (GRP, 449, 16384, 256, 8), (GRP, 324, 12288, 256, 5), (GRP, 404, 12288, 256, 7),
         (GRP, 1025, 1024, 512, True),
         (W8, 12001, 28672, 4096, 16), (W8, 2700, 28672, 1024, 16), (W8, 2305, 32768, 1024, 16), (W8, 2048, 32768, 1536, 16), (W8, 2049, 32768, 1536, 16), (W8, 1000, 12288, 2048, 16), (W8, 3000, 8192, 768, False), (W8, 300, 512, 768, False), (CHN, 128, 1024, 256, False), (GRP, 600, 768, 640, False)]


@pytest.mark.parametrize("mode,M,N,K,tiles", SIZES)
def test_unit_in_the_product(mode, M, N, K, tiles):
    from omniserve_amd import _lib
    from omniserve_amd.backend import fused_ext, qgemm_w4a8_per_chn, qgemm_w4a8_per_group, qgemm_w8a8
    ok, form = _plan(M, N, K, mode)
    assert bool(ok) == bool(tiles) and (isinstance(tiles, bool) or form == tiles)      # (True: whichever tiles; False: product and unit's quantiser)
    x, w, ops = _case(M, N, K, mode)
    product = (qgemm_w4a8_per_chn.gemm_forward_cuda, qgemm_w4a8_per_group.gemm_forward_cuda, qgemm_w8a8.w8a8_gemm_forward_cuda)[mode]
    gu = torch.empty((M, N), dtype=torch.half, device=DEV)
    outs = []
    for fused in (False, True):
        q = torch.full((M + 2, N // 2), 77, dtype=torch.int8, device=DEV)
        s, m = torch.zeros((M,), dtype=torch.half, device=DEV), torch.zeros((M,), dtype=torch.half, device=DEV) if mode == CHN else None
        room = torch.full((M * N + 64,), 7.0, dtype=torch.half, device=DEV)
        if fused:
            fused_ext.gate_up_rows(q[1:-1], x, w, ops, room[:M * N].view(M, N), m, s)
            assert (room[M * N:] == 7).all() and bool((room[M * N // 2:] == 7).all()) == bool(ok)
        else:
            product(x, w, *ops, gu)
            fused_ext.silu_mul_quant_fuse_sum(q[1:-1], gu, m, s)
        assert (q[0] == 77).all() and (q[-1] == 77).all()
        outs.append((q, s) if m is None else (q, s, m))
    assert outs[0][0].float().abs().sum() > 0 and torch.isfinite(outs[0][1]).all()
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    if ok and mode == W8 and M < 4000:      # rows that start between two 16-byte boundaries are refused
        y = torch.empty((M * N // 2 + 8,), dtype=torch.half, device=DEV)
        h = _lib.lib()
        assert h.omni_w8a8_gemm_silu_rows(x.data_ptr(), w.data_ptr(), ops[0].data_ptr(), ops[1].data_ptr(), y.data_ptr() + 8, M, N, K, True) != 0
        assert h.omni_w8a8_gemm_silu_rows(x.data_ptr(), w.data_ptr(), ops[0].data_ptr(), ops[1].data_ptr(), y.data_ptr(), 128, N, K, True) != 0


@pytest.mark.parametrize("M,N,K", [(700, 32768, 8192), (1300, 28672, 9216), (2305, 16384, 16384)])
def test_int8_tiles_of_operands_beyond_the_last_cache(M, N, K):
    """Operands of more than 256 MB, last row tiles that share rows, bands of three: against the kernel of the other tile heights"""
    from omniserve_amd import _lib
    from omniserve_amd.backend import qgemm_w8a8
    assert (M + N) * K > 256 << 20 and _plan(M, N, K, W8)[1] == 16
    x, w, ops = _case(M, N, K, W8)
    out = [torch.empty((M, N), dtype=torch.half, device=DEV) for _ in range(2)]
    qgemm_w8a8.w8a8_gemm_forward_cuda(x, w, *ops, out[0])
    _lib.lib().omni_gemm_set_plan_override(0, 1)
    try:
        assert _plan(M, N, K, W8)[1] < 16
        qgemm_w8a8.w8a8_gemm_forward_cuda(x, w, *ops, out[1])
    finally:
        _lib.lib().omni_gemm_set_plan_override(0, 0)
    assert torch.equal(*out) and out[0].isfinite().all() and out[0].any()
