"""A product's K slices added up by the norm behind it: the same bits as the product's own rows and the norm over those."""
import pytest
import torch

from omniserve_amd.backend.lm import lm_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 17, 48, 64])
@pytest.mark.parametrize("n,k,real", [(4096, 14336, 4096), (1024, 8192, 1000), (2048, 6144, 2044), (8192, 16384, 8192), (512, 512, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_same_bits(T, n, k, real, dtype):
    ops = lm_ops(dtype)
    g = torch.Generator(device="cuda")
    g.manual_seed(T + n + k)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")      # noqa: E731
    w, a, x0 = (k ** -0.5 * rnd(n, k)).to(dtype), rnd(T, k).to(dtype), rnd(T, n)
    pad = lambda v: torch.nn.functional.pad(v[:real], (0, n - real))      # noqa: E731
    w[real:] = 0
    bias, post, nxt = pad(0.1 * rnd(n)), (pad(1 + 0.1 * rnd(n)), pad(0.1 * rnd(n))), (pad(1 + 0.1 * rnd(n)), None)
    rows = torch.arange(T - 1, -1, -2, dtype=torch.int32, device="cuda")
    y = ops.matmul(a, w)
    s = ops.sums(a, w)
    assert (s.dim() == 3) == (ops._h.lm_gemm_rows_scratch(n, k, T, 0) > 0)
    for kw in (dict(kind="rms", y_bias=bias, post=post), dict(kind="layer", next=nxt), dict(kind="rms", y_bias=bias, post=post, next=nxt, rows=rows, store_x=False)):
        kw = dict(kw)
        kind = kw.pop("kind")
        out = []
        for v in (y, s):
            x, h = x0.clone(), torch.zeros((T if "rows" not in kw else rows.numel(), n), dtype=dtype, device="cuda")
            ops.residual_norm(x, real, kind, 1e-5, y=v, h=h, **kw)
            out.append((x, h))
        torch.cuda.synchronize()
        assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1]), kw.keys()


@pytest.mark.parametrize("T", [1, 17, 64])
@pytest.mark.parametrize("n,k", [(4096, 4096), (2048, 2048), (8192, 8192)])
def test_slices_that_the_product_alone_does_not_have(T, n, k):
    """bf16 rows of f32 sums: within a rounding of either (2^-8 of it), and the norm's addition is the slices' one after the other"""
    ops = lm_ops(torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(T + n)
    w, a = (k ** -0.5 * torch.randn(n, k, generator=g, device="cuda")).bfloat16(), torch.randn(T, k, generator=g, device="cuda").bfloat16()
    s = ops.sums(a, w)
    assert s.dim() == 3 and (n == 8192 or ops._h.lm_gemm_rows_scratch(n, k, T, 0) == 0)
    rows = s[0].clone()
    for part in s[1:]:
        rows += part
    want = a.double() @ w.double().t()
    assert (rows - want).norm() < 1e-6 * k ** 0.5 * want.norm()
    out = []
    for v in (rows.bfloat16(), s):
        x, h = torch.ones((T, n), device="cuda"), torch.zeros((T, n), dtype=torch.bfloat16, device="cuda")
        ops.residual_norm(x, n, "rms", 1e-5, y=v, next=(torch.ones(n, device="cuda"), None), h=h)
        out.append((x, h))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
