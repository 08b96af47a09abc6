"""Products of few rows at every number of row blocks, and of more rows than a launch streams at a time, against f32 sums of the same bf16 inputs: their
chains of f32 additions are off by less than 1e-5 of the row, the bf16 result by half an ulp (2^-9)."""
import ctypes

import pytest
import torch

from omniserve_amd.backend import lm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 48, 49, 64, 65, 129, 200])
@pytest.mark.parametrize("n,k", [(8192, 2048), (8256, 576)])
@pytest.mark.parametrize("epi", [lm.EPI_ELEM, lm.EPI_F32, lm.EPI_GLU, lm.EPI_GATE])
def test_rows(rows, n, k, epi):
    ops = lm.lm_ops(torch.bfloat16)
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + n + epi)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")      # noqa: E731
    w, x, z = (k ** -0.5 * rnd(n, k)).bfloat16(), rnd(rows, k + 64)[:, :k].bfloat16(), rnd(rows, n).bfloat16()
    x = torch.nn.functional.pad(x, (0, 64))[:, :k]      # rows with a stride of their own
    bias = 0.1 * rnd(n)
    cols = n // 2 if epi == lm.EPI_GLU else n
    out = torch.full((rows, cols + 8), float("nan"), dtype=torch.float32 if epi == lm.EPI_F32 else torch.bfloat16, device="cuda")[:, :cols]
    part = lm._Part(w.data_ptr(), x.data_ptr(), x.stride(0), out.data_ptr(), out.stride(0), n, k, bias=bias.data_ptr() if epi == lm.EPI_GLU else None,
                    gate=z.data_ptr() if epi == lm.EPI_GATE else None, ldg=z.stride(0))
    # (a hint of 64 rows where there are more: the streaming kernels for them, too)
    ops._call("lm_gemm_rows", ctypes.byref(part), None, 1, None, None, rows, 0, 1, rows if epi == lm.EPI_GLU else min(rows, 64), 1.0, epi,
              lm.ACT["silu"] if epi == lm.EPI_GLU else 0, None)
    torch.cuda.synchronize()
    y = x.double() @ w.double().T
    if epi == lm.EPI_GLU:
        y = (y + bias).view(rows, -1, 2, 16)
        y = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(rows, cols)
    if epi == lm.EPI_GATE:
        y = y * torch.sigmoid(z.double())
    bar = 1e-5 if epi == lm.EPI_F32 else 2.0 ** -9 + 1e-5
    err = (out.double() - y).norm(dim=1) / y.norm(dim=1)
    assert err.max() <= bar, float(err.max())
