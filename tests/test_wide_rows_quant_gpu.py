"""quant_fuse_sum and its silu form of many wide rows (csrc/elementwise.hip): rows whose copy in LDS is fp16, at the edges of the widths and row counts that take it, with
subnormal values, the largest one, a row of zeros and one with an infinity.  Codes, scales and ordered sums are the oracle's bit for bit."""
import numpy as np
import pytest
import torch

from oracle import elementwise as oe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,hidden", [(1024, 8192), (1023, 8224), (1024, 8224), (1026, 16384), (1500, 11008), (1024, 13344), (1023, 13376), (1024, 13376), (1500, 14336)])
def test_many_wide_rows(tokens, hidden):
    from omniserve_amd.backend import activation_ops, fused_ext, fused_kernels
    g = torch.Generator().manual_seed(hidden)
    x = (torch.randn((tokens, hidden), generator=g) * torch.logspace(-7, 2, tokens)[:, None]).half()
    x[3] = 0
    x[5, 7], x[6, 9], x[8, 11] = 65504.0, -65504.0, float("inf")
    dev = lambda t: torch.zeros(t, device="cuda")      # noqa: E731
    new = lambda: (dev((tokens, hidden)).to(torch.int8), dev((tokens,)).half(), dev((tokens,)).half())      # noqa: E731
    q, s, m = new()
    fused_kernels.invoke_quant_fuse_sum(q, x.cuda(), m, s)
    rows = [0, 1, 3, 5, 6, 8, 511, tokens - 1]
    want = oe.quant_per_token(x[rows].numpy(), True)
    for got, w in zip((q, s, m), want):
        assert np.array_equal(got[rows].cpu().numpy(), w, equal_nan=w.dtype != np.int8)
    gu = torch.cat([x.flip(0), x], dim=1).contiguous().cuda()
    gu[tokens - 9] = 1                                                   # (no infinities: both sides' NaN)
    gu[8] = 1
    act = torch.empty((tokens, hidden), dtype=torch.half, device="cuda")
    activation_ops.silu_and_mul(act, gu)
    a, b = new(), new()
    fused_kernels.invoke_quant_fuse_sum(a[0], act, a[2], a[1])
    fused_ext.silu_mul_quant_fuse_sum(b[0], gu, b[2], b[1])
    assert all(torch.equal(u, v) for u, v in zip(a, b))

