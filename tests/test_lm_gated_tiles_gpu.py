"""The gated unit of many rows in tiles that hold gate and up (backend/lm.py, csrc/lm/lm_gemm.hip): rows and channels at the
edges of whole and half tiles, one and two stages of k, a view with a row stride, with and without bias; where the rule leaves it to the vendor's product.
Against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _randn(seed, dtype, *shape):
    return torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).to(dtype)


@pytest.mark.parametrize("m,n,k,act,tiles", [(127, 32, 64, "silu", False), (128, 32, 64, "silu", True), (255, 544, 128, "gelu_tanh", True), (257, 2080, 1536, "silu", True), (1025, 12256, 192, "silu", True),
                                             (900, 7168, 2048, "gelu_tanh", True), (800, 14336, 4096, "silu", False), (2040, 8192, 4096, "silu", True),
                                             (700, 4128, 2112, "silu", False)])
def test_gated_unit_of_many_rows(m, n, k, act, tiles):
    from omniserve_amd.backend.lm import lm_ops
    ops = lm_ops(torch.bfloat16)
    x, w = _randn(1, torch.bfloat16, m, k + 64)[:, 64:], _randn(2, torch.bfloat16, 2 * n, k) * k ** -0.5
    b = _randn(3, torch.float32, 2 * n) if act == "silu" else None
    assert ops._unit_in_tiles(x, w) == tiles
    got = ops.glu(x, w, b, act)
    z = x.double() @ w.double().t()
    z = (z if b is None else z + b.double()).view(m, n // 16, 2, 16)
    f = torch.nn.functional
    gate = f.silu(z[:, :, 0]) if act == "silu" else f.gelu(z[:, :, 0], approximate="tanh")
    want = (gate * z[:, :, 1]).reshape(m, n)
    # one rounding to bf16 moves a value by at most 2^-8 of itself; the vendor's product is rounded before the unit, gate and up (a unit moves by at most 1.1 times its gate)
    bound = 1.05 * 2.0 ** -8 * (1 if tiles else 1 + 1 + 1.1)
    assert ((got.double() - want).norm(dim=1) / want.norm(dim=1)).max() < bound


def test_gated_unit_of_rows_between_boundaries():
    """x that starts between two 16-byte boundaries is left to the vendor's product"""
    from omniserve_amd.backend.lm import lm_ops
    ops = lm_ops(torch.bfloat16)
    x, w = _randn(4, torch.bfloat16, 200 * 256 + 4)[4:].view(200, 256), _randn(5, torch.bfloat16, 64, 256) / 16
    assert not ops._unit_in_tiles(x, w) and ops._unit_in_tiles(x.clone(), w)
    got, want = ops.glu(x, w, None, "silu").double(), ops.glu(x.clone(), w, None, "silu").double()
    assert ((got - want).norm(dim=1) / want.norm(dim=1)).max() < 1.05 * 2.0 ** -8 * 4.1
