"""The greedy head (csrc/head_product.hip): index of the first largest fp16 logit, against float64 logits."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,V,K", [(1, 32000, 4096), (7, 1000, 64), (8, 65, 512), (9, 64, 128), (16, 32000, 4096), (17, 131, 2048), (32, 4096, 448), (33, 63, 192),
                                   (64, 5001, 1088), (3, 1, 64), (65, 500, 256)])
def test_head_argmax_finds_the_largest_logit(M, V, K):
    from omniserve_amd.backend import fused_ext
    g = torch.Generator(device=dev())
    g.manual_seed(M + V + K)
    x = torch.randn((M, K), generator=g, device=dev()).half()
    w = (K ** -0.5 * torch.randn((V, K), generator=g, device=dev())).half()
    out = torch.full((M,), -1, dtype=torch.int64, device=dev())
    fused_ext.head_argmax(out, x, w)
    logits = x.double() @ w.double().T
    top = logits.amax(dim=1)
    # the chosen logit is the largest up to its fp16 rounding and that of the one that was not chosen (2^-11 each), and f32 sums of K products (2^-20 of the root of K)
    assert torch.all(top - logits.gather(1, out[:, None])[:, 0] <= 2.0 ** -10 * top.abs() + 1e-5)
    clear = (logits >= (top - 2.0 ** -9 * top.abs() - 1e-4)[:, None]).sum(dim=1) == 1
    assert torch.equal(out[clear], logits.argmax(dim=1)[clear])


def test_head_argmax_takes_the_first_of_equal_logits_and_nan_as_the_largest():
    from omniserve_amd.backend import fused_ext
    x = torch.ones((2, 128), device=dev()).half()
    w = torch.zeros((300, 128), device=dev()).half()
    w[[70, 71, 200]] = 1.0
    out = torch.empty((2,), dtype=torch.int64, device=dev())
    fused_ext.head_argmax(out, x, w)
    assert out.tolist() == [70, 70]
    w[250, 5] = float("nan")
    fused_ext.head_argmax(out, x, w)
    assert out.tolist() == [250, 250]
    w[250, 5] = 0.0
    w[:, :] = -1.0
    w[131] = -0.0                                            # (and 0 from below: -0 == +0)
    fused_ext.head_argmax(out, x, w)
    assert out.tolist() == [131, 131]


@pytest.mark.parametrize("M", [1, 8, 16, 17, 64])
@pytest.mark.parametrize("V,K", [(32000, 4096), (9000, 448), (16000, 8192)])
def test_head_argmax_takes_the_first_of_equal_rows(M, V, K):
    """Words with the same weights have the same logit wherever they stand: sums of cancelling products, whose f32 rounding is far above the fp16 logit's"""
    from omniserve_amd.backend import fused_ext
    w = torch.empty((V, K), dtype=torch.float16, device=dev())
    out = torch.empty((M,), dtype=torch.int64, device=dev())
    for seed in range(12):
        g = torch.Generator(device=dev()).manual_seed(seed)
        x = torch.randn((K,), generator=g, device=dev()) + 1.0
        r = torch.randn((K,), generator=g, device=dev())
        r = (r - (r @ x) / (x @ x) * x).half()
        w.fill_(-1.0)
        w[[100, 5000, V - 1]] = r
        fused_ext.head_argmax(out, x.half().repeat(M, 1), w)
        assert out.tolist() == [100] * M, seed


@pytest.mark.parametrize("M", [1, 5])
def test_head_argmax_of_strided_operands(M):
    """A head that is a view -- transposed, or columns of something wider -- goes through torch.matmul."""
    from omniserve_amd.backend import fused_ext
    g = torch.Generator(device=dev()).manual_seed(M)
    out = torch.empty((M,), dtype=torch.int64, device=dev())
    for x, w in ((torch.randn((M, 256), generator=g, device=dev()).half(), torch.randn((256, 700), generator=g, device=dev()).half().t()),
                 (torch.randn((M, 320), generator=g, device=dev()).half()[:, 64:], torch.randn((700, 320), generator=g, device=dev()).half()[:, :256])):
        fused_ext.head_argmax(out, x, w)
        logits = x.double() @ w.double().T
        top = logits.amax(dim=1)
        # fp16 logits, that of the largest and that of the chosen one (2^-11 each)
        assert torch.all(top - logits.gather(1, out[:, None])[:, 0] <= 2.0 ** -10 * top.abs() + 1e-5)
