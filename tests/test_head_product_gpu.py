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


def _kernel(out, x, w):
    from omniserve_amd import _lib
    (M, K), V, lib = x.shape, w.shape[0], _lib.lib()
    ws = torch.empty((lib.omni_head_argmax_workspace_bytes(M, V, K),), dtype=torch.uint8, device=dev())
    assert lib.omni_head_argmax_f16(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, V, K, ws.data_ptr(), ws.numel(), _lib.current_stream()) == 0
    return out


# every form of the kernel (8, 16, 32 and 64 rows), at sizes that head_argmax leaves to the product, too: vocabularies and rows that end inside a workgroup, K of one stage, of
# less than the ring, of a part of a chain
@pytest.mark.parametrize("M,V,K", [(1, 1, 64), (8, 65, 512), (9, 64, 128), (16, 1000, 4160), (17, 131, 2048), (31, 4096, 448), (33, 63, 192), (64, 5001, 1088), (40, 700, 8192)])
def test_kernel_finds_the_largest_logit(M, V, K):
    g = torch.Generator(device=dev()).manual_seed(M + V + K)
    x = torch.randn((M, K), generator=g, device=dev()).half()
    w = (K ** -0.5 * torch.randn((V, K), generator=g, device=dev())).half()
    out = _kernel(torch.full((M,), -1, dtype=torch.int64, device=dev()), x, w)
    logits = x.double() @ w.double().T
    top = logits.amax(dim=1)
    # (the bound of test_head_argmax_finds_the_largest_logit)
    assert torch.all(top - logits.gather(1, out[:, None])[:, 0] <= 2.0 ** -10 * top.abs() + 1e-5)


@pytest.mark.parametrize("M", [1, 8, 16, 17, 64])
@pytest.mark.parametrize("V,K", [(32000, 4096), (9000, 448), (16000, 8192)])
def test_head_argmax_takes_the_first_of_equal_rows(M, V, K):
    """Words with the same weights have the same logit wherever they stand: sums of cancelling products, whose f32 rounding is far above the fp16 logit's"""
    w = torch.empty((V, K), dtype=torch.float16, device=dev())
    out = torch.empty((M,), dtype=torch.int64, device=dev())
    for seed in range(12):
        g = torch.Generator(device=dev()).manual_seed(seed)
        x = torch.randn((K,), generator=g, device=dev()) + 1.0
        r = torch.randn((K,), generator=g, device=dev())
        r = (r - (r @ x) / (x @ x) * x).half()
        w.fill_(-1.0)
        w[[100, 5000, V - 1]] = r
        assert _kernel(out, x.half().repeat(M, 1), w).tolist() == [100] * M, seed


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


def test_sizes_of_the_one_launch():
    from omniserve_amd import _lib
    faster = _lib.lib().omni_head_argmax_faster
    for M, V, K, want in ((1, 32000, 4096, 1), (64, 32000, 4096, 1), (16, 128256, 4096, 1), (16, 16000, 8192, 1), (65, 32000, 4096, 0), (1, 32000, 4000, 0), (1, 1000, 4096, 0),
                          (16, 8000, 4096, 0), (1, 8000, 1024, 1), (64, 8000, 4096, 0), (16, 32000, 5120, 1), (48, 32000, 5120, 0), (32, 32000, 3072, 1)):
        assert faster(M, V, K) == want, (M, V, K)
