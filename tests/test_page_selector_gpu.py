"""The page selector's workgroups of 8 and of 16 pages: scores where there is history, zeros in the rest of an output that held something else, against torch."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu

D, TPB = 128, 64


@pytest.mark.parametrize("lengths,padded_pages,heads,group,sub", [([1, 2], 1, 2, 1, 16), ([65, 513, 17], 9, 2, 4, 16), ([1023, 640], 17, 3, 2, 8), ([8193] * 3 + [100] * 62, 129, 8, 2, 16),
                                                                  ([700], 20, 2, 8, 64)])
def test_scores_and_zeros(lengths, padded_pages, heads, group, sub):
    from omniserve_amd import _lib
    B, subs, gen = len(lengths), TPB // sub, torch.Generator(device=dev()).manual_seed(padded_pages)
    streaming = heads - 1                                                   # the last head has no statistics
    ranks, row = heads - 1, D // 2
    head_bytes = ranks * TPB * (row + 4)
    page = torch.zeros((padded_pages, head_bytes // 2 + 2 * subs * ranks * D), dtype=torch.float16, device=dev())
    stats = page[:, head_bytes // 2:].view(padded_pages, 2, subs, ranks, D)
    stats.copy_(torch.randn(stats.shape, generator=gen, device=dev()))
    table = page.data_ptr() + torch.arange(padded_pages, device=dev()) * page.stride(0) * 2
    table = table.expand(B, 2, padded_pages).contiguous()                   # (all sequences read the same pages)
    q = torch.randn((B, heads * group, D), generator=gen, device=dev()).half()
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=dev())       # noqa: E731
    flags, rank, lens = ints([int(h != streaming) for h in range(heads)]), ints(list(range(ranks)) + [0]), ints(lengths)
    rope = torch.tensor([1.0, 0.0], device=dev()).repeat(max(lengths) + 1, D // 2).contiguous()      # no turn
    out = torch.full((B, heads * group, padded_pages * subs), float("nan"), dtype=torch.float16, device=dev())
    rc = _lib.lib().omni_kv_page_selector(out.data_ptr(), q.data_ptr(), q.stride(0), table.data_ptr(), flags.data_ptr(), rank.data_ptr(), lens.data_ptr(), B, padded_pages,
                                          heads * group, heads, ranks, D, row, TPB, sub, out.shape[2], rope.data_ptr(), rope.shape[0], _lib.current_stream())
    assert rc == 0
    torch.cuda.synchronize()
    mx, mn = (stats[:, i].transpose(1, 2).reshape(padded_pages, ranks, subs, D).permute(1, 0, 2, 3).reshape(ranks, -1, D) for i in (0, 1))
    for b, n in enumerate(lengths):
        have = (n - 1 + sub - 1) // sub
        assert not out[b, :, have:].any() and not out[b, streaming * group:].any()
        for h in range(ranks * group):
            prod = torch.maximum(q[b, h] * mx[h // group, :have], q[b, h] * mn[h // group, :have]).double()
            # float32 sums of 128 fp16 values, rounded to fp16
            bound = 2.0 ** -11 * prod.sum(-1).abs() + 2.0 ** -17 * prod.abs().sum(-1) + 1e-7
            assert ((out[b, h, :have].double() - prod.sum(-1)).abs() <= bound).all(), (b, h)
