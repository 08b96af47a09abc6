"""How many parts of the keys the decode attention takes: the number with the least rounds of workgroups x (tokens of a part + 192), in the dense form and in the one over lists
of pages.  The order of the merge's sums hangs on it, and with it the bits of a step."""
import ctypes

import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu

D, TPB, PAGE_BYTES = 128, 64, 1 << 16                 # a page's bytes: more than 8 heads' codes, scales and statistics


def _planned(workgroups, tokens, most=1024, cap=2048):
    """cap: a part's most tokens"""
    most = min((tokens + 63) // 64, most)
    part = lambda n: ((tokens + n - 1) // n + 15) & ~15      # noqa: E731
    least = next(n for n in range(1, most + 1) if part(n) <= cap)
    end = min(max(2048 // workgroups + 1, 2 * least + 8), most)
    return min(range(least, end + 1), key=lambda n: ((workgroups * n + 511) // 512 * (part(n) + 192), n))


def _inputs(batch, heads, kv_heads, tokens):
    from omniserve_amd import _lib
    pages = (tokens + TPB - 1) // TPB
    gen = torch.Generator(device=dev()).manual_seed(tokens)
    pool = torch.zeros((2 * batch * pages, PAGE_BYTES), dtype=torch.uint8, device=dev())
    table = (pool.data_ptr() + torch.arange(2 * batch * pages, device=dev()) * PAGE_BYTES).view(batch, 2, pages)
    qkv = torch.randn((batch, (heads + 2 * kv_heads) * D), generator=gen, device=dev()).half()
    rope = torch.tensor([1.0, 0.0], device=dev()).repeat(tokens + 1, D // 2).contiguous()
    ws = torch.empty((_lib.lib().omni_kv4_decode_workspace_bytes(batch, heads, D, tokens),), dtype=torch.uint8, device=dev())
    lengths = torch.full((batch,), tokens, dtype=torch.int32, device=dev())
    at = [qkv.data_ptr() + 2 * D * c for c in (0, heads, heads + kv_heads)] + [qkv.stride(0)] * 2
    return at, pool, table, rope, ws, lengths, qkv


@pytest.mark.parametrize("batch,heads,kv_heads,tokens", [(1, 32, 8, 300), (1, 32, 8, 1500), (1, 32, 8, 3000), (1, 32, 8, 6000), (2, 32, 8, 3000), (3, 32, 8, 1000), (4, 32, 8, 1000),
                                                          (5, 32, 8, 2000), (16, 32, 8, 1024), (61, 32, 8, 1100), (1, 64, 8, 3000), (2, 8, 8, 700)])
def test_dense(batch, heads, kv_heads, tokens):
    from omniserve_amd import _lib
    at, pool, table, rope, ws, lengths, _ = _inputs(batch, heads, kv_heads, tokens)
    n = ctypes.c_int(0)
    rc = _lib.lib().omni_kv4_decode_attention_partial(*at, table.data_ptr(), lengths.data_ptr(), batch, table.shape[2], heads, kv_heads, D, TPB, tokens, rope.data_ptr(),
                                                      rope.shape[0], ws.data_ptr(), ws.numel(), ctypes.byref(n), _lib.current_stream())
    torch.cuda.synchronize()
    group = heads // kv_heads
    assert rc == 0 and n.value == _planned(batch * kv_heads * (group // (8 if group % 8 == 0 else min(group, 4))), tokens)


@pytest.mark.parametrize("tokens,listed", [(4096, 0), (2500, 0), (8000, 64), (8000, 16)])
def test_pages_of_heads(tokens, listed):
    """listed: pages of every head's list (0: all pages, a workgroup for four heads)"""
    from omniserve_amd import _lib
    batch, heads, kv_heads = 1, 32, 8
    at, pool, table, rope, ws, lengths, _ = _inputs(batch, heads, kv_heads, tokens)
    flags, rank = torch.ones((kv_heads,), dtype=torch.int32, device=dev()), torch.arange(kv_heads, dtype=torch.int32, device=dev())
    last = (tokens + TPB - 1) // TPB - 1
    pages = torch.arange(last + 1 - max(listed, 1), last + 1, dtype=torch.int32, device=dev()).repeat(batch, heads, 1).contiguous()
    n = ctypes.c_int(0)
    rc = _lib.lib().omni_kv_decode_attention_fine_grained_partial(
        *at, None, None, table.data_ptr(), None, flags.data_ptr(), rank.data_ptr(), lengths.data_ptr(), pages.data_ptr() if listed else None, listed, 16, batch, table.shape[2], 0,
        heads, kv_heads, kv_heads, 0, D, TPB, 0, 0, 0, 0, tokens, rope.data_ptr(), rope.shape[0], ws.data_ptr(), ws.numel(), ctypes.byref(n), _lib.current_stream())
    torch.cuda.synchronize()
    assert rc == 0 and n.value == _planned(batch * heads // (1 if listed else 4), listed * TPB or tokens)
