"""The engine kernels' binding and plans without a GPU: what a call passes by address lives until the call has been made; which form of a
kernel takes which sizes."""
import weakref

import pytest
import torch

from omniserve_amd.backend import lm


class Library:
    """answers the size queries"""

    def lm_gemm_rows_scratch(self, n, k, rows, epi):
        return 2 * rows * n


@pytest.fixture
def ops():
    o = lm.LmOps.__new__(lm.LmOps)
    o.dtype, o._h = torch.bfloat16, Library()
    return o


@pytest.mark.parametrize("call", [lambda o, x, w: o.matmul(x, w), lambda o, x, w: o.matmul(x, w, out_f32=True),
                                  lambda o, x, w: o.glu(x, w, None, "silu")])
def test_scratch_of_k_slices_outlives_its_call(ops, monkeypatch, call):
    made, seen = [], []
    empty = torch.empty

    def noting(size, **kw):
        t = empty(size, **kw)
        if len(size) == 1:
            made.append((weakref.ref(t), t.data_ptr()))
        return t

    monkeypatch.setattr(lm.torch, "empty", noting)

    def enqueue(name, *args):
        (tensor, address), = made
        seen.append((name, tensor() is not None and args[-1] == address))

    ops._call = enqueue
    call(ops, torch.zeros(3, 256, dtype=torch.bfloat16), torch.zeros(64, 256, dtype=torch.bfloat16))
    assert seen == [("lm_gemm_rows", True)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_per_wave_of_prompt_attention(dtype):
    """32 only where workgroups share compute units"""
    rows = lm.lm_ops(dtype)._h.lm_attn_prefill_rows
    for dk in (64, 128, 192, 256):
        for dv in (64, 128, 256):
            for tiles, heads in ((1, 32), (16, 16), (2, 128), (8, 32)):
                assert rows(dk, dv, tiles, heads) == 16
            for tiles, heads in ((9, 32), (126, 16), (43, 6)):
                assert rows(dk, dv, tiles, heads) == (32 if dtype == torch.bfloat16 and dk + dv == 320 else 16)


def test_tiles_of_prompt_products():
    """Whole tiles where they fill the chip's rounds, half tiles where they leave units idle or wait for weights"""
    channels = lm.lm_ops(torch.bfloat16)._h.lm_gemm_tile_channels
    for n, k, rows, want in ((32000, 4096, 65, 128), (32000, 4096, 257, 256), (32000, 4096, 1000, 256), (4096, 2048, 300, 128), (8192, 4096, 1000, 128),
                             (8192, 4096, 2000, 256), (1024, 4096, 2000, 128)):
        assert channels(n, k, 1, 0, rows, 0, 0, 0) == want
    tiles = lambda tokens, experts, top: lm.lm_ops(torch.bfloat16)._h.lm_route_max_tiles(tokens, experts, top)      # noqa: E731
    for tokens, experts, top, n, k, n_b, k_b, want in (
            (65, 32, 6, 4096, 1792, 4096, 3584, 128), (150, 32, 6, 3584, 4096, 7168, 4096, 128), (700, 32, 6, 4096, 1792, 4096, 3584, 128),
            (700, 32, 6, 3584, 4096, 7168, 4096, 256), (1500, 32, 6, 4096, 1792, 4096, 3584, 256), (7999, 32, 6, 4096, 1792, 4096, 3584, 256),
            (7999, 32, 6, 3584, 4096, 7168, 4096, 256), (100, 64, 8, 2048, 640, 2048, 1024, 128), (100, 64, 8, 1280, 2048, 2048, 2048, 128),
            (4000, 64, 8, 1280, 2048, 2048, 2048, 256)):
        assert channels(n, k, experts, tiles(tokens, experts, top), 0, n_b, k_b, tokens) == want, (tokens, n, k)
    assert lm.lm_ops(torch.float32)._h.lm_gemm_tile_channels(4096, 1024, 1, 0, 65, 0, 0, 0) == 128


def test_few_rows_of_short_k_spread_over_the_chip():
    """K of one to three stages: as many workgroups as the channels make, not 64 channels each whatever their number"""
    import ctypes
    for dtype in (torch.bfloat16, torch.float32):
        h, slices = lm.lm_ops(dtype)._h, ctypes.c_int(0)
        for k in (64, 128, 192) if dtype == torch.bfloat16 else (64,):
            assert h.lm_gemm_rows_channels(1, 4096, k, 20, 0, 1, ctypes.byref(slices)) == 16 and slices.value == 1
            assert h.lm_gemm_rows_channels(16, 256, k, 17, 0, 0, None) == 16
            assert h.lm_gemm_rows_channels(1, 4096, k, 15, 0, 1, ctypes.byref(slices)) == 0 and slices.value == 1
            assert h.lm_gemm_rows_channels(32, 512, k, 17, 0, 0, None) == 64
            assert h.lm_gemm_rows_channels(32, 512, k, 16, 0, 0, None) == (0 if k <= 128 else 64)


def test_prompts_do_not_ask_for_the_choice_in_one_launch(ops):
    """Prompts are launched eagerly: what no number of tokens above 32 has is not asked for in every layer"""
    real = lm.lm_ops(torch.bfloat16)
    w = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="meta")      # noqa: E731
    sizes = (w(64, 2048), 64, 8, w(64, 1280, 2048), w(64, 2048, 640))
    assert real.chooses(lm.CHOOSE_TOKENS, *sizes) and not real._h.lm_norm_choose_ok(lm.CHOOSE_TOKENS + 1, 2048, 64, 8)
    assert ops.chooses(lm.CHOOSE_TOKENS + 1, *sizes) is False      # (its library has no such query)
