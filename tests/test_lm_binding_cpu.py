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
