"""gate_up_rows' checks of its operands, which hand raw pointers to a kernel: what the product's call refuses is refused, with nothing launched."""
import types

import pytest
import torch

from omniserve_amd import _lib
from omniserve_amd.backend import fused_ext

M, N, K = 300, 512, 256


class Names(list):
    pass


@pytest.fixture
def launches(monkeypatch):
    """A library that takes every call and notes its name"""
    names = Names()

    class Library:
        answers = {"omni_gemm_workspace_bytes": 1}

        def __getattr__(self, name):
            return lambda *a: names.append(name) or self.answers.get(name, 0)

    monkeypatch.setattr(_lib, "_lib", Library())
    monkeypatch.setattr(_lib, "require_cuda", lambda *t: None)
    monkeypatch.setattr(_lib, "current_stream", lambda: 0)
    names.library = _lib._lib
    return names


def _call(mode):
    half, i8 = (lambda *s: torch.zeros(s, dtype=torch.half)), (lambda *s: torch.zeros(s, dtype=torch.int8))
    ops = [(half(N), half(M), half(N), half(M)), (i8(K // 128, N), i8(K // 128, N), half(N), half(M)), (half(N), half(M))][mode]
    return types.SimpleNamespace(out=i8(M, N // 2), in_feats=i8(M, K), weight=i8(N, K if mode == 2 else K // 2), operands=ops, gate_up=half(M, N),
                                 input_sum=half(M) if mode == 0 else None, scale=half(M))


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_operands_of_the_product_are_checked(mode, launches):
    fused_ext.gate_up_rows(**vars(_call(mode)))
    assert any(n.endswith("_silu_rows") for n in launches)
    bad = []
    for field, change in (("weight", lambda t: t[:, :-16]), ("weight", lambda t: t[:, :-16].contiguous()), ("weight", lambda t: t[:-256]), ("weight", lambda t: t.half()),
                          ("weight", lambda t: t.repeat(1, 2)[:, :t.shape[1]]), ("in_feats", lambda t: t.half()), ("in_feats", lambda t: t.repeat(1, 2)[:, :K]),
                          ("in_feats", lambda t: t[:-1]), ("gate_up", lambda t: t.float()), ("gate_up", lambda t: t[:-1]), ("gate_up", lambda t: t[:, :-256])):
        c = _call(mode)
        setattr(c, field, change(getattr(c, field)))
        bad.append((field, c))
    if mode == 1:
        for i in (0, 1):
            c = _call(mode)
            c.operands = tuple(t[:1] if j == i else t for j, t in enumerate(c.operands))
            bad.append(("second level", c))
    for what, c in bad:
        del launches[:]
        with pytest.raises(RuntimeError):
            fused_ext.gate_up_rows(**vars(c))
        assert not launches, what


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_the_library_is_not_asked_before_it_is_called(mode, launches, monkeypatch):
    """Host time counts where prompts are short: a call for the unit and one for the quantiser; one that refuses and the two that stand in for it"""
    kind = ("w4a8_per_chn", "w4a8_per_group", "w8a8")[mode]
    fused_ext.gate_up_rows(**vars(_call(mode)))
    assert launches == ["omni_%s_gemm_silu_rows" % kind, "omni_quant_fuse_sum" if mode == 0 else "omni_quant"]
    monkeypatch.setitem(launches.library.answers, launches[0], -22)
    monkeypatch.setattr(_lib, "workspace", lambda *a: torch.zeros(1, dtype=torch.uint8))
    del launches[:]
    fused_ext.gate_up_rows(**vars(_call(mode)))
    assert [n for n in launches if n != "omni_gemm_workspace_bytes"] == ["omni_%s_gemm_silu_rows" % kind, "omni_%s_gemm" % kind, "omni_silu_mul_quant_fuse_sum"]
