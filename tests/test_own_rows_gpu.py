"""Decode steps of one and two sequences, where each norm and the product behind it are one launch (DecodeRunner / LServeDecodeRunner, own_rows): the same tokens, residual and cache pages,
bit for bit, as without and as the reference's sequence of calls, eagerly and as a graph.  Layers hand the residual from buffer to buffer and slabs to the next layer's norm: one layer
and several; down_proj in slices of act_product and, where it has not the size, of the 16-row GEMV."""
import pytest
import torch

from omniserve_amd.lserve_runtime import LServeDecodeRunner
from omniserve_amd.runtime import DecodeRunner, LlamaConfig
from tests.util import dev

pytestmark = pytest.mark.gpu


def _config(layers, inter, group=-1):
    return LlamaConfig(hidden=2048, inter=inter, heads=16, kv_heads=4, layers=layers, vocab=1000, group_size=group)


def _state(r, steps):
    tokens = []
    for _ in range(steps):
        r.step()
        tokens.append(r.tokens.clone())
    torch.cuda.synchronize()
    assert torch.isfinite(r.x.float()).all()
    return [torch.stack(tokens), r.x.view(torch.int16).clone(), r.normed.view(torch.int16).clone(), *[p.clone() for layer in r.pools for p in layer]]


def _compare(make, steps):
    want = None
    for own, graph, fused in ((False, False, 0), (False, True, True), (True, False, True), (True, True, True)):
        r = make(use_graph=graph, fused=fused, own_rows=own)
        assert r.own_rows == own
        got = _state(r, steps)
        want = want or got
        assert all(torch.equal(a, b) for a, b in zip(got, want)), (own, graph, fused)
        del r


@pytest.mark.parametrize("layers,inter", [(1, 4096), (2, 2816), (3, 4096)])
@pytest.mark.parametrize("group", [-1, 128])
@pytest.mark.parametrize("batch", [1, 2])
def test_decode(batch, group, layers, inter):
    _compare(lambda **k: DecodeRunner(_config(layers, inter, group), batch=batch, context=70, max_new=8, device=dev(), seed=7, **k), 4)


@pytest.mark.parametrize("kv_format", ["kv8", "kv4"])
@pytest.mark.parametrize("layers,inter", [(1, 4096), (2, 2816), (3, 4096)])
def test_lserve_decode(layers, inter, kv_format):
    """(crosses a page boundary and three selections of pages)"""
    _compare(lambda **k: LServeDecodeRunner(_config(layers, inter), batch=1, context=700, max_new=16, device=dev(), seed=11, kv_format=kv_format, sink=64, local=128, budget_tokens=256,
                                            selector_interval=4, **k), 9)


def test_prefill_and_steps_behind_it():
    """the step takes up what prefill left in the runner's buffers"""
    out = []
    for own in (False, True):
        r = DecodeRunner(_config(2, 4096), batch=2, context=70, max_new=8, device=dev(), seed=3, own_rows=own)
        r.prefill(70, tokens=torch.arange(140, device=dev()))
        out.append(_state(r, 3))
    assert all(torch.equal(a, b) for a, b in zip(*out))


def test_a_model_without_layers():
    out = []
    for own in (False, True):
        r = DecodeRunner(_config(0, 4096), batch=1, context=70, max_new=8, device=dev(), seed=3, use_graph=False, own_rows=own)
        assert not r.own_rows
        out.append(_state(r, 2))
    assert all(torch.equal(a, b) for a, b in zip(*out))
