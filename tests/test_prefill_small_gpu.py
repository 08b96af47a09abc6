"""Prefill attention in workgroups of 64 query rows against those of 128: a row meets the same key tiles in the same order, so the outputs are the same
bits, whatever the lengths, masks and strides."""
import numpy as np
import pytest
import torch

from oracle import attention as oa
from tests.util import assert_attention_close, to_dev

pytestmark = pytest.mark.gpu


def _both(call):
    from omniserve_amd import _lib
    out = []
    try:
        for variant in (3, 4):
            _lib.lib().omni_prefill_set_variant(variant)
            out.append(call().clone())
    finally:
        _lib.lib().omni_prefill_set_variant(0)
    torch.cuda.synchronize()
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))
    return out[0]


def _qkv(rows, heads, seed):
    return np.random.default_rng(seed).standard_normal((rows, heads, 128)).astype(np.float16)


@pytest.mark.parametrize("lens_q,lens_k,Hq,Hk,causal", [
    ([1], None, 4, 1, True), ([63, 64, 65, 127, 128, 129], None, 8, 2, True), ([333] * 3, None, 32, 8, True), ([700, 1], None, 6, 3, True),
    ([5, 70], [200, 70], 8, 2, True), ([130, 64], [194, 300], 4, 4, True), ([65, 200], [191, 64], 8, 8, False)])
def test_dense(lens_q, lens_k, Hq, Hk, causal):
    import block_sparse_attn as bsa
    lens_k = lens_q if lens_k is None else lens_k
    q, k, v = _qkv(sum(lens_q), Hq, 1), _qkv(sum(lens_k), Hk, 2), _qkv(sum(lens_k), Hk, 3)
    cu_q, cu_k = (np.concatenate([[0], np.cumsum(n)]).astype(np.int32) for n in (lens_q, lens_k))
    args = [to_dev(a) for a in (q, k, v, cu_q, cu_k)]
    got = _both(lambda: bsa.flash_attn_varlen_func(*args, max(lens_q), max(lens_k), dropout_p=0.0, causal=causal))
    ref = oa.varlen_attention(q, k, v, cu_q, cu_k, causal).astype(np.float32)
    assert_attention_close(got.cpu().numpy().astype(np.float32), ref, "queries %s, keys %s" % (lens_q, lens_k))


@pytest.mark.parametrize("block,sink,local", [(False, 4, 33), (False, 128, 256), (True, 1, 2)])
def test_streaming_heads(block, sink, local):
    import block_sparse_attn as bsa
    lens, Hq, Hk = [513, 90, 700], 8, 4
    n = sum(lens)
    rows = to_dev(np.random.default_rng(5).standard_normal((n, (Hq + 2 * Hk) * 128)).astype(np.float16))      # (views of one buffer: strided rows)
    q, k, v = (rows[:, a * 128:b * 128].view(n, -1, 128) for a, b in ((0, Hq), (Hq, Hq + Hk), (Hq + Hk, Hq + 2 * Hk)))
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    mask, info = np.repeat(np.asarray([0, -1, -1, 0], np.int32), Hq // Hk), np.asarray([sink, local] * Hq, np.int32)
    d = [to_dev(a) for a in (cu, cu, mask, info)]
    call = bsa.block_streaming_attn_func if block else bsa.token_streaming_attn_func
    got = _both(lambda: call(q, k, v, *d, max(lens), max(lens)))
    host = [t.cpu().numpy() for t in (q, k, v)]
    ref = oa.varlen_attention(*host, cu, cu, True, mask, info, block=128 if block else 1).astype(np.float32)
    assert_attention_close(got.cpu().numpy().astype(np.float32), ref, "block %s, sink %d, local %d" % (block, sink, local))
