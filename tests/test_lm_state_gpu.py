"""Decode steps of the recurrent layers with a state larger than the caches (streamed) against the same sequences in batches whose state is
not: the same bits in outputs and states.  (The small batches are held against the oracle by the models' tests.)"""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layer", ["gla", "delta"])
@pytest.mark.parametrize("batch,heads,dk,dv,positions", [(16, 16, 128, 128, 1), (33, 8, 128, 128, 3), (64, 4, 64, 256, 2), (9, 16, 256, 128, 4)])
def test_streamed_state(layer, batch, heads, dk, dv, positions):
    assert batch * heads * dk * dv * 4 >= 16 << 20
    from omniserve_amd.backend.lm import lm_ops
    ops = lm_ops(torch.bfloat16)
    gen = torch.Generator(device=dev()).manual_seed(batch + dk)
    rnd = lambda *shape: torch.randn(*shape, device=dev(), generator=gen)      # noqa: E731
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=dev())      # noqa: E731
    qkv = 2 * heads * dk + heads * dv
    width = qkv + heads * dv + 64
    x = rnd(batch, width).bfloat16()
    state = rnd(batch + 1, heads, dk, dv) * 0.1
    ring = rnd(batch + 1, 4, qkv)
    slot = torch.randperm(batch + 1, device=dev(), generator=gen)[:batch].int()
    pos = [p % positions for p in range(batch)]                                 # some at the start of their sequence
    pos[batch // 2] = -1                                                        # an empty place
    pos = ints(pos)
    w = rnd(dv)
    a2, bias = rnd(heads * dk, 16).bfloat16() * 0.1, rnd(heads * dk)
    conv, a_log, dt_bias = rnd(4, qkv) * 0.5, rnd(heads), rnd(heads)

    def run(rows, st, rg):
        o = torch.zeros(len(rows), heads * dv, dtype=torch.bfloat16, device=dev())
        xs, sl, ps = x[rows], slot[rows], pos[rows]
        if layer == "gla":
            ops.gla_decode(xs, o, st, sl, ps, qkv + heads * dv, a2, bias, 16.0, dk ** -0.5, qkv, w, dv, 1e-6, heads, dk, dv)
        else:
            ops.delta_decode(xs, o, st, rg, sl, ps, conv, 1e-6, dk ** -0.5, qkv + heads * dv, a_log, dt_bias, qkv, w, dv, 1e-6, heads, heads, dk, dv)
        return o

    one, one_ring = state.clone(), ring.clone()
    whole = run(list(range(batch)), one, one_ring)
    parts, parts_ring = state.clone(), ring.clone()
    split = torch.cat([run(list(range(r, min(r + 4, batch))), parts, parts_ring) for r in range(0, batch, 4)])
    torch.cuda.synchronize()
    assert torch.equal(whole, split) and torch.equal(one, parts) and torch.equal(one_ring, parts_ring)
    assert not torch.equal(one, state) and whole.float().abs().sum() > 0


@pytest.mark.parametrize("layer", ["linear", "gla", "delta"])
def test_more_than_65535_places(layer):
    """A batch of mostly empty places, the last of them beyond what the second dimension of a grid may count: the sequences in it as in a batch of their own."""
    from omniserve_amd.backend.lm import lm_ops
    ops = lm_ops(torch.bfloat16)
    batch, dk, dv = 65600, 64, 64
    rows = [0, 65535, batch - 1]
    gen = torch.Generator(device=dev()).manual_seed(5)
    rnd = lambda *shape: torch.randn(*shape, device=dev(), generator=gen)      # noqa: E731
    qkv = 2 * dk + dv
    few, st0, rg0 = rnd(3, qkv + dv + 64).bfloat16(), rnd(3, 1, dk, dv) * 0.1, rnd(3, 4, qkv)
    x = torch.zeros((batch, few.shape[1]), dtype=torch.bfloat16, device=dev())
    x[rows] = few
    pos, slot = torch.full((batch,), -1, dtype=torch.int32, device=dev()), torch.zeros((batch,), dtype=torch.int32, device=dev())
    pos[rows], slot[rows] = 2, torch.arange(3, dtype=torch.int32, device=dev())
    w, a2, bias, conv, a_log, dt_bias, decay = rnd(dv), rnd(dk, 16).bfloat16() * 0.1, rnd(dk), rnd(4, qkv) * 0.5, rnd(1), rnd(1), -rnd(1).abs()

    def run(xs, sl, ps):
        o, st, rg = torch.zeros((xs.shape[0], dv), dtype=torch.bfloat16, device=dev()), st0.clone(), rg0.clone()
        if layer == "linear":
            ops.linear_decode(xs, o, st, sl, ps, decay, 1, dk, dv, "silu")
        elif layer == "gla":
            ops.gla_decode(xs, o, st, sl, ps, qkv + dv, a2, bias, 16.0, dk ** -0.5, qkv, w, dv, 1e-6, 1, dk, dv)
        else:
            ops.delta_decode(xs, o, st, rg, sl, ps, conv, 1e-6, dk ** -0.5, qkv + dv, a_log, dt_bias, qkv, w, dv, 1e-6, 1, 1, dk, dv)
        torch.cuda.synchronize()
        return o, st, rg

    o, *after = run(x, slot, pos)
    want, *want_after = run(few, slot[rows].contiguous(), pos[rows].contiguous())
    assert torch.equal(o[rows], want) and not o[1:65535].any()
    assert all(torch.equal(a, b) for a, b in zip(after, want_after))
