"""Latent attention's decode step with 16 and with 32 heads a workgroup: against float64 at lengths around a tile of 32 keys (the new row alone in a tile, at its end, first in the
next), and the same bits from a batch too large for 16 heads a workgroup as from its parts."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu

PAGE, RP, TP = 64, 64, 64
R, HALF, DK, ROT = 60, 12, 128, 72                    # latent columns and pairs that are there; a head's row, its first turned column


def _setup(lengths, heads, seed):
    gen = torch.Generator().manual_seed(seed)
    B, per = len(lengths), (max(lengths) + PAGE - 1) // PAGE
    row = RP + TP
    cache = torch.randn(B * per, PAGE, row, generator=gen)
    cache[..., R:RP] = 0
    cache[..., RP + 2 * HALF:] = 0
    x = torch.randn(B, heads * DK + row, generator=gen)
    x[:, heads * DK + R:heads * DK + RP] = 0
    qa = 0.3 * torch.randn(B, heads, RP, generator=gen)
    qa[..., R:] = 0
    bt = torch.randperm(B * per, generator=gen).int().view(B, per)
    pos = torch.tensor([n - 1 for n in lengths], dtype=torch.int32)
    slot = (bt[torch.arange(B), (pos // PAGE).long()] * PAGE + pos % PAGE).int()
    w, freq = 1 + 0.1 * torch.randn(RP, generator=gen), 0.7 ** torch.arange(HALF, dtype=torch.float32)
    return [t.to(dev()) for t in (x.bfloat16(), cache.bfloat16(), qa.bfloat16(), bt, pos, slot, w, freq)]


def _decode(x, cache, qa, bt, pos, slot, w, freq, heads, nsplit=1):
    from omniserve_amd.backend.lm import lm_ops
    ops, B, cache = lm_ops(torch.bfloat16), x.shape[0], cache.clone()
    o = torch.empty(B, heads * RP, dtype=torch.bfloat16, device=dev())
    part = torch.empty(B * heads * nsplit * (RP + 2), device=dev()) if nsplit > 1 else None
    ops.latent_decode(x, heads * DK, w, 1e-5, freq, pos, slot, cache, bt, qa.reshape(B, -1), o, part, nsplit, DK ** -0.5, (heads, DK, ROT, R, RP, TP))
    torch.cuda.synchronize()
    return o.view(B, heads, RP), cache


def _turn(t, pos, freq):
    a, b, ang = t[..., :HALF], t[..., HALF:2 * HALF], pos.double()[:, None] * freq.double()
    c, s = (f(ang).view(ang.shape[0], *([1] * (t.dim() - 2)), HALF) for f in (torch.cos, torch.sin))
    return torch.cat([a * c - b * s, b * c + a * s], -1)


@pytest.mark.parametrize("heads", [5, 16, 18, 32])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_latent_decode(heads, nsplit):
    lengths = [1, 31, 32, 33, 64, 65, 96, 97, 200, 300]
    args = _setup(lengths, heads, heads)
    x, cache, qa, bt, pos, slot, w, freq = [t.cpu().double() if t.is_floating_point() else t.cpu() for t in args]
    got, written = _decode(*args, heads, nsplit)
    new = x[:, heads * DK:]
    lat = new[:, :RP] / (new[:, :R].square().sum(-1, keepdim=True) / R + 1e-5).sqrt() * w
    rows = torch.cat([lat, _turn(new[:, RP:RP + 2 * HALF], pos, freq), torch.zeros(len(lengths), TP - 2 * HALF)], -1)
    flat = written.cpu().double().view(-1, RP + TP)
    # rounded once: half a unit of bf16 in the last place, and the float32 arithmetic before it
    assert ((flat[slot.long()] - rows).abs() <= 2.0 ** -8 * rows.abs() + 1e-5).all()
    q = _turn(x[:, :heads * DK].view(len(lengths), heads, DK)[..., ROT:ROT + 2 * HALF], pos, freq).bfloat16().double()
    for b, n in enumerate(lengths):
        c = written.cpu().double()[bt[b].long()].reshape(-1, RP + TP)[:n]
        p = torch.softmax((qa[b] @ c[:, :RP].T + q[b] @ c[:, RP:RP + 2 * HALF].T) * DK ** -0.5, -1)
        want = p @ c[:, :RP]
        # probabilities in bf16 (2^-8 of each term at most), queries' turned part rounded at a neighbouring value now and then, the result in bf16
        bound = 2.0 ** -6 * (p @ c[:, :RP].abs()) + 2.0 ** -8 * want.abs()
        assert ((got[b].cpu().double() - want).abs() <= bound).all(), (heads, n)


def test_large_batches_give_the_same_bits():
    heads, B = 32, 1100                               # 2200 workgroups of 16 heads: more than are on the chip at once
    args = _setup([1 + (37 * i) % 130 for i in range(B)], heads, 3)
    whole, _ = _decode(*args, heads)
    x, cache, qa, bt, pos, slot, w, freq = args
    for i in range(0, B, 100):
        cut = slice(i, i + 100)
        part, _ = _decode(x[cut], cache, qa[cut], bt[cut], pos[cut], slot[cut], w, freq, heads)
        assert torch.equal(whole[cut], part), i
