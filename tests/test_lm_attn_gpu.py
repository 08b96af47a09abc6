"""Prompt attention of the engine's models (lm_attn_prefill) against float64: every form of the kernel, tiles that end inside a wave, a page
and a workgroup, prompts continued at a position, windows, grouped heads, gated outputs."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu
PAGE = 64


def _run(dtype, dk, dv, heads, kv_heads, entries, window, gated, seed):
    """entries: (tokens, position of the first one)"""
    from omniserve_amd.backend.lm import lm_ops
    ops = lm_ops(dtype)
    gen = torch.Generator(device=dev()).manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, device=dev(), generator=gen)      # noqa: E731
    total = sum(n for n, _ in entries)
    pages = [(n + p0 + PAGE - 1) // PAGE for n, p0 in entries]
    q = rnd(total, heads * dk).to(dtype)
    k, v = rnd(sum(pages) + 1, kv_heads, PAGE, dk).to(dtype), rnd(sum(pages) + 1, kv_heads, PAGE, dv).to(dtype)
    gate = rnd(total, heads * dv).to(dtype) if gated else None
    number = torch.randperm(sum(pages) + 1, device=dev(), generator=gen).int()
    bt = torch.zeros(len(entries), max(pages), dtype=torch.int32, device=dev())
    entry, tiles, t0, p_at = [], [], 0, 0
    for i, (n, p0) in enumerate(entries):
        bt[i, :pages[i]] = number[p_at:p_at + pages[i]]
        entry.append([t0, n, p0, i])
        tiles += [[i, r] for r in range(0, n, 128)]
        t0, p_at = t0 + n, p_at + pages[i]
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device=dev())      # noqa: E731
    out = torch.full((total, heads * dv), float("nan"), dtype=dtype, device=dev())
    scale = dk ** -0.5
    ops.attn_prefill(q, k, v, bt, ints(entry), ints(tiles), gate, out, scale, window, heads, kv_heads, dk, dv)
    torch.cuda.synchronize()
    assert not out.isnan().any()

    for i, (t, n, p0, _) in enumerate(entry):
        length = n + p0
        kk = k[bt[i, :pages[i]].long()].transpose(0, 1).reshape(kv_heads, -1, dk)[:, :length].double()
        vv = v[bt[i, :pages[i]].long()].transpose(0, 1).reshape(kv_heads, -1, dv)[:, :length].double()
        kk, vv = kk.repeat_interleave(heads // kv_heads, 0), vv.repeat_interleave(heads // kv_heads, 0)
        qq = q[t:t + n].double().view(n, heads, dk).transpose(0, 1).contiguous()
        qpos = torch.arange(p0, p0 + n, device=dev())[:, None]
        key = torch.arange(length, device=dev())[None]
        s = (qq @ kk.transpose(1, 2).contiguous()) * scale
        s = s.masked_fill((key > qpos) | (key <= qpos - window), float("-inf"))
        prob = s.softmax(-1)
        ref, size = prob @ vv, prob @ vv.abs()
        sums = (qq.abs() @ kk.abs().transpose(1, 2).contiguous()).max() * scale
        if gated:
            g = torch.sigmoid(gate[t:t + n].double()).view(n, heads, dv).transpose(0, 1)
            ref, size = ref * g, size * g
        got = out[t:t + n].double().view(n, heads, dv).transpose(0, 1)
        # the result's rounding; then relative to sum p |v|: scores in f32 (their error enters every p and the sum), 16 bits of a p, the exponential
        unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
        bound = 1.01 * unit * ref.abs() + (2 * dk * 2.0 ** -24 * sums + 2.0 ** -16 + length * 2.0 ** -24 + 1e-6) * size
        assert ((got - ref).abs() <= bound).all(), ((got - ref).abs() / bound).max()


@pytest.mark.parametrize("entries,window", [([(1, 0), (31, 0), (33, 5), (127, 64)], 1 << 30), ([(130, 0), (257, 190)], 1 << 30), ([(300, 0), (64, 127), (129, 300)], 100),
                                            ([(200, 50)], 1), ([(385, 0)], 64)])
@pytest.mark.parametrize("dk,dv", [(192, 128), (64, 256), (256, 64), (128, 128), (64, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_prompt_attention(dtype, dk, dv, entries, window):
    _run(dtype, dk, dv, 4, 2, entries, window, gated=False, seed=dk + dv)


@pytest.mark.parametrize("heads,kv_heads", [(3, 3), (8, 1), (16, 16)])
def test_prompt_attention_heads_and_gate(heads, kv_heads):
    _run(torch.bfloat16, 192, 128, heads, kv_heads, [(150, 10), (97, 0)], 1 << 30, gated=True, seed=heads)


def _rows_per_wave(dtype, dk, dv, heads, entries):
    from omniserve_amd.backend.lm import lm_ops
    return lm_ops(dtype)._h.lm_attn_prefill_rows(dk, dv, sum(-(-n // 128) for n, _ in entries), heads)


# The 32-row form of bf16, which takes more than 256 workgroups: the same ends of tiles, pages and windows with as many heads, kv heads whole to an
# XCD (8) and not (17, 136).
@pytest.mark.parametrize("entries,window", [([(1, 0), (31, 0), (33, 5), (127, 64)], 1 << 30), ([(130, 0), (257, 190)], 1 << 30), ([(300, 0), (64, 127), (129, 300)], 100),
                                            ([(200, 50)], 1), ([(385, 0)], 64)])
@pytest.mark.parametrize("dk,dv,kv_heads,gated", [(192, 128, 8, False), (192, 128, 17, True), (192, 128, 136, False), (64, 256, 17, False), (256, 64, 8, True)])
def test_prompt_attention_rows32(dk, dv, kv_heads, gated, entries, window):
    assert _rows_per_wave(torch.bfloat16, dk, dv, 136, entries) == 32
    _run(torch.bfloat16, dk, dv, 136, kv_heads, entries, window, gated=gated, seed=dk + kv_heads)
