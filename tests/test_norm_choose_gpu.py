"""Norm, router product and expert choice in one launch, and products over choices that are not sorted: the same bits as residual_norm, matmul, route and the
products over its order."""
import pytest
import torch

from omniserve_amd.backend.lm import lm_ops
from omniserve_amd.models.layers import padded

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(T, k, n, experts, ff, shared_ff, seed, ties):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV)      # noqa: E731
    wide = lambda t: padded(t, t.shape[0], k)      # noqa: E731
    vec = lambda: torch.nn.functional.pad(1 + 0.1 * rnd(n), (0, k - n))      # noqa: E731
    router = n ** -0.5 * rnd(experts, n)
    if ties:
        router[1::2] = router[:experts // 2 * 2:2][:router[1::2].shape[0]]      # pairs of experts with equal logits
    return dict(x=wide(rnd(T, n)), y=wide(rnd(T, n)).bfloat16(), post=(vec(), vec()), next=(vec(), vec()),
                router=padded(router.bfloat16(), (experts + 15) // 16 * 16, k), bias=None if ties else 0.1 * rnd(experts),
                w_in=(n ** -0.5 * rnd(experts, 2 * ff, k)).bfloat16(), w_out=(ff ** -0.5 * rnd(experts, k, ff)).bfloat16(),
                shared_in=(n ** -0.5 * rnd(2 * shared_ff, k)).bfloat16(), shared_out=(shared_ff ** -0.5 * rnd(k, shared_ff)).bfloat16())


@pytest.mark.parametrize("T,k,n,experts,top,kind", [
    (1, 2048, 2048, 64, 8, "layer"), (16, 2048, 2048, 64, 8, "layer"), (32, 2048, 2000, 64, 16, "rms"), (7, 2304, 2300, 48, 5, "layer"),
    (16, 4096, 4096, 32, 6, "layer"), (31, 4096, 4090, 64, 2, "rms"), (5, 2048, 2048, 17, 16, "layer"), (32, 2048, 2048, 9, 1, "layer")])
@pytest.mark.parametrize("ties", [False, True])
def test_one_launch(T, k, n, experts, top, kind, ties):
    ops = lm_ops(torch.bfloat16)
    ff, shared_ff = 640, 1024
    m = _inputs(T, k, n, experts, ff, shared_ff, T + k + experts, ties)
    assert ops.chooses(T, m["router"], experts, top, m["w_in"], m["w_out"])
    out = []
    for one in (False, True):
        x = m["x"].clone()
        h = torch.full((T, k), float("nan"), dtype=torch.bfloat16, device=DEV)
        if one:
            wts, order = ops.norm_choose(x, n, kind, 1e-5, m["y"], m["post"], m["next"], h, m["router"], m["bias"], experts, top)
        else:
            ops.residual_norm(x, n, kind, 1e-5, y=m["y"], post=m["post"], next=m["next"], h=h)
            wts, order = ops.route(ops.matmul(h, m["router"], out_f32=True), m["bias"], experts, top)
        act = torch.full((T * top, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
        act_s = torch.full((T, shared_ff), float("nan"), dtype=torch.bfloat16, device=DEV)
        y = torch.full((T * top + T, k), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.grouped(order, T, h, m["w_in"], act, False, True, (h, m["shared_in"], act_s))
        ops.grouped(order, T, act, m["w_out"], y, True, False, (act_s, m["shared_out"], y[T * top:]))
        out.append((x, h, wts, act, act_s, y))
    torch.cuda.synchronize()
    for name, a, b in zip(("residual", "h", "weights", "act", "shared act", "rows"), *out):
        assert torch.equal(a, b), name


def test_sizes_that_it_leaves():
    ops = lm_ops(torch.bfloat16)
    shape = lambda *s: torch.empty(s, dtype=torch.bfloat16, device="meta")      # noqa: E731
    big = (shape(64, 1280, 2048), shape(64, 2048, 640))
    assert ops.chooses(32, shape(64, 2048), 64, 8, *big)
    for T, experts, k in ((33, 64, 2048), (16, 65, 2048), (16, 64, 1024), (16, 64, 8192), (16, 64, 2112)):
        assert not ops.chooses(T, shape((experts + 15) // 16 * 16, k), experts, 8, *big)
    assert not lm_ops(torch.float32).chooses(16, shape(64, 2048), 64, 8, *big)


def test_empty_places_choose_nothing():
    ops, T, k, experts, top = lm_ops(torch.bfloat16), 8, 2048, 64, 8
    m = _inputs(T, k, k, experts, 640, 1024, 3, False)
    pos = torch.tensor([4, -1, 0, 7, -1, -1, 9, 1], dtype=torch.int32, device=DEV)
    full, out = pos >= 0, []
    for p in (None, pos):
        x, h = m["x"].clone(), torch.zeros((T, k), dtype=torch.bfloat16, device=DEV)
        wts, ids = ops.norm_choose(x, k, "layer", 1e-5, m["y"], m["post"], m["next"], h, m["router"], m["bias"], experts, top, p)
        act = torch.full((T * top, 640), -3.0, dtype=torch.bfloat16, device=DEV)
        ops.grouped(ids, T, h, m["w_in"], act, False, True)
        out.append((x, h, wts, ids, act.view(T, top, -1)))
    torch.cuda.synchronize()
    for a, b in zip(*out):
        assert torch.equal(a[full], b[full])
    x, h, wts, ids, act = out[1]
    assert torch.equal(x[~full], m["x"][~full]) and not h[~full].any() and not wts[~full].any() and (ids[~full] == -1).all() and (act[~full] == -3).all()


@pytest.mark.parametrize("shared_ff", [0, 1024])
def test_rows_that_nobody_wrote_stay_out_of_the_residual(shared_ff):
    """An empty place's pairs have no rows: whatever bits their memory holds, the norm behind adds none of them"""
    ops, T, k, experts, top = lm_ops(torch.bfloat16), 8, 2048, 64, 8
    m = _inputs(T, k, k, experts, 640, 1024, 5, False)
    pos = torch.tensor([4, -1, 0, 7, -1, -1, 9, 1], dtype=torch.int32, device=DEV)
    full, out = pos >= 0, []
    for p in (None, pos):
        x, h = m["x"].clone(), torch.ones((T, k), dtype=torch.bfloat16, device=DEV)
        wts, ids = ops.norm_choose(x, k, "layer", 1e-5, m["y"], m["post"], m["next"], h, m["router"], m["bias"], experts, top, p)
        new = lambda *s: torch.full(s, float("nan"), dtype=torch.bfloat16, device=DEV)      # noqa: E731
        act, act_s, y = new(T * top, 640), new(T, 1024), new(T * top + (T if shared_ff else 0), k)
        up, down = ((h, m["shared_in"], act_s), (act_s, m["shared_out"], y[T * top:])) if shared_ff else (None, None)
        ops.grouped(ids, T, h, m["w_in"], act, False, True, up)
        ops.grouped(ids, T, act, m["w_out"], y, True, False, down)
        if p is not None:
            assert y[:T * top].view(T, top, k)[~full].isnan().all()
        ops.residual_norm(x, k, "layer", 1e-5, y=y, experts=(wts, bool(shared_ff)), post=m["post"], next=m["next"], h=h)
        out.append((x, h))
    # weights of 0 behind others are weights: what their rows hold counts
    wts = torch.tensor([[0.5, 0.0]] * T, device=DEV)
    y = torch.ones((2 * T, k), dtype=torch.bfloat16, device=DEV)
    y[1::4] = float("nan")
    x = m["x"].clone()
    ops.residual_norm(x, k, "rms", 1e-5, y=y, experts=(wts, False))
    torch.cuda.synchronize()
    assert x[::2].isnan().all() and torch.equal(x[1::2], m["x"][1::2] + 0.5)
    for a, b in zip(*out):
        assert torch.equal(a[full], b[full]) and b.isfinite().all()


@pytest.mark.parametrize("top", [1, 2, 4, 5, 8, 9])
@pytest.mark.parametrize("k", [1024, 2048, 4096])
def test_weights_of_minus_zero_are_weights(top, k):
    """... but where a token has no other: a row behind them counts, wherever it stands"""
    ops = lm_ops(torch.bfloat16)
    x0 = torch.randn((top, k), device=DEV)
    y = torch.randn((top * top, k), device=DEV).bfloat16()
    x, wts = x0.clone(), torch.full((top, top), -0.0, device=DEV)
    wts.fill_diagonal_(0.5)
    ops.residual_norm(x, k, "rms", 1e-5, y=y, experts=(wts, False))
    assert torch.equal(x, x0 + 0.5 * y.view(top, top, k).diagonal().T.float())
