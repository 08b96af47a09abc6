"""The engine's products (csrc/lm/lm_gemm.hip).  Few rows: every width of a workgroup, K in parts and in slices, fewer stages than parts, row counts
at the edges of 16, views with a row stride, the gated unit, one matrix per head, experts with many rows.  Many rows: whole and half tiles, several in
turn on a workgroup, experts without rows.  Against float64."""
import ctypes

import pytest
import torch

from tests.hybrid_util import errors

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = [torch.bfloat16, torch.float32]
TOL = {torch.bfloat16: 4e-3, torch.float32: 2e-6}      # the output's rounding (up to 2^-8 of a value); f32 sums


def _ops(dtype):
    from omniserve_amd.backend.lm import lm_ops
    return lm_ops(dtype)


def _randn(seed, dtype, *shape):
    return torch.randn(shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).to(dtype)


def _close(got, want, dtype):
    assert errors(got.float().cpu().numpy(), want.cpu().numpy()).max() < TOL[dtype]


def _rows_close(got, want, dtype):
    """Rounding a value to bf16 moves it by at most 2^-8 of itself (7 fraction bits), so a row's error is at most 2^-8 of the row's own norm (5 % for the f32
    sums in front of it); in f32 the exponential's few ulp."""
    d = (got.double().cpu() - want.cpu()).norm(dim=1) / want.cpu().norm(dim=1)
    assert d.max() < (1.05 * 2.0 ** -8 if dtype == torch.bfloat16 else 5e-6)


# one stage for four K parts; 16 .. 80 channels per workgroup; more than 256 of them; slices of K with an uneven rest
SHAPES = [(1, 16, 64), (2, 48, 192), (15, 4096, 320), (16, 64, 4096), (17, 4112, 256), (31, 6208, 128), (32, 10816, 64), (33, 16448, 192),
          (47, 12352, 64), (48, 1024, 8256), (49, 32016, 64), (64, 2048, 6144), (64, 528, 3136)]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_products(m, n, k, dtype):
    ops = _ops(dtype)
    x, w = _randn(1, dtype, m, k + 64)[:, 64:], _randn(2, dtype, n, k) * k ** -0.5
    want = x.double() @ w.double().t()
    guard = torch.full((m + 2, n), 7.0, dtype=dtype, device=DEV)
    _close(ops.matmul(x, w, out=guard[1:-1]), want, dtype)
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()
    assert errors(ops.matmul(x, w, out_f32=True, scale=0.5).cpu().numpy(), 0.5 * want.cpu().numpy()).max() < 2e-6
    assert torch.equal(ops.matmul(x, w), ops.matmul(x, w))


def _rows_plan(ops, groups, n, k, rows, epi=0, sliced=1):
    slices = ctypes.c_int(0)
    return ops._h.lm_gemm_rows_channels(groups, n, k, rows, epi, sliced, ctypes.byref(slices)), slices.value


# Every width with whole rings and with fewer stages than the ring holds, in slices of K, in K parts (at most 256 workgroups) and without; the kernel
# without a stream.  Channels that end inside a workgroup, row counts around 16.
# (k of bf16; half of it in f32, whose stages hold half as many)
WIDTHS = [(16, 1, 16, 4096, 1024), (16, 8, 17, 256, 4096), (32, 1, 33, 6224, 256), (32, 8, 64, 528, 3200), (48, 1, 48, 10816, 4096), (48, 1, 33, 10816, 512),
          (64, 1, 64, 12352, 4096), (64, 1, 49, 32016, 128), (64, 8, 64, 2048, 6144), (80, 1, 48, 16448, 4096), (80, 1, 17, 16448, 256), (80, 8, 1, 12352, 4096),
          (0, 1, 33, 64, 1024), (0, 1, 64, 240, 2048), (0, 1, 16, 4096, 128), (0, 1, 3, 528, 256)]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("channels,slices,m,n,k", WIDTHS)
def test_every_width(channels, slices, m, n, k, dtype):
    ops, k = _ops(dtype), k // (1 if dtype == torch.bfloat16 else 2)
    assert _rows_plan(ops, 1, n, k, m) == (channels, slices)
    x, w = _randn(21, dtype, m, k + 64)[:, 64:], _randn(22, dtype, n, k) * k ** -0.5
    want = x.double() @ w.double().t()
    guard = torch.full((m + 2, n), 7.0, dtype=dtype, device=DEV)
    _close(ops.matmul(x, w, out=guard[1:-1]), want, dtype)
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()
    assert errors(ops.matmul(x, w, out_f32=True, scale=0.5).cpu().numpy(), 0.5 * want.cpu().numpy()).max() < 2e-6


@pytest.mark.parametrize("m,n,k", [(64, 32032, 2048), (17, 28704, 4160), (1, 32768, 4096), (48, 28672, 4096)])
def test_workgroups_of_128_channels(m, n, k):
    """bf16 only: one round of them; channels that end inside one, uneven stages, the gated unit"""
    ops = _ops(torch.bfloat16)
    assert _rows_plan(ops, 1, n, k, m) == (128, 1) and _rows_plan(ops, 1, n, k, m, 2) == (128, 1)
    x, w = _randn(31, torch.bfloat16, m, k + 64)[:, 64:], _randn(32, torch.bfloat16, n, k) * k ** -0.5
    want = x.double() @ w.double().t()
    guard = torch.full((m + 2, n), 7.0, device=DEV)
    ops.matmul(x, w, out=guard[1:-1], out_f32=True)
    assert errors(guard[1:-1].cpu().numpy(), want.cpu().numpy()).max() < 2e-6
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()
    y = want.view(m, n // 32, 2, 16)
    unit = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(m, n // 2)
    assert errors(ops.glu(x, w, None, "silu").float().cpu().numpy(), unit.cpu().numpy()).max() < TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (16, 1040, 128), (33, 2064, 192), (64, 512, 4160), (48, 9216, 64)])
def test_gated_unit(m, n, k, dtype):
    ops = _ops(dtype)
    x, w, b = _randn(3, dtype, m, k), _randn(4, dtype, 2 * n, k) * k ** -0.5, _randn(5, torch.float32, 2 * n) * 0.1
    y = (x.double() @ w.double().t() + b.double()).view(m, n // 16, 2, 16)
    want = (torch.nn.functional.gelu(y[:, :, 0], approximate="tanh") * y[:, :, 1]).reshape(m, n)
    got = ops.glu(x, w, b, "gelu_tanh")
    assert errors(got.float().cpu().numpy(), want.cpu().numpy()).max() < max(TOL[dtype], 5e-6)      # (the exponential's few ulp)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m", [1, 16, 50, 65, 130])
@pytest.mark.parametrize("heads,n,k", [(32, 128, 512), (16, 256, 128), (3, 64, 64)])
def test_one_matrix_per_head(heads, n, k, m, dtype):
    ops = _ops(dtype)
    x, w = _randn(6, dtype, m, heads * k), _randn(7, dtype, heads, n, k) * k ** -0.5
    gate, out = _randn(8, dtype, m, heads * n), torch.empty((m, heads * n), dtype=dtype, device=DEV)
    want = torch.cat([x[:, h * k:(h + 1) * k].double() @ w[h].double().t() for h in range(heads)], dim=1)
    _close(ops.head_products(x, w, out, k, n), want, dtype)
    got = ops.head_products(x, w, out, k, n, gate=gate)
    assert errors(got.float().cpu().numpy(), (want * torch.sigmoid(gate.double())).cpu().numpy()).max() < max(TOL[dtype], 5e-6)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("tokens,skew", [(1, False), (16, False), (64, False), (64, True)])
def test_experts(tokens, skew, dtype):
    """skew: every token chooses the same experts, 64 rows each"""
    ops = _ops(dtype)
    E, top, ff, W = 6, 3, 192, 256
    z, bias = _randn(9, torch.float32, tokens, E), torch.zeros((E,), device=DEV)
    if skew:
        z = z * 0 + torch.arange(E, device=DEV)
    wts, order = ops.route(z.contiguous(), bias, E, top)
    h, w, ws = _randn(10, dtype, tokens, W), _randn(11, dtype, E, ff, W) * W ** -0.5, _randn(12, dtype, 2 * ff, W) * W ** -0.5
    y, ys = (torch.empty((r, c), dtype=dtype, device=DEV) for r, c in ((tokens * top, ff), (tokens, 2 * ff)))
    ops.grouped(order, tokens, h, w, y, False, False, (h, ws, ys))
    ids = torch.argsort(-z, dim=1, stable=True)[:, :top]
    want = torch.einsum("tw,tcfw->tcf", h.double(), w.double()[ids]).reshape(tokens * top, ff)
    _close(y, want, dtype)
    _close(ys, h.double() @ ws.double().t(), dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m,n,k", [(65, 144, 64), (256, 256, 128), (257, 272, 192), (700, 1040, 320), (1300, 528, 1792)])
def test_tiles(m, n, k, dtype):
    """many rows: two stages of k and more, one tile and parts of tiles in both directions"""
    ops = _ops(dtype)
    x, w = _randn(13, dtype, m, k + 64)[:, 64:], _randn(14, dtype, n, k) * k ** -0.5
    guard = torch.full((m + 2, n), 7.0, device=DEV)
    ops.matmul(x, w, out=guard[1:-1], out_f32=True)
    assert errors(guard[1:-1].cpu().numpy(), (x.double() @ w.double().t()).cpu().numpy()).max() < 2e-6
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("tokens,E,top,ff,W,skew", [(66, 6, 3, 192, 256, False), (300, 4, 2, 272, 320, True), (1000, 8, 2, 64, 128, False)])
def test_experts_of_a_prompt(tokens, E, top, ff, W, skew, dtype):
    """experts without rows, with whole tiles and parts of them; the gated unit and the plain product, a shared expert beside them"""
    ops = _ops(dtype)
    z, bias = _randn(15, torch.float32, tokens, E), torch.zeros((E,), device=DEV)
    if skew:
        z = z * 0 + torch.arange(E, device=DEV)
    wts, order = ops.route(z.contiguous(), bias, E, top)
    h = _randn(16, dtype, tokens, W)
    wi, ws = _randn(17, dtype, E, 2 * ff, W) * W ** -0.5, _randn(18, dtype, 96, W) * W ** -0.5
    wo, wd = _randn(19, dtype, E, W, (ff + 63) // 64 * 64) * ff ** -0.5, _randn(20, dtype, W, 64) * 0.1
    act = torch.zeros((tokens * top, wo.shape[2]), dtype=dtype, device=DEV)
    acts, y = torch.zeros((tokens, 64), dtype=dtype, device=DEV), torch.empty((tokens * (top + 1), W), dtype=dtype, device=DEV)
    ops.grouped(order, tokens, h, wi, act, False, True, (h, ws, acts))
    ids = torch.argsort(-z, dim=1, stable=True)[:, :top].cpu()

    def glu(x, w):
        v = (x @ w.t()).view(x.shape[0], w.shape[0] // 32, 2, 16)
        return (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(x.shape[0], w.shape[0] // 2)

    hd = h.double().cpu()
    want, wid, wod = torch.empty((tokens * top, ff), dtype=torch.float64), wi.double().cpu(), wo.double().cpu()
    for e in range(E):
        t, c = torch.nonzero(ids == e, as_tuple=True)
        want[t * top + c] = glu(hd[t], wid[e])
    _rows_close(act[:, :ff], want, dtype)
    _rows_close(acts[:, :48], glu(hd, ws.double().cpu()), dtype)
    ops.grouped(order, tokens, act, wo, y, True, False, (acts, wd, y[tokens * top:]))
    down = torch.empty((tokens * top, W), dtype=torch.float64)
    a = act.double().cpu()
    for e in range(E):
        t, c = torch.nonzero(ids == e, as_tuple=True)
        down[t * top + c] = a[t * top + c] @ wod[e].t()
    _rows_close(y[:tokens * top], down, dtype)
    _rows_close(y[tokens * top:], acts.double() @ wd.double().t(), dtype)


def _channels(ops, n, k, groups=1, max_tiles=0, rows=0, n_b=0, k_b=0, rows_b=0):
    return ops._h.lm_gemm_tile_channels(n, k, groups, max_tiles, rows, n_b, k_b, rows_b)


def _matrix_close(got, want, dtype):
    """errors() of the whole result, on the GPU"""
    want = want.float() if got.dtype == torch.float32 else want
    assert ((got.double() - want).norm() / want.double().norm()) < TOL[dtype] and ((got.double() - want).abs().max() / want.double().square().mean().sqrt()) < 16 * TOL[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m,n,k,channels", [(2000, 16112, 2048, 256), (3000, 16112, 1024, 256), (255, 32784, 1024, 256), (255, 32016, 1024, 128), (1000, 8160, 2048, 128), (4100, 16400, 64, 128), (2100, 4112, 192, 128)])
def test_tiles_in_turn(m, n, k, channels, dtype):
    """many rows to f32: whole and half tiles, two and three whole ones in turn on a workgroup"""
    ops = _ops(dtype)
    assert _channels(ops, n, k, rows=m) == channels
    x, w = _randn(23, dtype, m, k + 64)[:, 64:], _randn(24, dtype, n, k) * k ** -0.5
    guard = torch.full((m + 2, n), 7.0, device=DEV)
    ops.matmul(x, w, out=guard[1:-1], out_f32=True)
    _matrix_close(guard[1:-1], x.double() @ w.double().t(), torch.float32)
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("tokens,E,top,n,k,channels", [(70, 62, 3, 4096, 64, 256), (71, 62, 3, 3072, 128, 256), (66, 62, 3, 2048, 192, 256), (80, 62, 3, 4064, 1024, 256),
                                                       (70, 64, 3, 1376, 64, 128), (700, 16, 4, 2080, 192, 128), (2800, 16, 4, 4096, 2048, 256)])
@pytest.mark.parametrize("glu", [False, True])
def test_experts_in_turn(tokens, E, top, n, k, channels, glu, dtype):
    """Experts and a shared one: two to four whole tiles in turn on a workgroup, of one, two and more stages of k, experts without rows between them;
    half tiles.  Every row, and what lies around the results stays as it was."""
    ops = _ops(dtype)
    max_tiles = ops._h.lm_route_max_tiles(tokens, E, top)
    assert _channels(ops, n, k, E, max_tiles, n_b=544, k_b=k, rows_b=tokens) == channels
    z = _randn(25, torch.float32, tokens, E)
    z[:, E // 4:E // 2] -= 100                                           # nobody chooses these
    wts, order = ops.route(z.contiguous(), torch.zeros((E,), device=DEV), E, top)
    h, w, ws = _randn(26, dtype, tokens, k), _randn(27, dtype, E, n, k) * k ** -0.5, _randn(28, dtype, 544, k) * k ** -0.5
    out = n // 2 if glu else n
    y = torch.full((tokens * top + 2, out), 7.0, dtype=dtype, device=DEV)
    ys = torch.full((tokens + 2, 272 if glu else 544), 7.0, dtype=dtype, device=DEV)
    ops.grouped(order, tokens, h, w, y[1:-1], False, glu, (h, ws, ys[1:-1]))
    for edge in (y[0], y[-1], ys[0], ys[-1]):
        assert (edge == 7).all()

    def product(x, m):
        v = x.double() @ m.double().t()
        if glu:
            v = v.view(x.shape[0], m.shape[0] // 32, 2, 16)
            v = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(x.shape[0], m.shape[0] // 2)
        return v

    ids = torch.argsort(-z, dim=1, stable=True)[:, :top]
    want = torch.empty((tokens * top, out), dtype=torch.float64, device=DEV)
    for e in range(E):
        t, c = torch.nonzero(ids == e, as_tuple=True)
        want[t * top + c] = product(h[t], w[e])
    _rows_close(y[1:-1], want.cpu(), dtype)
    _rows_close(ys[1:-1], product(h, ws).cpu(), dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("n,k", [(12288, 64), (12288, 192), (4096, 512)])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("empty,says", [(0, 0), (3, 14), (3, 0)])
def test_tables_of_experts_rows(empty, says, glu, n, k, dtype):
    """Whole tiles of a table without an entry to spare, with empty ones that say how many tiles there are, and with empty ones that do not; tiles of 1, 128 and 129 rows among them"""
    ops, counts = _ops(dtype), [256, 129, 1100, 1, 128, 1025]
    off, tiles = [0], []
    for e, c in enumerate(counts):
        tiles += [(e, off[-1] + r, min(256, c - r), 0) for r in range(0, c, 256)]
        off.append(off[-1] + c)
    assert len(tiles) == 14
    tiles += [(0, 0, 0, says)] * empty
    assert _channels(ops, n, k, len(counts), len(tiles)) == 256
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)      # noqa: E731
    perm = torch.randperm(off[-1], generator=torch.Generator(device=DEV).manual_seed(3), device=DEV).int()
    x, w = _randn(41, dtype, off[-1], k), _randn(42, dtype, len(counts), n, k) * k ** -0.5
    y = torch.full((off[-1] + 2, n // 2 if glu else n), 7.0, dtype=dtype, device=DEV)
    ops.grouped((i32(off), perm, i32(tiles), len(tiles), 1), 0, x, w, y[1:-1], True, glu)
    assert (y[0] == 7).all() and (y[-1] == 7).all()
    want = torch.empty(y[1:-1].shape, dtype=torch.float64, device=DEV)
    for e in range(len(counts)):
        rows = perm[off[e]:off[e + 1]].long()
        v = x[rows].double() @ w[e].double().t()
        if glu:
            v = v.view(len(rows), n // 32, 2, 16)
            v = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(len(rows), n // 2)
        want[rows] = v
    _rows_close(y[1:-1], want.cpu(), dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m", [1, 20, 64])
def test_few_rows_between_boundaries(m, dtype):
    """x and w that start between two 16-byte boundaries, which the stream's DMA does not take: plain, gated, per head, experts"""
    ops, shift = _ops(dtype), 8 // torch.empty((), dtype=dtype).element_size()

    def between(seed, gain, *shape):      # (all rows of one size, unlike each other: errors() relates a row to the mean of all)
        n = torch.Size(shape).numel()
        t = (_randn(seed, torch.float32, n + 16) * gain).to(dtype)[shift:shift + n].view(shape)
        assert t.data_ptr() % 16 == 8
        return t

    x, w, b = between(29, 1, m, 1024), _randn(30, dtype, 544, 1024) / 32, _randn(33, torch.float32, 544) * 0.1
    ws = between(31, 1 / 32, 544, 1024)
    want = x.double() @ ws.double().t()
    _close(ops.matmul(x, ws), want, dtype)
    _close(ops.matmul(x, w), x.double() @ w.double().t(), dtype)
    y = (want + b.double()).view(m, 17, 2, 16)
    got = ops.glu(x, ws, b, "gelu_tanh")
    want = (torch.nn.functional.gelu(y[:, :, 0], approximate="tanh") * y[:, :, 1]).reshape(m, 272)
    assert errors(got.float().cpu().numpy(), want.cpu().numpy()).max() < max(TOL[dtype], 5e-6)
    wh, out = between(32, 1 / 16, 4, 128, 256), torch.empty((m, 512), dtype=dtype, device=DEV)
    ops.head_products(x, wh, out, 256, 128)
    _close(out, torch.cat([x[:, 256 * h:256 * h + 256].double() @ wh[h].double().t() for h in range(4)], dim=1), dtype)
    z = _randn(34, torch.float32, m, 6)
    wts, order = ops.route(z, torch.zeros((6,), device=DEV), 6, 3)
    we, y, ys = _randn(35, dtype, 6, 192, 1024) / 32, torch.empty((m * 3, 192), dtype=dtype, device=DEV), torch.empty((m, 544), dtype=dtype, device=DEV)
    ops.grouped(order, m, x, we, y, False, False, (x, ws, ys))
    ids = torch.argsort(-z, dim=1, stable=True)[:, :3]
    _close(y, torch.stack([x[t].double() @ we[ids[t, c]].double().t() for t in range(m) for c in range(3)]), dtype)
    _close(ys, x.double() @ ws.double().t(), dtype)


# What goes around the stream: 32 channels per workgroup (short K of many channels, some past the last whole workgroup), 16 rows in turn (heads of few
# channels), the gated unit in 16 - 64 rows at once.
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("heads,n,k,m", [(1, 9616, 64, 16), (1, 16368, 128, 9), (32, 512, 128, 1), (36, 272, 64, 16), (8, 256, 256, 17), (16, 128, 192, 32)])
def test_short_k(heads, n, k, m, dtype):
    ops = _ops(dtype)
    assert _rows_plan(ops, heads, n, k, m, sliced=heads == 1) == (0, 1)
    x, w = _randn(36, dtype, m, heads * k), _randn(37, dtype, heads, n, k) * k ** -0.5
    gate, guard = _randn(38, dtype, m, heads * n), torch.full((m + 2, heads * n), 7.0, dtype=dtype, device=DEV)
    want = torch.cat([x[:, h * k:(h + 1) * k].double() @ w[h].double().t() for h in range(heads)], dim=1)
    _close(ops.head_products(x, w, guard[1:-1], k, n), want, dtype)
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()
    got = ops.head_products(x, w, guard[1:-1], k, n, gate=gate)
    assert errors(got.float().cpu().numpy(), (want * torch.sigmoid(gate.double())).cpu().numpy()).max() < max(TOL[dtype], 5e-6)
    if heads == 1:
        assert errors(ops.matmul(x, w[0], out_f32=True, scale=0.5).cpu().numpy(), 0.5 * want.cpu().numpy()).max() < 2e-6


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m,n,k", [(1, 2080, 512), (17, 2048, 512), (32, 4096, 448), (31, 2080, 64), (33, 2080, 512), (64, 4096, 512)])
def test_small_gated_units(m, n, k, dtype):
    ops = _ops(dtype)
    assert (_rows_plan(ops, 1, n, k, m, epi=2)[0] == 0) == (m <= 32 or dtype == torch.float32)
    x, w, b = _randn(39, dtype, m, k), _randn(40, dtype, n, k) * k ** -0.5, _randn(41, torch.float32, n) * 0.1
    y = (x.double() @ w.double().t() + b.double()).view(m, n // 32, 2, 16)
    want = (torch.nn.functional.gelu(y[:, :, 0], approximate="tanh") * y[:, :, 1]).reshape(m, n // 2)
    assert errors(ops.glu(x, w, b, "gelu_tanh").float().cpu().numpy(), want.cpu().numpy()).max() < max(TOL[dtype], 5e-6)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("tokens", [1, 5, 16])
@pytest.mark.parametrize("E,n", [(24, 400), (16, 512), (5, 80)])
def test_experts_of_few_tokens(E, n, tokens, dtype):
    """more than 8192 channels (the stream) and fewer, a part b that ends before and behind the experts' channels"""
    ops, top, W = _ops(dtype), 3, 320
    z = _randn(42, torch.float32, tokens, E)
    wts, order = ops.route(z, torch.zeros((E,), device=DEV), E, top)
    h, w, ws = _randn(43, dtype, tokens, W), _randn(44, dtype, E, n, W) * W ** -0.5, _randn(45, dtype, 432, W) * W ** -0.5
    y, ys = torch.full((tokens * top + 2, n), 7.0, dtype=dtype, device=DEV), torch.full((tokens + 2, 432), 7.0, dtype=dtype, device=DEV)
    ops.grouped(order, tokens, h, w, y[1:-1], False, False, (h, ws, ys[1:-1]))
    for t in (y, ys):
        assert (t[0] == 7).all() and (t[-1] == 7).all()
    ids = torch.argsort(-z, dim=1, stable=True)[:, :top]
    _close(y[1:-1], torch.stack([h[t].double() @ w[ids[t, c]].double().t() for t in range(tokens) for c in range(top)]), dtype)
    _close(ys[1:-1], h.double() @ ws.double().t(), dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("n,k", [(4096, 64), (4096, 128), (4096, 192), (2048, 320), (4096, 640), (4096, 1088), (10816, 1536), (2048, 4096)])
def test_sums_of_the_stream_are_as_exact(n, k, dtype):
    """Against those of the kernel without a stream (operands that start between two 16-byte boundaries go there), which adds up eighths of K: chains as short or
    shorter.  The mean over 64 n values is known to 3 / sqrt(128 n) of itself, 0.6 % at 2048 channels: 2 % for two of them."""
    ops, m = _ops(dtype), 64
    shift = 8 // torch.empty((), dtype=dtype).element_size()
    buf = _randn(46, dtype, m * k + 16)
    w = _randn(47, dtype, n, k) * k ** -0.5
    inside = buf[shift:shift + m * k].view(m, k)
    x = inside.clone()
    want = x.double() @ w.double().t()
    assert _rows_plan(ops, 1, n, k, m)[0] > 0 and x.data_ptr() % 16 == 0 and inside.data_ptr() % 16 == 8
    stream, plain = ((ops.matmul(a, w, out_f32=True).double() - want).norm().item() for a in (x, inside))
    assert 0 < stream < 1.02 * plain, (stream / want.norm().item(), plain / want.norm().item())


# experts of a router (16 channels a workgroup), heads of 80 and of 128 channels a workgroup, in K parts and in slices
@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("m,n,k", [(1, 256, 2048), (16, 512, 2048), (48, 512, 1024), (3, 4096, 4096), (5, 16448, 2048), (48, 32000, 4096), (1, 32768, 2048)])
def test_equal_channels_have_equal_sums(m, n, k, dtype):
    """A channel's sum does not hang on its place: experts or words with the same weights are as likely as each other."""
    ops = _ops(dtype)
    x, w = _randn(41, dtype, m, k), _randn(42, dtype, 32, k).repeat(n // 32, 1)
    y = ops.matmul(x, w, out_f32=True).view(m, n // 32, 32)
    assert torch.equal(y, y[:, :1].expand_as(y))


def test_equal_channels_have_equal_gated_units():
    """... nor does a gated unit of 128 channels a workgroup"""
    ops, m, n, k = _ops(torch.bfloat16), 48, 28672, 4096
    assert _rows_plan(ops, 1, n, k, m, 2) == (128, 1)
    y = ops.glu(_randn(43, torch.bfloat16, m, k), _randn(44, torch.bfloat16, 32, k).repeat(n // 32, 1), None, "silu").view(m, n // 32, 16)
    assert torch.equal(y, y[:, :1].expand_as(y))


@pytest.mark.parametrize("epi,n,k,m,narrow", [(0, 43536, 4096, 1, (80, 4)), (0, 28688, 8192, 1, (80, 2)), (0, 11136, 14336, 49, (48, 1)), (0, 16384, 28672, 64, (64, 1)),
                                               (2, 34848, 4096, 1, (64, 4)), (2, 57376, 4096, 1, (64, 8))])
def test_128_channels_keep_the_order_of_sums(epi, n, k, m, narrow):
    """Workgroups of 128 channels take K in one chain of stages: they stand in for narrower ones that do, too, not for those with K slices or K parts."""
    assert _rows_plan(_ops(torch.bfloat16), 1, n, k, m, epi) == narrow


@pytest.mark.parametrize("m,n,k", [(128, 32, 64), (1000, 14336, 2048), (2000, 6144, 2048), (300, 1024, 512)])
def test_gated_unit_of_many_rows_has_the_bits_of_product_and_unit(m, n, k):
    """Gate and up of more than 64 rows are the product's rows, rounded to the element type, whatever the number of rows."""
    ops = _ops(torch.bfloat16)
    x, w, b = _randn(61, torch.bfloat16, m, k), _randn(62, torch.bfloat16, 2 * n, k) * k ** -0.5, _randn(63, torch.float32, 2 * n)
    y, want = ops.matmul(x, w), torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    ops._call("lm_glu", want.data_ptr(), n, y.data_ptr(), 2 * n, b.data_ptr(), m, n, 1)
    assert torch.equal(ops.glu(x, w, b, "silu"), want)


@pytest.mark.parametrize("m,n,k,plan", [(1, 28672, 4096, (128, 1)), (3, 20512, 2048, (128, 1)), (64, 24576, 4096, (128, 1)), (1, 16416, 1024, (128, 1)), (2, 10240, 4096, (64, 1)), (16, 5120, 2048, (64, 2))])
def test_gated_unit_of_few_rows_in_wide_workgroups(m, n, k, plan):
    """... of 64 channels in one round, of 128 where those are more; slices where they leave units idle"""
    ops = _ops(torch.bfloat16)
    assert _rows_plan(ops, 1, n, k, m, 2) == plan
    x, w, b = _randn(71, torch.bfloat16, m, k), _randn(72, torch.bfloat16, n, k) * k ** -0.5, _randn(73, torch.float32, n) * 0.1
    y = (x.double() @ w.double().t() + b.double()).view(m, n // 32, 2, 16)
    want = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(m, n // 2)
    assert errors(ops.glu(x, w, b, "silu").float().cpu().numpy(), want.cpu().numpy()).max() < TOL[torch.bfloat16]
