"""Prompts' products whose last round's tiles share out their K (csrc/tile_share.h): one tile of an XCD and many, two parts of a tile and many, with and without whole
rounds in front, parts of the fewest stages, row tiles that share rows.  Against the same product with whole tiles: the same bits, whatever the scratch holds, launch after launch, and the
scratch shows which of them it was."""
import pytest
import torch

from tests.test_cabi_cpu import _parts
from tests.test_silu_rows_gpu import CHN, GRP, W8, _case

pytestmark = pytest.mark.gpu
DEV = "cuda"
#        mode, rows, N, K                         tiles of an XCD's last round (of 32), parts
SIZES = [(GRP, 2331, 4096, 14336), (W8, 2100, 4096, 14336),           # 20, 18, two and three
         (GRP, 2791, 6144, 8192), (W8, 2791, 6144, 8192),             # 1 behind a round, five: the most
         (W8, 2133, 8192, 28672), (GRP, 4200, 4096, 14336),           # 4 and 2 behind a whole round
         (GRP, 6000, 4096, 14336), (W8, 6000, 4096, 14336),           # 16 behind one: two
         (GRP, 3165, 4096, 14336), (W8, 3000, 4096, 28672),           # 26, 24: one workgroup has the ends of several tiles
         (GRP, 1570, 5120, 13824), (W8, 653, 4096, 14336),            # 18 (some XCDs 17), 6
         (W8, 513, 4608, 12800), (CHN, 1025, 7680, 16384),            # 7 and 6, 19 and 18; parts of four stages, as in 1570 rows above
         (CHN, 2830, 4096, 28672), (CHN, 2140, 8192, 28672)]          # 24; 4 behind a whole round
UNIT = [(CHN, 2600, 16384, 16384), (GRP, 2331, 28672, 4096), (GRP, 1500, 16384, 8192), (W8, 2100, 16384, 16384),
        (W8, 513, 26624, 8192), (CHN, 1025, 10240, 16384)]           # parts of four stages, as in 2331 rows


def _left(M, N, K):
    """Tiles of each XCD's last round that are shared out"""
    from omniserve_amd import _lib
    tiles = (M + 255) // 256 * (N // 256)
    return [len({p[1] for p in _parts(_lib.lib(), tiles // 8 + (x < tiles % 8), K // 128) if p[4] >= 0}) for x in range(8)]


def _shared(scratch, M, N, K):
    """Has a launch with shared tiles been over these bytes of 255?  Sums lie in them, and every shared tile's mark is 0 again"""
    marks, left = scratch[-2048:].view(torch.int64).view(8, 32).cpu(), _left(M, N, K)
    assert any(left)
    return bool((scratch[:-2048] != 255).any()) and all((marks[x, :n] == 0).all() and (marks[x, n:] == -1).all() for x, n in enumerate(left))


def _calls(mode, M, N, K, unit):
    from omniserve_amd import _lib
    h, (x, w, ops) = _lib.lib(), _case(M, N, K, mode)
    need = h.omni_gemm_share_bytes(M, N, K, mode)
    fn = {(CHN, False): h.omni_w4a8_per_chn_gemm, (CHN, True): h.omni_w4a8_per_chn_gemm_silu_rows, (GRP, False): h.omni_w4a8_per_group_gemm, (W8, False): h.omni_w8a8_gemm, (GRP, True): h.omni_w4a8_per_group_gemm_silu_rows, (W8, True): h.omni_w8a8_gemm_silu_rows}[mode, unit]
    ws = torch.empty((max(h.omni_gemm_workspace_bytes(M, N, K), 1),), dtype=torch.uint8, device=DEV)

    def call(out, scratch=None):
        if scratch is not None:
            assert h.omni_gemm_arm_share(scratch.data_ptr(), scratch.numel()) == 0
        a = [t.data_ptr() for t in (x, w) + ops] + [out.data_ptr(), M, N, K]
        a += [] if unit else [N, ws.data_ptr(), ws.numel()]
        assert fn(*a, _lib.current_stream()) == 0
        return out
    n = N // 2 if unit else N
    return need, call, lambda: torch.full((M, n), 7.0, dtype=torch.half, device=DEV), (x, w, ops, ws)


@pytest.mark.parametrize("mode,M,N,K,unit", [s + (False,) for s in SIZES] + [s + (True,) for s in UNIT])
def test_parts_add_up_to_the_whole(mode, M, N, K, unit):
    need, call, out, keep = _calls(mode, M, N, K, unit)
    assert need > 0
    want = call(out())
    assert torch.isfinite(want).all() and want.abs().sum() > 0
    room = torch.randint(0, 256, (need + 4096,), dtype=torch.uint8, device=DEV)
    scratch, behind = room[:need], room[need:].clone()
    for fill in (None, 0, 255, None):      # what was there, and what the launch before left
        if fill is not None:
            scratch.fill_(fill)
        assert torch.equal(call(out(), scratch), want)
        assert fill != 255 or _shared(scratch, M, N, K)
    assert torch.equal(room[need:], behind)
    scratch.fill_(7)
    assert torch.equal(call(out()), want) and (scratch == 7).all()      # one launch an arming
    assert torch.equal(call(out(), scratch[:-16]), want) and (scratch == 7).all()      # too few bytes: whole tiles


def test_captured_launches_run_again():
    need, call, out, keep = _calls(GRP, 2331, 4096, 14336, False)
    want, got, scratch = call(out()), out(), torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    call(got, scratch)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call(got, scratch)
        call(got, scratch)
    for _ in range(4):
        got.fill_(7)
        scratch.fill_(255)
        g.replay()
        assert torch.equal(got, want) and _shared(scratch, 2331, 4096, 14336)
        assert torch.equal(call(out(), scratch), want)


def test_mirror_takes_them_on_two_streams():
    """The functions that allocate the scratch themselves, side by side"""
    from omniserve_amd import _lib
    from omniserve_amd.backend import qgemm_w4a8_per_group
    assert _lib.fast() is not None      # (the functions in Python alone take whole tiles)
    need, call, out, (x, w, ops, ws) = _calls(GRP, 2331, 4096, 14336, False)
    want, streams, got = call(out()), [torch.cuda.Stream(), torch.cuda.Stream()], [[out() for _ in range(6)] for _ in range(2)]
    torch.cuda.synchronize()
    for i in range(6):
        for s, o in zip(streams, got):
            with torch.cuda.stream(s):
                qgemm_w4a8_per_group.gemm_forward_cuda(x, w, *ops, o[i])
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for os in got for o in os)


@pytest.mark.parametrize("mode,M,N,K,unit", [(GRP, 2331, 4096, 14336, False), (W8, 2100, 4096, 14336, False), (CHN, 1025, 7680, 16384, False),
                                             (GRP, 2331, 28672, 4096, True), (W8, 513, 26624, 8192, True), (CHN, 1025, 10240, 16384, True)])
@pytest.mark.parametrize("native", [True, False])
def test_mirror_arms_its_scratch(mode, M, N, K, unit, native, monkeypatch):
    """... where the compiled binding is there: the block that the caching allocator gives it is the one freed in front of the call.  The functions in Python alone take whole tiles"""
    from omniserve_amd import _lib
    from omniserve_amd.backend import fused_ext, qgemm_w4a8_per_chn, qgemm_w4a8_per_group, qgemm_w8a8
    assert _lib.fast() is not None
    if not native:
        monkeypatch.setattr(_lib, "USE_EXT", False)
    need, call, out, (x, w, ops, ws) = _calls(mode, M, N, K, False)
    product = (qgemm_w4a8_per_chn.gemm_forward_cuda, qgemm_w4a8_per_group.gemm_forward_cuda, qgemm_w8a8.w8a8_gemm_forward_cuda)[mode]
    got, codes, scale, sums = out(), torch.empty((M, N // 2), dtype=torch.int8, device=DEV), torch.empty((M,), dtype=torch.half, device=DEV), torch.empty((M,), dtype=torch.half, device=DEV)
    run = (lambda: fused_ext.gate_up_rows(codes, x, w, ops, got, sums if mode == CHN else None, scale)) if unit else (lambda: product(x, w, *ops, got))
    run()
    torch.cuda.empty_cache()
    scratch = torch.full((need,), 255, dtype=torch.uint8, device=DEV)
    place = scratch.data_ptr()
    del scratch
    run()
    scratch = torch.empty((need,), dtype=torch.uint8, device=DEV)
    assert scratch.data_ptr() == place
    assert _shared(scratch, M, N, K) if native else (scratch == 255).all()


@pytest.mark.parametrize("unit", [False, True])
def test_mirror_without_room_for_scratch(unit):
    """A device filled up to a few megabytes, as its pages of keys and values may leave it: whole tiles, and no error"""
    from omniserve_amd import _lib
    from omniserve_amd.backend import fused_ext, qgemm_w4a8_per_group
    assert _lib.fast() is not None
    M, N, K = UNIT[1][1:] if unit else (2331, 4096, 14336)
    need, call, out, (x, w, ops, ws) = _calls(GRP, M, N, K, False)
    got, want = out(), call(out())
    codes, scale = [torch.empty((M, N // 2), dtype=torch.int8, device=DEV) for _ in range(2)], [torch.empty((M,), dtype=torch.half, device=DEV) for _ in range(2)]
    run = (lambda i: fused_ext.gate_up_rows(codes[i], x, w, ops, got, None, scale[i])) if unit else (lambda i: qgemm_w4a8_per_group.gemm_forward_cuda(x, w, *ops, got))
    run(0)
    assert need > 32 << 20
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (24 << 20)) / torch.cuda.get_device_properties(0).total_memory)
    try:
        full = []
        with pytest.raises(torch.cuda.OutOfMemoryError):
            while len(full) < 64:      # (what is cached beside tensors of other tests)
                full.append(torch.empty((need,), dtype=torch.uint8, device=DEV))
        got.fill_(7)
        run(1)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    if unit:
        assert torch.equal(*codes) and torch.equal(*scale) and codes[0].any()
    else:
        assert torch.equal(got, want)


def test_what_is_refused():
    from omniserve_amd import _lib
    h = _lib.lib()
    t = torch.empty((1 << 20,), dtype=torch.uint8, device=DEV)
    assert h.omni_gemm_arm_share(t.data_ptr(), t.numel()) != 0 and h.omni_gemm_arm_share(None, 0) == 0
    for M, N, K, mode in ((2331, 4096, 14336, 3), (255, 4096, 14336, 1), (4000, 4096, 14336, 1), (2331, 4096, 512, 1), (2331, 4100, 14336, 2), (0, 0, 0, 1)):
        assert h.omni_gemm_share_bytes(M, N, K, mode) == 0
