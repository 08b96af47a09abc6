"""Parity of the HIP W4A8 / W8A8 GEMMs against the oracle: bit-exact fp16 outputs
(int32 accumulators exact, epilogue evaluated in the same fp32 order)."""
import numpy as np
import pytest
import torch

from oracle import w4a8
from tests.util import assert_f16_equal, dev, quantize_act, to_dev

pytestmark = pytest.mark.gpu


def _acts(M, K, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((M, K)).astype(np.float16)
    return quantize_act(x)


def _run_chn(M, N, K, seed=0, out_view=False):
    import omniserve_backend.qgemm_w4a8_per_chn as mod
    u, z, s1 = w4a8.synth_per_channel(N, K, seed)
    qw, s1h, szh = w4a8.pack_per_channel(u, z, s1)
    a, sa, asum = _acts(M, K, seed + 1)
    want = w4a8.gemm_per_chn(a, qw, s1h, sa, szh, asum)
    if out_view == "cols":  # rows that start 8 bytes into a wider buffer (row stride not a multiple of 16 bytes: the 8-byte store forms)
        buf = torch.full((M, N + 4), 7.0, dtype=torch.float16, device=dev())
        out = buf[:, 4:]
    elif out_view:  # pre-allocated larger buffer, row-slice view (llama_w4a8_unpad.py:356-361)
        buf = torch.full((M + 3, N), 7.0, dtype=torch.float16, device=dev())
        out = buf[1:M + 1]
    else:
        out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.gemm_forward_cuda(to_dev(a), to_dev(qw), to_dev(s1h), to_dev(sa), to_dev(szh), to_dev(asum), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "per_chn M=%d N=%d K=%d" % (M, N, K))
    if out_view == "cols":
        assert (buf[:, :4] == 7).all()
    elif out_view:
        assert (buf[0] == 7).all() and (buf[M + 1:] == 7).all()


@pytest.mark.parametrize("M", [1, 7, 16, 17, 33, 64, 100, 128])
@pytest.mark.parametrize("N,K", [(64, 64), (256, 256), (320, 448), (192, 1024)])
def test_per_chn_decode_shapes(M, N, K):
    _run_chn(M, N, K, seed=M + N + K)


@pytest.mark.parametrize("M,N,K", [(129, 256, 256), (300, 320, 192), (1000, 512, 1024), (257, 64, 64),
                                   (2100, 2304, 128)])   # last: 17 x 9 tiles = several 8 x 8 super-blocks (XCD order)
def test_per_chn_prefill_shapes(M, N, K):
    _run_chn(M, N, K, seed=M)


# Decode at batch 129 .. 512 (the reference's published A100 figure is quoted at bs = 256): few 128 x 256 tiles, so the plan
# offers K slices over grid.y into int32 slabs + the slab epilogue (qgemm_plan.hip: down_proj 8 ways, o_proj / qkv 4 ways at
# bs = 256; gate_up has 224 tiles and stays whole), with scratch for them; whether they run is plan_prefill's choice (forced, with
# the tile heights: test_prefill_forms).  Ragged M (row tiles partly filled), all three flavours.
FEW_TILE_SHAPES = [(256, 4096, 14336), (256, 6144, 4096), (256, 4096, 4096), (129, 4096, 14336), (300, 512, 2048), (512, 4096, 4096)]


@pytest.mark.parametrize("M,N,K", FEW_TILE_SHAPES)
def test_per_chn_few_tiles_split_k(M, N, K):
    import ctypes
    from omniserve_amd import _lib
    sk = ctypes.c_int(0)
    _lib.lib().omni_gemm_get_plan(M, N, K, 64, None, None, ctypes.byref(sk))
    assert sk.value > 1 and _lib.lib().omni_gemm_workspace_bytes(M, N, K) >= sk.value * M * N * 4
    _run_chn(M, N, K, seed=M + N)


@pytest.mark.parametrize("M,N,K", [(256, 4096, 14336), (256, 4096, 4096), (384, 512, 2048), (300, 512, 2048)])
def test_per_chn_partial_few_tiles(M, N, K):
    """The slab-only form (fused_ext.gemm_partial_per_chn: o_proj / down_proj of the decode drivers at batch 129 .. 512): the
    sum of the int32 slabs is the exact accumulator."""
    from omniserve_amd.backend import fused_ext
    u, z, s1 = w4a8.synth_per_channel(N, K, M)
    qw, _, _ = w4a8.pack_per_channel(u, z, s1)
    a, _, _ = _acts(M, K, M + 1)
    slab = torch.zeros((8, M, N), dtype=torch.int32, device=dev())
    sk = fused_ext.gemm_partial_per_chn(to_dev(a), to_dev(qw), slab)
    torch.cuda.synchronize()
    assert sk > 1 and not slab[sk:].any()
    assert np.array_equal(slab[:sk].sum(dim=0).cpu().numpy(), w4a8.gemm_per_chn_acc(a, qw))


@pytest.mark.parametrize("M,N,K", FEW_TILE_SHAPES[:3] + FEW_TILE_SHAPES[4:5])
def test_per_group_few_tiles_split_k(M, N, K):
    _run_grp(M, N, K, False)


@pytest.mark.parametrize("M,N,K", FEW_TILE_SHAPES[1:3] + FEW_TILE_SHAPES[4:5])
def test_w8a8_few_tiles_split_k(M, N, K):
    _run_w8(M, N, K)


@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336)])
def test_per_chn_llama3_8b_decode_bs16(N, K):
    _run_chn(16, N, K, seed=1)


def test_per_chn_output_row_slice_view():
    _run_chn(16, 256, 512, seed=9, out_view=True)


def test_per_chn_config1_4096_cubed():
    _run_chn(4096, 4096, 4096, seed=0)


@pytest.mark.parametrize("waves,sk", [(1, 1), (1, 4), (4, 1), (4, 2), (4, 8)])
def test_per_chn_plan_overrides(waves, sk):
    from omniserve_amd import _lib
    _lib.lib().omni_gemm_set_plan_override(waves, sk)
    try:
        _run_chn(16, 512, 2048, seed=waves * 10 + sk)
        _run_chn(32, 512, 2048, seed=waves * 10 + sk + 1)
    finally:
        _lib.lib().omni_gemm_set_plan_override(0, 0)


def _run_grp(M, N, K, wrap, seed=None):
    import omniserve_backend.qgemm_w4a8_per_group as mod
    u, z, s2, s1 = w4a8.synth_per_group(N, K, seed=M + K if seed is None else seed, wrap=wrap)
    qw, s1h, s2s, s2z = w4a8.pack_per_group(u, z, s2, s1)
    a, sa, _ = _acts(M, K, M + 2)
    want = w4a8.gemm_per_group(a, qw, s2z, s2s, s1h, sa)
    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.gemm_forward_cuda(to_dev(a), to_dev(qw), to_dev(s2z), to_dev(s2s), to_dev(s1h), to_dev(sa), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "per_group M=%d N=%d K=%d wrap=%s" % (M, N, K, wrap))


def _run_w8(M, N, K):
    import omniserve_backend.qgemm_w8a8 as mod
    rng = np.random.default_rng(M + N)
    w = rng.integers(-128, 128, size=(N, K), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, size=(N,)).astype(np.float16)
    a, sa, _ = _acts(M, K, M + 3)
    want = w4a8.gemm_w8a8(a, w, sw, sa)
    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.w8a8_gemm_forward_cuda(to_dev(a), to_dev(w), to_dev(sw), to_dev(sa), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "w8a8 M=%d N=%d K=%d" % (M, N, K))


# ---- every M regime of the tile dispatch has an oracle case (the reference's: w4a8_per_group/gemm_cuda.cu:659-705) ----
# Prefill kernel (M > 128), K >= 3 whole 256-k chunks: the branch-free STEADY loop of w4a8_gemm_kernel (two-step weight
# ring refills, next-chunk group parameters, in-chunk activation publishing) with full and ragged M tiles and a ragged
# N tile (N = 320: five 64-channel groups = 1.25 workgroup tiles).
@pytest.mark.parametrize("wrap", [False, True])
@pytest.mark.parametrize("M,N,K", [(300, 256, 1024), (1000, 512, 1024), (256, 320, 2048), (1000, 512, 4096)])
def test_per_group_prefill_steady_loop(M, N, K, wrap):
    _run_grp(M, N, K, wrap)


@pytest.mark.parametrize("M,N,K", [(300, 256, 1024), (1000, 512, 1024), (256, 320, 2048), (1000, 512, 4096)])
def test_w8a8_prefill_steady_loop(M, N, K):
    _run_w8(M, N, K)


@pytest.mark.parametrize("M,N,K", [(1000, 512, 1024), (300, 320, 2304)])
def test_per_chn_prefill_steady_loop_ragged(M, N, K):
    _run_chn(M, N, K, seed=M + K)


def test_per_group_4096_cubed():
    _run_grp(4096, 4096, 4096, False)


def test_w8a8_4096_cubed():
    _run_w8(4096, 4096, 4096)


# Exact-shape prefill kernel (csrc/qgemm_exact.h: M % 128 == N % 256 == K % 256 == 0; activations by LDS-DMA into the swizzled
# row image, lane transpose of the packed int4 registers, last chunk without prefetch, packed 16-B stores) against the oracle:
# one tile x one chunk (no steady loop: prologue -> last chunk), two chunks (one steady iteration), several tiles in both
# directions incl. a partly filled 8 x 8 super-block, a long K, and the per-group wrap set (byte products above 255).
EXACT_SHAPES = [(128, 256, 256), (256, 512, 512), (384, 256, 1024), (128, 768, 2048), (1152, 2304, 256), (640, 512, 4096)]


@pytest.mark.parametrize("M,N,K", EXACT_SHAPES)
def test_per_chn_exact_shapes(M, N, K):
    _run_chn(M, N, K, seed=M + N + K)


@pytest.mark.parametrize("wrap", [False, True])
@pytest.mark.parametrize("M,N,K", EXACT_SHAPES)
def test_per_group_exact_shapes(M, N, K, wrap):
    _run_grp(M, N, K, wrap)


@pytest.mark.parametrize("M,N,K", EXACT_SHAPES)
def test_w8a8_exact_shapes(M, N, K):
    _run_w8(M, N, K)


# Llama-2-70B TP=8 shard shapes (bs up to 128): qkv (64+16)/8 heads x 128 = 1280 x 8192,
# o 8192 x 1024, gate_up 2 x 28672/8 = 7168 x 8192, down 8192 x 3584 -- the M = 65..128 decode tile with split-K slabs.
LLAMA2_70B_TP8 = [(1280, 8192), (8192, 1024), (7168, 8192), (8192, 3584)]


@pytest.mark.parametrize("M", [65, 100, 128])
@pytest.mark.parametrize("N,K", LLAMA2_70B_TP8)
def test_per_chn_llama2_70b_tp8_shard(M, N, K):
    _run_chn(M, N, K, seed=M + N)


@pytest.mark.parametrize("M", [65, 128])
@pytest.mark.parametrize("N,K", LLAMA2_70B_TP8)
def test_per_group_llama2_70b_tp8_shard(M, N, K):
    _run_grp(M, N, K, False)


# BASELINE.json configs[2] (g128, bs = 64) and the LServe W8A8 decode shapes at M = 64, Llama-3-8B projections
@pytest.mark.parametrize("N,K", [(6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336)])
def test_per_group_llama3_8b_decode_bs64(N, K):
    _run_grp(64, N, K, False)


@pytest.mark.parametrize("M,N,K", [(64, 28672, 4096), (64, 4096, 14336), (1, 6144, 4096), (1, 28672, 4096)])
def test_w8a8_llama3_8b_decode(M, N, K):
    _run_w8(M, N, K)


@pytest.mark.parametrize("M", [17, 32, 48, 64])
def test_per_chn_llama3_8b_gate_up_mid_batches(M):
    _run_chn(M, 28672, 4096, seed=M)


@pytest.mark.parametrize("wrap", [False, True])
@pytest.mark.parametrize("M,N,K", [(16, 256, 512), (64, 320, 1024), (5, 64, 128), (200, 256, 384), (16, 4096, 4096)])
def test_per_group(M, N, K, wrap):
    import omniserve_backend.qgemm_w4a8_per_group as mod
    u, z, s2, s1 = w4a8.synth_per_group(N, K, seed=M + K, wrap=wrap)
    qw, s1h, s2s, s2z = w4a8.pack_per_group(u, z, s2, s1)
    a, sa, _ = _acts(M, K, M + 2)
    want = w4a8.gemm_per_group(a, qw, s2z, s2s, s1h, sa)
    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.gemm_forward_cuda(to_dev(a), to_dev(qw), to_dev(s2z), to_dev(s2s), to_dev(s1h), to_dev(sa), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "per_group M=%d N=%d K=%d wrap=%s" % (M, N, K, wrap))


@pytest.mark.parametrize("M,N,K", [(16, 256, 512), (64, 320, 1024), (3, 64, 64), (200, 256, 320), (16, 4096, 4096)])
def test_w8a8(M, N, K):
    import omniserve_backend.qgemm_w8a8 as mod
    rng = np.random.default_rng(M + N)
    w = rng.integers(-128, 128, size=(N, K), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, size=(N,)).astype(np.float16)
    a, sa, _ = _acts(M, K, M + 3)
    want = w4a8.gemm_w8a8(a, w, sw, sa)
    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.w8a8_gemm_forward_cuda(to_dev(a), to_dev(w), to_dev(sw), to_dev(sa), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "w8a8 M=%d N=%d K=%d" % (M, N, K))


def test_gemm_linearity_full_size():
    """Size-independent property at the BASELINE size: with ascales=1, asum=0 and wscales=2^-k the
    epilogue is exact, so acc(A1) + acc(A2) == acc(A1 + A2) can be checked through the fp16
    outputs (values kept below 2048 so fp16 holds them exactly)."""
    import omniserve_backend.qgemm_w4a8_per_chn as mod
    M, N, K = 16, 4096, 4096
    rng = np.random.default_rng(5)
    u = rng.integers(0, 2, size=(N, K), dtype=np.uint8)           # codes 0/1
    qw = to_dev(w4a8.pack_w4(u))
    a1 = rng.integers(-1, 2, size=(M, K), dtype=np.int8)
    a2 = rng.integers(-1, 2, size=(M, K), dtype=np.int8)
    ones_n = to_dev(np.ones(N, np.float16)); zeros_n = to_dev(np.zeros(N, np.float16))
    ones_m = to_dev(np.ones(M, np.float16)); zeros_m = to_dev(np.zeros(M, np.float16))
    outs = []
    for a in (a1, a2, (a1 + a2).astype(np.int8)):
        o = torch.empty((M, N), dtype=torch.float16, device=dev())
        mod.gemm_forward_cuda(to_dev(a), qw, ones_n, ones_m, zeros_n, zeros_m, o)
        outs.append(o.float())
    torch.cuda.synchronize()
    assert torch.equal(outs[0] + outs[1], outs[2])
    assert outs[2].abs().max() < 2048


# ---- mid-M kernel (csrc/qgemm_midm.h): forced on through omni_gemm_set_midm_override so that every row-tile height, ragged M,
# short slices (fewer chunks than ring slots), forced K splits and all three flavours meet the oracle -- the planner itself
# only sends it the big matrices (test_midm_planner_takes_the_big_matrices) ----
class _ForcedMidm:
    def __init__(self, sk=0):
        self.sk = sk

    def __enter__(self):
        from omniserve_amd import _lib
        from omniserve_amd.backend import _gemm_common
        _lib.lib().omni_gemm_set_midm_override(1, self.sk)
        _gemm_common._ws_bytes.clear()
        self.keep_ext, _lib.USE_EXT = _lib.USE_EXT, False      # (the fast binding caches scratch sizes per shape as well)

    def __exit__(self, *exc):
        from omniserve_amd import _lib
        from omniserve_amd.backend import _gemm_common
        _lib.lib().omni_gemm_set_midm_override(-1, 0)
        _gemm_common._ws_bytes.clear()
        _lib.USE_EXT = self.keep_ext


MIDM_SMALL = [(33, 128, 256, 0), (64, 256, 512, 0), (65, 128, 1024, 0), (100, 384, 2048, 2), (128, 256, 4096, 4), (48, 128, 768, 0),
              (127, 256, 1280, 0), (64, 128, 2048, 8), (128, 128, 256, 0), (96, 640, 1536, 2)]


@pytest.mark.parametrize("M,N,K,sk", MIDM_SMALL)
def test_midm_forced_per_chn(M, N, K, sk):
    with _ForcedMidm(sk):
        _run_chn(M, N, K, seed=M + K)
        _run_chn(M, N, K, seed=M + K + 1, out_view=True)
        _run_chn(M, N, K, seed=M + K + 2, out_view="cols")


@pytest.mark.parametrize("wrap", [False, True])
@pytest.mark.parametrize("M,N,K,sk", MIDM_SMALL)
def test_midm_forced_per_group(M, N, K, sk, wrap):
    with _ForcedMidm(sk):
        _run_grp(M, N, K, wrap)


@pytest.mark.parametrize("M,N,K,sk", MIDM_SMALL)
def test_midm_forced_w8a8(M, N, K, sk):
    with _ForcedMidm(sk):
        _run_w8(M, N, K)


@pytest.mark.parametrize("M,N,K", [(128, 28672, 4096), (64, 28672, 4096), (128, 4096, 14336), (100, 7168, 8192), (128, 8192, 3584)])
def test_midm_forced_model_shapes(M, N, K):
    with _ForcedMidm():
        _run_chn(M, N, K, seed=N)
        _run_grp(M, N, K, wrap=True)


@pytest.mark.parametrize("M,N,K,sk", [(128, 4096, 14336, 0), (64, 512, 2048, 2), (100, 256, 1024, 1), (128, 8192, 8192, 4)])
def test_midm_forced_partial_slabs(M, N, K, sk):
    """The slab-only forms (o_proj / down_proj of the decode drivers at fusion level 2): the slabs sum to the exact accumulator."""
    from omniserve_amd.backend import fused_ext
    u, z, s1 = w4a8.synth_per_channel(N, K, M)
    qw, _, _ = w4a8.pack_per_channel(u, z, s1)
    a, _, _ = _acts(M, K, M + 1)
    slab = torch.zeros((16, M, N), dtype=torch.int32, device=dev())
    with _ForcedMidm(sk):
        got = fused_ext.gemm_partial_per_chn(to_dev(a), to_dev(qw), slab)
        torch.cuda.synchronize()
    assert got >= 1 and (sk == 0 or got == sk) and not slab[got:].any()
    assert np.array_equal(slab[:got].sum(dim=0).cpu().numpy(), w4a8.gemm_per_chn_acc(a, qw))


def test_midm_planner_takes_the_big_matrices():
    """Unforced: Llama-3-8B gate_up at 64 / 128 rows and the Llama-2-70B projections go to the mid-M kernel (plan: 8 waves per
    workgroup reported as 2 channel groups), Llama-3-8B qkv / o and the TP = 8 shards stay on the single-wave tiles."""
    import ctypes
    from omniserve_amd import _lib
    lib = _lib.lib()

    def waves(M, N, K):
        w = ctypes.c_int(0)
        lib.omni_gemm_get_plan(M, N, K, 64, None, ctypes.byref(w), None)
        return w.value
    for M, N, K in [(128, 28672, 4096), (64, 28672, 4096), (128, 57344, 8192), (128, 8192, 28672), (65, 10240, 8192)]:
        assert waves(M, N, K) == 2, (M, N, K)
    for M, N, K in [(128, 6144, 4096), (128, 4096, 4096), (128, 1280, 8192), (16, 28672, 4096), (32, 28672, 4096), (128, 8192, 1024)]:
        assert waves(M, N, K) == 1, (M, N, K)
    _run_chn(128, 28672, 4096, seed=5)
    _run_chn(64, 28672, 4096, seed=6)


# The straight-line prefill kernel at row counts that are not whole tiles: its last row tile starts at M - 128 and shares rows with the
# tile before it (127 shared rows at M = 129, one at 255), on both tile orders (fewer than 8 row tiles, and super-blocks), one K chunk
# and several, and a destination of which the rows around the output stay untouched.
@pytest.mark.parametrize("M,N,K", [(129, 256, 256), (255, 512, 768), (257, 256, 512), (1101, 512, 256), (1501, 1024, 1024)])
@pytest.mark.parametrize("mode", ["chn", "grp", "w8"])
def test_prefill_rows_not_whole_tiles(mode, M, N, K):
    if mode == "chn":
        _run_chn(M, N, K, seed=M, out_view=True)
    elif mode == "grp":
        _run_grp(M, N, K, True)
    else:
        _run_w8(M, N, K)


# Its tile heights (4 .. 8 blocks of 16 rows) and its two forms (K whole, K in two parts that meet in LDS): the sizes at which
# plan_prefill's model picks each of them.
@pytest.mark.parametrize("M,N,K", [(129, 256, 256), (513, 8192, 256), (700, 16384, 256), (333, 16384, 256), (449, 16384, 256), (129, 256, 2048),
                                   (513, 8192, 2048), (333, 16384, 2048), (385, 16384, 2048), (449, 16384, 2048), (225, 28672, 4096), (161, 28672, 4096), (385, 16384, 4096)])
@pytest.mark.parametrize("mode", ["chn", "grp", "w8"])
def test_prefill_tile_heights(mode, M, N, K):
    {"chn": lambda: _run_chn(M, N, K, seed=M), "grp": lambda: _run_grp(M, N, K, False), "w8": lambda: _run_w8(M, N, K)}[mode]()


# W8A8 in 256 x 256 tiles (sizes at which plan_prefill's model picks them): one tile per workgroup and more, 8 .. 32 stages of K, last row
# tiles of 1 row to all of them.
@pytest.mark.parametrize("M,N,K", [(512, 18944, 1536), (768, 13312, 1536), (1281, 7936, 2048), (1537, 6656, 2048), (1024, 10240, 2048), (2017, 13824, 1024),
                                   (333, 28672, 4096)])
def test_w8a8_whole_tiles(M, N, K):
    _run_w8(M, N, K)


# Per-group weights whose second level is unpacked in 16-bit lanes (scales up to 17) in some chunks and in whole words (a scale above 17) in
# others: the edge between the two forms.  (Tiles of 64 rows whole and with K slices over the grid, 96 rows; 128 rows, which have the second
# form only.  K in two parts inside a workgroup: test_per_group_scales_around_the_lane_limit_two_k_parts.)
@pytest.mark.parametrize("M,N,K", [(140, 512, 1024), (333, 512, 2048), (300, 512, 768), (449, 16384, 256), (700, 16384, 256)])
def test_per_group_scales_around_the_lane_limit(M, N, K):
    import omniserve_backend.qgemm_w4a8_per_group as mod
    u, z, s2, s1 = w4a8.synth_per_group(N, K, seed=M)
    rng = np.random.default_rng(M)
    s2[:] = rng.integers(14, 18, size=s2.shape)            # products up to 255, to within one of the limit
    big = rng.random(s2.shape) < 0.004                     # ... and a few beyond it
    big[N // 2, 1] = big[N - 1, -1] = True
    s2[big] = rng.integers(18, 41, size=int(big.sum()))
    u[:, 0] = 15
    qw, s1h, s2s, s2z = w4a8.pack_per_group(u, z, s2, s1)
    a, sa, _ = _acts(M, K, M + 2)
    want = w4a8.gemm_per_group(a, qw, s2z, s2s, s1h, sa)
    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    mod.gemm_forward_cuda(to_dev(a), to_dev(qw), to_dev(s2z), to_dev(s2s), to_dev(s1h), to_dev(sa), out)
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "per_group M=%d N=%d K=%d" % (M, N, K))


def _prefill_plan(mode, M, N, K, slabs_only=False):
    """(rows / 16 of a tile, K parts inside a workgroup, K slices over the grid) of the straight-line kernels; None: the general kernel"""
    import ctypes
    from omniserve_amd import _lib
    mb, kw, sk = (ctypes.c_int(0) for _ in range(3))
    which = _lib.lib().omni_gemm_get_prefill_plan(M, N, K, MODES.index(mode), int(slabs_only), ctypes.byref(mb), ctypes.byref(kw), ctypes.byref(sk))
    assert which in (1, 2)
    return (mb.value, kw.value, sk.value) if which == 1 else None


MODES = ["chn", "grp", "w8"]
# Every instantiation of the straight-line kernels that plan_prefill takes somewhere, with the plan that is to run: whole K, two K parts that
# meet in LDS, K slices over the grid with the slab epilogue.
PREFILL_FORMS = [(m, *f) for m in MODES for f in (
    (4, 1, 1, 129, 256, 256), (5, 1, 1, 324, 12288, 256), (7, 1, 1, 404, 12288, 256), (8, 1, 1, 449, 16384, 256),
    (5, 1, 8, 129, 3072, 8192), (8, 1, 8, 229, 3072, 8192)) if not (m == "w8" and f[0] == 7)] + [
    (m, *f) for m in MODES for f in ((6, 1, 1, 700, 16384, 256), (5, 2, 1, 513, 8192, 2048), (8, 2, 1, 449, 16384, 2048))] + [
    ("chn", 4, 2, 1, 300, 512, 2048), ("chn", 6, 2, 1, 161, 28672, 4096), ("chn", 7, 2, 1, 385, 16384, 4096),
    ("chn", 4, 1, 4, 129, 256, 4096), ("chn", 7, 1, 8, 164, 3072, 8192),
    ("grp", 4, 2, 1, 700, 256, 2048), ("grp", 6, 2, 1, 333, 16384, 2048), ("grp", 7, 2, 1, 385, 16384, 2048),
    ("grp", 4, 1, 2, 300, 512, 2048), ("grp", 6, 1, 8, 164, 6144, 8192), ("grp", 7, 1, 8, 164, 3072, 8192),
    ("w8", 7, 1, 1, 484, 12288, 256), ("w8", 4, 2, 1, 300, 512, 2048), ("w8", 6, 2, 1, 333, 16384, 2048), ("w8", 7, 2, 1, 385, 16384, 2048),
    ("w8", 4, 1, 4, 256, 4096, 4096), ("w8", 6, 1, 8, 164, 3072, 8192), ("w8", 7, 1, 8, 194, 3072, 8192),
    ("w8", 16, 1, 1, 512, 18944, 1536), ("w8", 16, 1, 1, 2369, 17920, 1024)]      # the last: up to three 256 x 256 tiles per workgroup
# ... and of the slab-only calls, which take the K slices as they are
SLAB_FORMS = [(m, *f) for m in MODES for f in ((4, 4, 256, 4096, 4096), (5, 8, 129, 3072, 8192), (8, 8, 229, 3072, 8192), (5, 1, 324, 12288, 256))] + [
    ("chn", 6, 8, 164, 6144, 8192), ("chn", 7, 8, 164, 3072, 8192), ("grp", 6, 8, 164, 6144, 8192), ("grp", 7, 8, 164, 3072, 8192),
    ("w8", 6, 8, 164, 3072, 8192), ("w8", 7, 8, 194, 3072, 8192)]


@pytest.mark.parametrize("mode,mb,kw,sk,M,N,K", PREFILL_FORMS)
def test_prefill_forms(mode, mb, kw, sk, M, N, K):
    assert _prefill_plan(mode, M, N, K) == (mb, kw, sk)
    {"chn": lambda: _run_chn(M, N, K, seed=M, out_view=True), "grp": lambda: _run_grp(M, N, K, True), "w8": lambda: _run_w8(M, N, K)}[mode]()


@pytest.mark.parametrize("mode,mb,sk,M,N,K", SLAB_FORMS)
def test_prefill_slab_forms(mode, mb, sk, M, N, K):
    """Sums of the slabs: the exact accumulators; what lies behind them stays as it was."""
    from omniserve_amd.backend import fused_ext
    assert _prefill_plan(mode, M, N, K, slabs_only=True) == (mb, 1, sk)
    rng = np.random.default_rng(M + N)
    a = rng.integers(-127, 128, size=(M, K), dtype=np.int8)
    if mode == "w8":
        w = rng.integers(-128, 128, size=(N, K), dtype=np.int8)
        call, want = lambda s: fused_ext.gemm_partial_w8a8(to_dev(a), to_dev(w), s), w4a8._int_matmul_fast(a, w)
    elif mode == "chn":
        qw = rng.integers(-128, 128, size=(N, K // 2), dtype=np.int8)
        call, want = lambda s: fused_ext.gemm_partial_per_chn(to_dev(a), to_dev(qw), s), w4a8.gemm_per_chn_acc(a, qw)
    else:
        u, z, s2, s1 = w4a8.synth_per_group(N, K, seed=M, wrap=True)
        qw, _, s2s, s2z = w4a8.pack_per_group(u, z, s2, s1)
        call = lambda s: fused_ext.gemm_partial_per_group(to_dev(a), to_dev(qw), to_dev(s2z), to_dev(s2s), s)      # noqa: E731
        want = w4a8.gemm_per_group_acc(a, qw, s2z, s2s)
    slab = torch.full((sk + 1, M, N), 7, dtype=torch.int32, device=dev())
    assert call(slab) == sk
    torch.cuda.synchronize()
    assert (slab[sk:] == 7).all() and np.array_equal(slab[:sk].sum(dim=0).cpu().numpy(), want)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("M,N,K,sk", [(140, 256, 4096, 2), (255, 256, 2048, 4), (300, 512, 2048, 2), (512, 4096, 4096, 2)])
def test_prefill_forced_k_slices(mode, M, N, K, sk):
    """omni_gemm_set_plan_override's K splits run as they are asked for"""
    from omniserve_amd import _lib
    _lib.lib().omni_gemm_set_plan_override(0, sk)
    try:
        assert _prefill_plan(mode, M, N, K)[1:] == (1, sk)
        {"chn": lambda: _run_chn(M, N, K, seed=M), "grp": lambda: _run_grp(M, N, K, True), "w8": lambda: _run_w8(M, N, K)}[mode]()
    finally:
        _lib.lib().omni_gemm_set_plan_override(0, 0)


@pytest.mark.parametrize("mb,M,N,K", [(4, 700, 256, 2048), (5, 513, 8192, 2048), (6, 333, 16384, 2048), (7, 385, 16384, 2048)])
def test_per_group_scales_around_the_lane_limit_two_k_parts(mb, M, N, K):
    assert _prefill_plan("grp", M, N, K) == (mb, 2, 1)
    test_per_group_scales_around_the_lane_limit(M, N, K)


@pytest.mark.parametrize("M,N,K,mb", [(512, 2304, 256, 4), (505, 4352, 256, 4), (1000, 2304, 768, 4), (1920, 2560, 256, 5)])
@pytest.mark.parametrize("mode", MODES)
def test_prefill_whole_bands(mode, M, N, K, mb):
    """row tiles in whole bands of 8, whose blocks of 8 x 8 tiles end in one or two columns (and in none)"""
    assert _prefill_plan(mode, M, N, K) == (mb, 1, 1) and -(-M // (16 * mb)) % 8 == 0
    {"chn": lambda: _run_chn(M, N, K, seed=M, out_view=True), "grp": lambda: _run_grp(M, N, K, True), "w8": lambda: _run_w8(M, N, K)}[mode]()


def _shifted(a):
    """The same values, contiguous, from 8 bytes behind a 16-byte boundary on"""
    t = torch.from_numpy(np.ascontiguousarray(a)).to(dev())
    base = torch.empty((t.numel() + 16,), dtype=t.dtype, device=dev())
    out = base[8:8 + t.numel()].view(t.shape)
    out.copy_(t)
    assert out.data_ptr() % 16 == 8
    return out


@pytest.mark.parametrize("M,N,K", [(129, 256, 256), (300, 512, 768), (300, 512, 2048), (512, 18944, 1536)])
@pytest.mark.parametrize("mode", MODES)
def test_prefill_operands_between_boundaries(mode, M, N, K):
    """operands that start between two 16-byte boundaries, which the straight-line kernels' DMA does not take"""
    from omniserve_amd.backend import fused_ext, qgemm_w4a8_per_chn, qgemm_w4a8_per_group, qgemm_w8a8
    a, sa, asum = _acts(M, K, M)
    out = torch.empty((M, N), dtype=torch.float16, device=dev())
    if mode == "chn":
        u, z, s1 = w4a8.synth_per_channel(N, K, M)
        qw, s1h, szh = w4a8.pack_per_channel(u, z, s1)
        want = w4a8.gemm_per_chn(a, qw, s1h, sa, szh, asum)
        qgemm_w4a8_per_chn.gemm_forward_cuda(_shifted(a), to_dev(qw), to_dev(s1h), to_dev(sa), to_dev(szh), to_dev(asum), out)
    elif mode == "grp":
        u, z, s2, s1 = w4a8.synth_per_group(N, K, seed=M, wrap=True)
        qw, s1h, s2s, s2z = w4a8.pack_per_group(u, z, s2, s1)
        want = w4a8.gemm_per_group(a, qw, s2z, s2s, s1h, sa)
        qgemm_w4a8_per_group.gemm_forward_cuda(_shifted(a), to_dev(qw), to_dev(s2z), to_dev(s2s), to_dev(s1h), to_dev(sa), out)
    else:
        rng = np.random.default_rng(M)
        w, sw = rng.integers(-128, 128, size=(N, K), dtype=np.int8), rng.uniform(0.001, 0.01, size=(N,)).astype(np.float16)
        want = w4a8.gemm_w8a8(a, w, sw, sa)
        qgemm_w8a8.w8a8_gemm_forward_cuda(_shifted(a), _shifted(w), to_dev(sw), to_dev(sa), out)
        if M <= 300:
            slab = torch.empty((8, M, N), dtype=torch.int32, device=dev())
            sk = fused_ext.gemm_partial_w8a8(_shifted(a), _shifted(w), slab)
            assert np.array_equal(slab[:sk].sum(dim=0).cpu().numpy(), w4a8._int_matmul_fast(a, w))
    torch.cuda.synchronize()
    assert_f16_equal(out, want, "%s M=%d N=%d K=%d" % (mode, M, N, K))
