"""Host logic that chooses the launches of a tiled matmul (no GPU needed): one tile shape,
a K split when the caller brings a workspace, or two regions when the last round of the
main shape would leave most of the chip idle."""
import re

import bench
from modular_amd import _lib


def parse(text):
    parts = [re.match(r"(\d+)x(\d+) x(\d+)", p.strip()) for p in re.split(r"\+ (?:columns|rows) from \d+:", text)]
    return [(int(m.group(1)), int(m.group(2)), int(m.group(3))) for m in parts]


def test_single_shapes_and_k_split():
    assert _lib.matmul_describe(2048, 6144, 4096 + 128) == "256x256 x192 persistent"
    assert _lib.matmul_describe(2040, 6144, 4096 + 128) == "256x256 x192"
    assert _lib.matmul_describe(8, 4096, 4096) == "skinny"
    assert "block's waves" in _lib.matmul_describe(32, 28672, 4096)
    # 33 to 64 rows: the tiles whose blocks split K among their waves, or the 128-row tiles: wide matrices of short K, and narrow ones
    # of long K split over the chip
    assert "block's waves" in _lib.matmul_describe(64, 4096, 4096) and "block's waves" in _lib.matmul_describe(33, 6144, 4096)
    assert _lib.matmul_describe(64, 32768, 512).startswith("128x128")
    assert "K split" in _lib.matmul_describe(48, 8192, 28672)
    assert "block's waves" in _lib.matmul_describe(48, 8192, 28672, True, False)  # no workspace, no split: the small tiles
    # up to 32 rows
    assert "block's waves" in _lib.matmul_describe(32, 8192, 28672) and "block's waves" in _lib.matmul_describe(24, 8192, 28672)
    assert "block's waves" in _lib.matmul_describe(32, 8192, 8192) and "block's waves" in _lib.matmul_describe(32, 10240, 16384)
    # (K longer than the small tiles' registers hold scales of: the decode kernel)
    assert _lib.matmul_describe(24, 4096, 32768 + 128) == "skinny"
    with_ws, without = _lib.matmul_describe(256, 4096, 14336), _lib.matmul_describe(256, 4096, 14336, True, False)
    assert "K split" in with_ws and "K split" not in without
    # where the pieces of a K split would fill three quarters of the chip with at least 16 slabs each, the four-wave kernel
    # cuts every tile and its blocks exchange their sums inside the one launch
    assert _lib.matmul_describe(256, 7168, 16384) == "128x256 x56 persistent, four waves, every tile cut in pieces of 32 slabs"
    # (not with pieces of 8 slabs, not with eight pieces of 16, not where the rows fill less than three quarters of the tiles)
    assert "K split" in _lib.matmul_describe(1536, 1024, 4096) and "K split" in _lib.matmul_describe(128, 8192, 16384)
    assert "K split" in _lib.matmul_describe(48, 8192, 28672)
    assert _lib.matmul_describe(512, 2048, 28672) == "128x256 x32 persistent, four waves, every tile cut in pieces of 28 slabs"
    assert _lib.lib().maxfp8_matmul_workspace_bytes(256, 7168, 16384) >= 224 * 128 * 256 * 4
    assert _lib.matmul_describe(0, 10, 10) == "nothing to do"


def test_two_regions_cover_the_problem_once(tune):
    tune(MAXFP8_W4="0")  # (the four-wave kernel, which takes such shapes in one launch, has its own test below)
    for (M, N, K) in [(2048, 28672, 4096), (28672, 2048, 4096), (2040, 28600, 4096)]:
        text = _lib.matmul_describe(M, N, K)
        assert " + " in text, text
        cut = int(re.search(r"from (\d+)", text).group(1))
        (bm1, bn1, n1), (bm2, bn2, n2) = parse(text)
        ceil = lambda a, b: -(-a // b)
        if "columns" in text:
            assert cut % bn1 == 0 and 0 < cut < N
            assert n1 == ceil(M, bm1) * (cut // bn1) and n2 == ceil(M, bm2) * ceil(N - cut, bn2)
        else:
            assert cut % bm1 == 0 and 0 < cut < M
            assert n1 == (cut // bm1) * ceil(N, bn1) and n2 == ceil(M - cut, bm2) * ceil(N, bn2)
        assert n1 % 256 == 0, "the first region runs in whole rounds of the 256 CUs"


def test_four_wave_kernel_where_its_tile_count_fits_the_chip(tune):
    # DeepSeek-V3 o_proj at M = 4096: 448 tiles of 256 x 256 are 1.75 rounds of the 256 CUs, 728 tiles of 160 x 256 are 2.84
    assert _lib.matmul_describe(4096, 7168, 16384, True, False) == "160x256 x728 persistent, four waves"
    # with a workspace for the pieces: 616 tiles of 192 x 256 as two whole rounds and 104 tiles in two pieces each
    assert _lib.matmul_describe(4096, 7168, 16384) == "192x256 x616 persistent, four waves, tail cut in pieces of 64 slabs"
    assert _lib.lib().maxfp8_matmul_workspace_bytes(4096, 7168, 16384) >= 256 * 192 * 256 * 4
    # a ragged last column tile is fine as long as C's rows keep their 16-byte alignment (N a multiple of 8): the one matmul
    # over DeepSeek-V3's stacked q_a and kv_a weights, N = 1536 + 576
    assert _lib.matmul_describe(4096, 2112, 7168) == "160x256 x234 persistent, four waves"
    # N not a multiple of 8, an odd number of slabs, and well under one round of tiles stay with the eight-wave shapes
    assert "four waves" not in _lib.matmul_describe(4096, 7164, 16384)
    assert "four waves" not in _lib.matmul_describe(4096, 7168, 16384 + 128)
    assert "four waves" not in _lib.matmul_describe(128, 28672, 4096, False)
    # tiles of 256 x 192, named wherever they are what runs
    assert _lib.matmul_describe(2048, 6144, 4096) == _lib.matmul_describe(2040, 6144, 4096) == "256x192 x256 persistent, four waves"
    for M, N, K, block in ((4096, 57344, 8192, True), (4096, 18432, 7168, True), (512, 24576, 1536, True), (1024, 24576, 1536, False), (1216, 28672, 4096, True),
                           (1024, 24576, 1536, True), (16384, 8192, 28672, True), (2048, 2112, 4096, True), (2040, 6144, 4096 + 128, True), (117, 6144, 4096, True)):
        for workspace in (True, False):
            text = _lib.matmul_describe(M, N, K, block, workspace)
            assert _lib.matmul_tall(M, N, K, block, workspace) == text.startswith("256x192 "), (M, N, K, text)
            if text.startswith("256x192 "):
                assert text == f"256x192 x{-(-M // 256) * -(-N // 192)} persistent, four waves"
                assert bench.kernels_launched("block", M, K, N) == ("gemm_w4_kernel", text) or not block
    tune(MAXFP8_W4="0")
    assert "four waves" not in _lib.matmul_describe(4096, 7168, 16384)
    tune(MAXFP8_W4="8")
    assert _lib.matmul_describe(4096, 7168, 16384) == "256x192 x608 persistent, four waves"
    tune(MAXFP8_W4="6", MAXFP8_W4_SPLIT="0")
    assert _lib.matmul_describe(4096, 7168, 16384) == "192x256 x616 persistent, four waves"
    # the cut wants a last round of at most half the CUs' number of tiles (216 of 160 x 256 are too many), slabs in fours
    tune(MAXFP8_W4="5", MAXFP8_W4_SPLIT="1")
    assert _lib.matmul_describe(4096, 7168, 16384) == "160x256 x728 persistent, four waves"
    assert "tail cut in pieces of 8 slabs" in _lib.matmul_describe(2040, 6144, 4096)
    assert "tail cut" not in _lib.matmul_describe(2040, 6144, 4096 + 256)


def test_the_kernel_for_tens_of_tokens(tune):
    """Up to 16 rows the decode kernel; beyond, the small tiles but for row scales on weights of one decode block per CU, up to 32, and where
    the tiles' estimate is the better one."""
    kind = lambda *a, **kw: "mid" if "block's waves" in _lib.matmul_describe(*a, **kw) else _lib.matmul_describe(*a, **kw)
    for block in (True, False):
        for M in (1, 16):
            assert kind(M, 4096, 4096, block) == "skinny"
        for M in (17, 24, 32):
            for N, K in ((28672, 4096), (10240, 8192), (16384, 1024), (576, 7168)):
                assert kind(M, N, K, block) == "mid", (M, N, K)
        for M in (33, 48, 64):
            for N, K in ((4096, 4096), (1536, 7168), (10240, 8192), (6272, 512)):
                assert kind(M, N, K, block) == "mid", (M, N, K)
        assert "K split" in kind(42, 8192, 28672, block) and "K split" in kind(55, 7168, 18432, block)
    for M, N, K in ((18, 6144, 4096), (22, 5536, 640), (24, 5536, 1280), (17, 4096, 14336)):
        assert kind(M, N, K, False) == "skinny" and kind(M, N, K, True) == "mid", (M, N, K)
        assert kind(33, N, K, False) != "skinny"
    # wide weights of few slabs: 128 x 128 tiles with block scales
    assert "128x128" in kind(45, 24576, 1536) and "128x128" in kind(50, 32768, 512) and "128x128" in kind(24, 32768, 512)
    # ... and as many blocks as the chip holds at once, of 64 columns
    assert kind(64, 28672, 4096) == "mid" == kind(20, 18784, 6656)
    # (no scaling is named: what either of them uses)
    assert kind(42, 8192, 28672).endswith("K split 8") and _lib.lib().maxfp8_matmul_auto_workspace_bytes(42, 8192, 28672) > 0
    assert _lib.lib().maxfp8_matmul_auto_workspace_bytes(24, 1536, 7168) == 0
    # switches of the other kernels, and the small tiles' own, leave the decode kernel in their place
    for switch in ({"MAXFP8_MID": "0"}, {"MAXFP8_TILE": "2"}, {"MAXFP8_SPLITK": "2"}, {"MAXFP8_W4": "4"}, {"MAXFP8_SKINNY": "1408"}):
        tune(**switch)
        assert kind(24, 4096, 4096) == "skinny", switch
        tune(**{name: None for name in switch})


def test_small_tiles_stand_back_where_long_k_comes_from_memory():
    """65 to 512 rows, from 64 slabs of K on: near the tiles' estimate a K split is the quicker one with the weights from memory.  Further from it, with
    fewer slabs or with whole tiles on the other side the small tiles stay."""
    small = lambda *a: "block's waves" in _lib.matmul_describe(*a)
    for M, N, K, block in ((239, 4784, 9984, True), (223, 4096, 14336, True), (182, 2176, 14464, True), (142, 4096, 14336, False), (212, 2544, 12544, False), (73, 7056, 12032, True)):
        assert "K split" in _lib.matmul_describe(M, N, K, block) and not small(M, N, K, block), (M, N, K)
    for M, N, K, block in ((197, 1632, 14464, True), (99, 4096, 14336, True), (87, 4096, 14336, False), (207, 7168, 5120, False), (204, 4096, 4096, True), (380, 576, 7168, True), (601, 1312, 9856, False)):
        assert small(M, N, K, block), (M, N, K)


def test_small_tiles_stand_back_behind_one_round_of_large_ones():
    """Few slabs of block scales on at most one round of whole 256-row tiles: 1.2 to 1.4 times as quick as small tiles at every size measured."""
    for M, N, K in ((148, 16656, 384), (674, 5408, 384), (257, 21792, 384), (169, 20240, 640), (1602, 2496, 640), (181, 18112, 896), (162, 18160, 1152), (812, 4848, 1152), (301, 12960, 1408), (1423, 2720, 1664)):
        text = _lib.matmul_describe(M, N, K)
        assert text.startswith("256x") and "K split" not in text, (M, N, K, text)


def test_rows_quantised_inside_the_decode_kernel():
    """With row scales at most three blocks per CU for more than one token, and four tokens on two; with block scales four of them."""
    need = lambda M, N, K, gran: _lib.lib().maxfp8_linear_workspace_bytes(M, N, K, gran)
    for M, N, inside in ((1, 28672, True), (2, 24576, True), (2, 28672, False), (3, 16384, True), (3, 24576, False), (4, 16384, True), (5, 4096, False)):
        assert (need(M, N, 4096, _lib.GRAN_ROWWISE) == 0) == inside, (M, N)
    assert need(4, 28672, 4096, _lib.GRAN_BLOCK) == 0 < need(5, 28672, 4096, _lib.GRAN_BLOCK)


def test_no_workspace_for_a_plan_that_does_not_run():
    """Where tiles of 256 x 192, which need none, are ahead of a plan that cuts a tail, a linear's workspace is its quantised rows and their scales."""
    L = _lib.lib()
    for M, N, K in ((4096, 18432, 7168), (1216, 28672, 4096), (4096, 24576, 7168)):
        for granularity, scales in ((_lib.GRAN_BLOCK, K // 128 * M * 4), (_lib.GRAN_ROWWISE, M * 4), (_lib.GRAN_TENSOR, 256)):
            assert _lib.matmul_tall(M, N, K, granularity == _lib.GRAN_BLOCK)
            assert L.maxfp8_linear_workspace_bytes(M, N, K, granularity) == M * K + -(-scales // 256) * 256
        assert L.maxfp8_matmul_auto_workspace_bytes(M, N, K) == 0 < L.maxfp8_matmul_workspace_bytes(M, N, K)
    # (tall with block scales only; a cut that does run)
    assert L.maxfp8_linear_workspace_bytes(4096, 57344, 8192, _lib.GRAN_ROWWISE) > 48 << 20 > L.maxfp8_linear_workspace_bytes(4096, 57344, 8192, _lib.GRAN_BLOCK)
    assert L.maxfp8_linear_workspace_bytes(4096, 7168, 16384, _lib.GRAN_BLOCK) > 4096 * 16384 + (48 << 20)
