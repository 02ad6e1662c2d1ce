"""The int8 GEMM's kernel selection on the host (csrc/gemm_plan.h, compiled by tests/gemm_plan.cpp): at sizes
too large to multiply in a test, no chosen kernel forms an offset that wraps."""
import os
import subprocess

import pytest

import x100hip

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "x100-gemm_amd", "csrc")
VARIANTS = [x100hip.GEMM_AUTO, x100hip.GEMM_TILE256, x100hip.GEMM_TILE256_W4, x100hip.GEMM_TILE128, x100hip.GEMM_TILE64,
            x100hip.GEMM_TILE32]


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "gemm_plan")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-I", CSRC, os.path.join(HERE, "gemm_plan.cpp"), "-o", exe])

    def ask(cases):   # (M, N, K, aligned, acc, variant) -> (kernel, tile, aligned, fits)
        text = "".join("%d %d %d %d %d %d\n" % tuple(map(int, c)) for c in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
        return [(k, t, int(a), int(f)) for k, t, a, f in (line.split() for line in out if line)]

    return ask


def exists(M, N, K):   # operands that fit one device
    return M * N * 4 + M * K + K * N < 200e9


def test_wide_and_long_products_keep_their_offsets(plans):
    edge = [7508480, 7508736, 1 << 23, (1 << 24) - 256, 1 << 24, 1 << 25, 1 << 27, (1 << 31) - 256]
    cases = [(M, N, K, 1, acc, v) for v in VARIANTS for acc in (0, 1) for M in (48, 256, 512) for N in [4096] + edge
             for K in [512, 576] + edge if exists(M, N, K)]
    for c, p in zip(cases, plans(cases)):
        assert p[3] and p[0] != "refused", (c, p)


def test_the_largest_256_tiles_stay(plans):
    # the last sizes whose offsets fit still take k_gemm_big
    cases = [(256, 7508480, 512, 1, 1, 1), (256, 1 << 27, 512, 1, 0, 1), (256, 512, 1 << 25, 1, 1, 1)]
    assert [p[0] for p in plans(cases)] == ["big8"] * 3
    cases = [(256, 7508736, 512, 1, 1, 1), (256, (1 << 27) + (1 << 26), 512, 1, 0, 1), (256, 512, 1 << 27, 1, 1, 1)]
    assert not any(p[0] == "big8" for p in plans(cases))


def test_aligned_products_never_fall_to_the_scalar_kernel(plans):
    sizes = [16, 48, 272, 512, 4096, (1 << 24) - 16, 1 << 24, (1 << 24) + 16, 1 << 28, (1 << 31) - 256]
    cases = [(M, N, K, 1, acc, v) for v in VARIANTS for acc in (0, 1) for M in (1, 16, 17, 256, 1 << 24) for N in sizes
             for K in sizes if exists(M, N, K) and (v == x100hip.GEMM_AUTO or N <= 1 << 28)]
    for c, p in zip(cases, plans(cases)):
        assert p[0] not in ("generic", "refused") and p[3], (c, p)


def test_tall_products_launch(plans):
    # one column of tiles: the grid of every plan holds at most 2^32 - 1 threads
    cases = [(M, N, K, K % 16 == 0 and N % 16 == 0, acc, 0) for acc in (0, 1) for K in (15, 16) for N in (1, 15, 16, 32, 48, 64)
             for M in ((1 << 29) - 32, 1 << 29, (1 << 30) - 128, 1 << 30, (1 << 30) + 1, (1 << 31) - 256) if exists(M, N, K)]
    got = plans(cases)
    for c, p in zip(cases, got):
        assert p[3] and p[0] != "refused" and (p[0] != "generic" or not c[3]), (c, p)
    assert any(p[0] == "mfma" for p in got) and any(p[0] == "generic" for p in got)


def test_short_k_takes_the_kernel_with_several_blocks_per_cu(plans):
    from test_gemm_short_k_gpu import SHAPES
    got = {(M, N, K, acc): p[:2] for (M, N, K, _, acc, _), p in zip(
        [s + (1, acc, 0) for s in SHAPES for acc in (0, 1)], plans([s + (1, acc, 0) for s in SHAPES for acc in (0, 1)]))}
    for acc in (0, 1):   # both tiles, whole and ragged, are among the GPU test's sizes
        assert {k[:3] for k, p in got.items() if k[3] == acc and p == ("mfma", "128")} >= {(2048, 2176, 64), (2049, 2128, 80),
                                                                                        (4096, 1152, 192), (8000, 4112, 176)}
        assert {k[:3] for k, p in got.items() if k[3] == acc and p == ("mfma", "64")} >= {(1024, 1024, 64), (1601, 1040, 48),
                                                                                       (64, 65536, 64), (70001, 32, 64)}
    # sizes that were 1.1 to 1.6 times slower on k_gemm_tile
    slow = [(4096, 4096, 64, 1), (4096, 4096, 256, 0), (4096, 4096, 256, 1), (7168, 4096, 320, 1), (256, 1 << 20, 128, 0), (16384, 16384, 256, 0), (65536, 256, 128, 1)]
    assert {p[0] for p in plans([(M, N, K, 1, acc, 0) for M, N, K, acc in slow])} == {"mfma"}
    # and sizes that are faster there
    fast = [(333, 6144, 2048, 0), (256, 256, 256, 1), (2000, 8128, 512, 1), (512, 512, 64, 0), (31, 209280, 128, 1),
            (35584, 192, 128, 1), (1024, 3584, 384, 0)]
    assert {p[0] for p in plans([(M, N, K, 1, acc, 0) for M, N, K, acc in fast])} == {"tile"}


def test_the_gpu_tests_reach_every_form_of_the_tiles(plans):
    from test_gemm_tile_gpu import FORMS
    cases = [(M, N, K, a, acc, 0) for _, a, M, N, K in FORMS for acc in (0, 1)]
    want = [("tile", t, a) for t, a, *_ in FORMS for _ in (0, 1)]
    assert [p[:3] for p in plans(cases)] == want


def test_few_rows_of_a_long_k_split_it(plans):
    # the split-K kernels were up to twice as fast as 32x32 tiles here; and sizes that the tiles win
    split = [(9, 3072, 9984), (10, 3456, 8768), (16, 3232, 10096), (14, 4096, 13120)]
    tile = [(16, 1280, 1280), (14, 154960, 80), (14, 174832, 160), (14, 2016, 5792), (12, 2048, 9024)]
    for sizes, kernel in ((split, "skinny"), (tile, "tile")):
        assert {p[0] for p in plans([(M, N, K, 1, acc, 0) for M, N, K in sizes for acc in (0, 1)])} == {kernel}, kernel
