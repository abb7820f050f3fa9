"""The launch rules (csrc/launch_rules.hpp) over sizes up to the operators' limits, built for the host:
every launch they choose fits a dispatch, whose work-items (blocks x threads) count in 32 bits."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BIG = (1 << 31) - 1


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++") or "/opt/rocm/bin/amdclang++"
    so = str(tmp_path_factory.mktemp("rules") / "rules.so")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "launch_rules", "rules_abi.cpp")], check=True)
    lib = ctypes.CDLL(so)
    i64 = ctypes.c_int64
    lib.rule_grid_fits.argtypes = [i64, i64]
    lib.rule_dqsq_blocks.argtypes = [i64, i64]
    lib.rule_dqsq_blocks.restype = i64
    gl = ctypes.POINTER(i64)
    lib.rule_pick_deq.argtypes = [gl, i64, i64, i64, i64, i64, ctypes.c_int]
    lib.rule_pick_gmm.argtypes = [gl, i64, i64, i64, i64]
    lib.rule_gmsq_skips_empty.argtypes = [gl, i64]
    lib.rule_ring_skips_empty.argtypes = [gl, i64]
    lib.rule_gmsq_decode_grid.argtypes = [i64, i64, i64]
    lib.rule_gmsq_decode_grid.restype = i64
    return lib


@pytest.mark.parametrize("threads", [64, 128, 192, 256, 320, 512])
def test_dqsq_grid(rules, threads):
    """The row walk launches at least one workgroup, at most one per row, and never more than a dispatch
    holds, up to the operator's row limit (2^27 rows of 64 threads are one too many at two rows each)."""
    for M in (1, 2, 3, 1000, 16385, 131072, (1 << 27) - 1, 1 << 27, (1 << 27) + 1, 1 << 30, BIG):
        n = rules.rule_dqsq_blocks(M, threads)
        assert 1 <= n <= M
        assert rules.rule_grid_fits(n, threads), (M, n)
    # below the limit: two rows each
    assert rules.rule_dqsq_blocks(131072, threads) == max(65536, 512 * (2048 // threads))


# tile numbers of the rules: (rows, columns, threads)
DEQ_TILES = [(32, 64, 256), (64, 128, 256), (64, 256, 256), (128, 128, 512), (128, 256, 512)]
GMM_TILES = DEQ_TILES + [(256, 256, 512)]
RING, SKINNY, LDS, SKINNY2 = 5, 6, 7, 8  # the other kernels of the int8 rule


def _one_group(M):
    return (ctypes.c_int64 * 1)(M)


# outputs of at most 64 GB: rows up to the operators' limit with the narrowest vector columns, and wide ones
BIG_SHAPES = [(M, n) for M in (1, 1 << 20, 1 << 27, (1 << 28) + 1, 1 << 29, 1 << 30, BIG)
              for n in (8, 16, 48, 512, 8192) if M * n <= 1 << 35]


@pytest.mark.parametrize("M,N", BIG_SHAPES)
@pytest.mark.parametrize("K", [16, 64, 256])
def test_tile_grids(rules, M, N, K):
    """The tile that a rule picks fits a dispatch: 2^30 x 16 outputs are 2^24 tiles of 64 x 128 with 256
    threads, one dispatch too many.  (A rule that finds no fitting tile names none, and the caller takes
    the kernels that tile coarser or walk their tiles.)"""
    tiles = lambda t: -(-M // t[0]) * -(-N // t[1])
    if N % 16 == 0:
        p = rules.rule_pick_deq(_one_group(M), 1, M, K, N, 1, K >= 256)
        if 0 <= p < len(DEQ_TILES):
            t = DEQ_TILES[p]
            assert rules.rule_grid_fits(tiles(t), t[2]), (p, tiles(t))
    p = rules.rule_pick_gmm(_one_group(M), 1, M, K, N)
    if p >= 0:
        t = GMM_TILES[p]
        assert rules.rule_grid_fits(tiles(t), t[2]), (p, tiles(t))


def _gl(counts):
    ends, s = [], 0
    for c in counts:
        s += c
        ends.append(s)
    return (ctypes.c_int64 * len(ends))(*ends)


@pytest.mark.parametrize("counts,skips", [
    ([33] * 64, True), ([47] * 256, True), ([192] * 8, True),          # no tile full enough to lose
    ([256] * 256, False), ([224] * 64, False), ([512] * 64, False),    # full tiles
    ([257] * 128, False), ([288] * 128, False), ([300] * 256, False),  # a full and a nearly empty tile each
    ([300] + [40] * 255, True), ([300] + [40] * 15, True),             # small groups beside a full tile
    ([1000, 700, 400] + [224, 130, 90, 60] * 2, True),                 # skewed: most groups of one tile
    ([250] * 60 + [300] * 4, False),                                   # nearly full tiles
    ([0] * 200 + [0, 40, 0], True),
])
def test_gmsq_skip_rule(rules, counts, skips):
    """Leaving out the empty fragments is taken where it gains (groups far below a tile) and not where it loses
    (full tiles; groups of just over a tile)."""
    assert bool(rules.rule_gmsq_skips_empty(_gl(counts), len(counts))) is skips


@pytest.mark.parametrize("counts,skips", [
    ([33] * 64, True), ([129] * 16, True), ([256] * 8, True), ([224, 7, 0, 256], True),  # one tile per group
    ([274] * 256, False), ([336] * 64, False), ([571] * 64, False),  # a full and a lighter tile in each group
    ([600] + [40] * 31, True),                                       # mostly empty fragments
    ([1000, 700, 400] + [224, 130, 90, 60] * 2, True),               # most groups of one tile
])
def test_ring_skip_rule(rules, counts, skips):
    assert bool(rules.rule_ring_skips_empty(_gl(counts), len(counts))) is skips


@pytest.mark.parametrize("counts,K,N,batch,kernel", [
    # wide products of partly filled rounds, and groups of about a tile: the ring core
    ([1614], 3648, 12288, 1, RING), ([3647], 8640, 4928, 1, RING), ([217] * 16, 3392, 5056, 1, RING),
    # short K and small batches of more than 32 rows: the 8-wave 256 x 256 kernel, not the ring's constants
    ([11288], 208, 1088, 1, LDS), ([1862], 96, 6976, 1, LDS), ([94], 832, 1280, 32, LDS), ([1362], 960, 1344, 4, LDS),
    # small products: tiles that fill the chip; few rows of many experts: the streaming kernel
    ([24], 7168, 4096, 1, 0), ([300], 7168, 4096, 1, 1), ([8] * 256, 2048, 7168, 1, SKINNY),
    ([8] * 254 + [18, 2], 2048, 7168, 1, SKINNY2), ([29], 960, 1472, 32, 2),
])
def test_dequant_kernel_choice(rules, counts, K, N, batch, kernel):
    assert rules.rule_pick_deq(_gl(counts), len(counts), sum(counts), K, N, batch, K >= 256) == kernel


@pytest.mark.parametrize("rows", [1, 16, 32])
@pytest.mark.parametrize("batch", [1, 4])
def test_dequant_choice_of_few_rows(rules, rows, batch):
    """Calls whose groups have at most 32 rows have no 256 x 256 kernel: the rule offers none."""
    for K in (16, 256, 7168):
        for N in (16, 1024, 16384):
            assert rules.rule_pick_deq(_gl([rows]), 1, rows, K, N, batch, K >= 256) not in (RING, LDS)


@pytest.mark.parametrize("counts,K,N,tile", [
    ([156] * 32, 2496, 4352, 5), ([175] * 8, 1984, 4416, 5), ([1687, 1688], 4544, 3776, 5),  # uneven rounds, long K
    ([8] * 64, 4096, 4096, 2), ([256] * 64, 4096, 4096, 5), ([64] * 64, 4096, 4096, 2),
])
def test_grouped_matmul_tile_choice(rules, counts, K, N, tile):
    assert rules.rule_pick_gmm(_gl(counts), len(counts), sum(counts), K, N) == tile


def test_gmsq_decode_grid(rules):
    """One workgroup per CU; fewer only where the call has fewer column tiles in all its groups, empty ones
    included."""
    assert rules.rule_gmsq_decode_grid(256, 9, 256) == 256
    assert rules.rule_gmsq_decode_grid(8, 5, 256) == 40
    assert rules.rule_gmsq_decode_grid(1, 1, 256) == 1
    assert rules.rule_gmsq_decode_grid(256, 16, 0) == 0  # the kernel cannot be resident
