"""Extents and selection rules of the GEMM launchers, as host functions.

The rules are inline functions of the kernel headers; a small library of
C entry points is compiled from them for the host only, so no GPU is needed.
"""
import ctypes
import subprocess

import numpy as np
import pytest

from baracuda_amd import build as B

SOURCE = r"""
#include "moe_rules.hpp"
using namespace bk;
extern "C" {
int64_t row_b_bytes(int K, int N, int64_t ld) { return mfma2::row_b_bytes(K, N, ld); }
int dma_extent_ok(int rows, int64_t ld) { return mfma2::dma_extent_ok(rows, ld); }
unsigned row_offset(int row, int64_t ld) { return (unsigned)mfma2::row_offset(row, ld); }
int moe_fit(int64_t x_rows, int N, int64_t kb, int operands, int out16) {
    const MoeFit f = moe_fit(x_rows, N, kb, operands != 0, out16 != 0);
    return f.decode + 2 * f.ring + 4 * f.tiles256;
}
int moe_decode_width(int pairs, int E, int N, int64_t kb) { return bk::moe_decode_width(pairs, E, N, kb); }
int last_rows_width(int N, int rem, int K) { return mfma2::last_rows_width(N, rem, K); }
int last_rows_pass(int M, int N) { return mfma2::last_rows_pass(M, N, 128); }
int last_rows_pay(int M, int N, int K, int rem) { return mfma2::last_rows_pay(M, N, K, rem); }
int last_rows_col_frags(int N, int blocks) { return mfma2::last_rows_col_frags(N, blocks); }
int last_rows_blocks(int rem, int N) {
    int rf, blocks, nb;
    mfma2::last_rows_blocks(rem, N, rf, blocks, nb);
    return rf * 100 + nb * 10 + blocks;
}
int stages_fit(int K, int SB) { return mfma2::stages_fit(K, SB); }
int tail_split_pays(int M, int N, int K, int full, int tail) { return mfma2::tail_split_pays(M, N, K, full, tail); }
int row_blocks_pay(int M, int N, int K) { return mfma2::row_blocks_pay(M, N, K); }
int ring_tile(int M, int N, int K, int first) { return mfma2::ring_tile(M, N, K, nullptr, (mfma2::RingTile)first); }
}
"""


@pytest.fixture(scope="session")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.hip").write_text(SOURCE)
    cmd = [B.HIPCC, *B.HIP_FLAGS, "--offload-host-only", "-w", "-shared", str(d / "rules.hip"), "-o", str(d / "rules.so")]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    lib = ctypes.CDLL(str(d / "rules.so"))
    lib.row_b_bytes.restype = ctypes.c_int64
    lib.row_b_bytes.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64]
    lib.dma_extent_ok.argtypes = [ctypes.c_int, ctypes.c_int64]
    lib.row_offset.restype = ctypes.c_uint32
    lib.row_offset.argtypes = [ctypes.c_int, ctypes.c_int64]
    lib.moe_decode_width.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int64]
    lib.moe_fit.argtypes = [ctypes.c_int64, ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    return lib


@pytest.mark.parametrize("k,n,ld", [(1, 16, 16), (16, 250, 256), (48, 262, 272), (208, 520, 1040), (144, 4100, 4608),
                                    (336, 1000, 1008), (512, 256, 256), (400, 2064, 14336)])
def test_row_major_b_extent(rules, k, n, ld):
    """Every 16-byte unit of a 256-column tile that the extent admits holds a
    byte of the view (the last row owns n bytes, the others the pitch), and
    the units of the k-rows past the last one are not admitted."""
    extent = rules.row_b_bytes(k, n, ld)
    own = (k - 1) * ld + n                      # bytes of the strided view
    assert own <= extent < own + 16 and extent % 16 == 0
    rows = np.arange((k + 127) // 128 * 128 + 128)[:, None]
    units = np.arange(0, (n + 255) // 256 * 256, 16)[None, :]
    off = rows * ld + units
    admitted = off < extent
    assert not admitted[k:].any()
    assert (off[admitted] < own).all()
    assert admitted[:k, : (n + 15) // 16].all()


@pytest.mark.parametrize("rem", [1, 2, 5, 16, 17, 32])
@pytest.mark.parametrize("k", [16, 512, 4096, 8192, 14336])
def test_last_rows_width(rules, rem, k):
    """One fragment only where it is one round of 256 workgroups; past one round
    of the widest group no width needs more than a half over the fewest columns
    per CU; the launchers have every width that the rule gives."""
    for n in range(16, 65536, 16):
        nb = rules.last_rows_width(n, rem, k)
        groups = -(-n // (16 * nb))
        assert nb in (1, 2, 3, 4, 6, 7)
        assert nb > 1 or groups <= 256
        if n <= 28672:
            assert groups <= 512
        per_cu = {w: -(-(-(-n // (16 * w))) // 256) * w for w in (1, 2, 3, 4, 6, 7)}
        assert per_cu[nb] <= 1.5 * min(per_cu.values())


def test_stage_depths(rules):
    """A stage deeper than 512 bytes only where K fills it as far as it fills
    stages of 512."""
    for k in range(16, 20000, 16):
        assert rules.stages_fit(k, 512) and rules.stages_fit(k, 256)
        for sb in (1024, 2048):
            assert rules.stages_fit(k, sb) == (-(-k // 512) % (sb // 512) == 0)


def test_row_blocks_or_tiles(rules):
    """Row blocks and tiles on the sides of the line where each was measured the
    faster (int8 and e4m3)."""
    blocks = [(200, 1024, 4096), (128, 4096, 14336), (512, 1024, 4096), (160, 6144, 8192), (256, 8192, 8192),
              (300, 4096, 14336), (384, 4096, 14336), (512, 4096, 14336), (300, 5120, 14336), (100, 14336, 8192),
              (80, 14336, 14336), (160, 5120, 14336), (200, 4096, 11264), (256, 4096, 14336)]
    tiles = [(200, 4096, 4096), (384, 2048, 1024), (128, 8192, 4096), (64, 14336, 4096), (384, 4096, 8192),
             (128, 5120, 14336), (128, 11008, 14336), (80, 11008, 14336), (256, 4096, 11264), (300, 2048, 14336),
             (128, 14336, 4096), (512, 4096, 4096)]
    assert [s for s in blocks if not rules.row_blocks_pay(*s)] == []
    assert [s for s in tiles if rules.row_blocks_pay(*s)] == []


def test_tile_of_many_rounds(rules):
    """Past three rounds of 256 x 256 tiles nothing smaller; the shapes of one
    round keep their tile (0 .. 5: 64x64, 64x128, 128x128, 128x256, 192x256, 256x256)."""
    for s in [(3072, 17920, 4096), (4096, 13824, 4096), (3072, 28672, 2048), (1024, 50176, 4096)]:
        assert rules.ring_tile(*s, 0) == rules.ring_tile(*s, 3) == 5
    for s, t in [((777, 11008, 4096), 4), ((1500, 5120, 2880), 3), ((810, 2352, 1856), 1), ((3072, 4096, 4096), 4),
                 ((600, 50176, 4096), 3), ((1000, 17920, 1024), 4), ((4096, 4096, 4096), 5)]:
        assert rules.ring_tile(*s, 0) == t


@pytest.mark.parametrize("m,n,k,full,tail,split", [
    (512, 512, 8192, 0, 4, False), (512, 1024, 4096, 0, 8, False), (768, 1152, 16384, 0, 15, False),
    (256, 256, 24576, 0, 1, False), (768, 768, 20480, 0, 9, True), (200, 520, 24576, 0, 3, True),
    (4296, 4096, 4096, 256, 16, True), (4296, 4096, 2048, 256, 16, False), (5120, 4096, 4096, 256, 64, False),
    (5120, 4096, 8192, 256, 64, True), (8448, 4096, 4096, 512, 16, False), (8448, 4096, 14336, 512, 16, True),
    (12544, 4096, 4096, 768, 16, True)])
def test_tail_split_where_it_was_faster(rules, m, n, k, full, tail, split):
    """A workspace does not move a call to the slower of the two measured ways."""
    assert bool(rules.tail_split_pays(m, n, k, full, tail)) == split


@pytest.mark.parametrize("rows", [1, 64, 200, 256, 257, 600, 12000])
def test_row_offsets_of_padded_tiles(rules, rows):
    """The offsets of every tile height and column group stay exact in 32 bits,
    the rows past the operand's end included, for the widest pitch accepted."""
    ld = (2 ** 31 - 1) // (-(-rows // 256) * 256) // 16 * 16
    assert rules.dma_extent_ok(rows, ld) and not rules.dma_extent_ok(rows, 2 * ld)
    for edge in (16, 32, 48, 64, 96, 112, 128, 192, 256):
        last = -(-rows // edge) * edge - 1
        assert rules.row_offset(last, ld) == last * ld < 2 ** 32 - ld
        assert rules.row_offset(rows, ld) >= rows * ld      # past the extent


def test_last_rows_block_forms(rules):
    """The launchers have kernels for every row-block form the rule gives: 2 or 4
    row fragments by 1 or 2 column fragments."""
    forms = {rules.last_rows_blocks(rem, n) // 10 for n in range(16, 70000, 16) if rules.last_rows_col_frags(n, 1) == 1
             for rem in (33, 48, 64, 65, 96, 97, 128)}
    assert forms == {21, 22, 41, 42}


def test_moe_fit(rules):
    """Decode-sized problems keep their kernels with an output of any alignment."""
    decode, ring, tiles256 = 1, 2, 4
    assert rules.moe_fit(64, 14336, 8192, 1, 1) == decode + ring + tiles256
    assert rules.moe_fit(64, 14336, 8192, 1, 0) == decode + tiles256
    assert rules.moe_fit(64, 1408, 2064, 1, 1) == decode + ring
    assert rules.moe_fit(64, 1412, 2064, 1, 1) == rules.moe_fit(64, 1408, 2056, 1, 1) == 0
    assert rules.moe_fit(64, 14336, 8192, 0, 1) == 0


def test_routes_of_wide_last_rows(rules):
    """The shapes with which tests/test_gpu_tiles.py means the 32-column
    kernels of four and eight fragments, and row blocks past 128 tiles, get them."""
    assert rules.row_blocks_pay(40, 6176, 304) and rules.last_rows_col_frags(6176, 1) == 2
    for m, rem in [(1856, 64), (1892, 100)]:
        assert rules.last_rows_pass(m, 8224) == rem and rules.last_rows_pay(m, 8224, 144, rem)
        assert not rules.row_blocks_pay(m, 8224, 144) and rules.last_rows_col_frags(8224, 1) == 2
    # (rows, N, K, rows of a block, fragments): one round of workgroups each
    for m, n, k, rb, nb in [(160, 5120, 11280, 64, 4), (384, 2720, 9232, 128, 2), (200, 8192, 8208, 128, 4)]:
        assert rules.row_blocks_pay(m, n, k)
        blocks = -(-m // rb)
        assert rules.last_rows_col_frags(n, blocks) == nb and blocks * (n // (16 * nb)) <= 256
        if rb == 128:
            b4 = -(-m // 64)
            assert b4 * (n // (16 * rules.last_rows_col_frags(n, b4))) > 256


def test_moe_decode_width(rules):
    """The measured best width, or one within 3% of it: (pairs, experts, N, bytes of a row)."""
    for width, cases in {1: [(2, 8, 1024, 2048), (4, 8, 1024, 8192), (8, 8, 7168, 8192), (16, 16, 2048, 8192)],
                         2: [(2, 8, 2048, 2048), (8, 8, 1024, 4096), (16, 8, 7168, 4096), (32, 16, 7168, 2048),
                             (16, 16, 2048, 4096), (64, 8, 1024, 2048)],
                         4: [(2, 8, 14336, 8192), (8, 16, 2048, 4096), (24, 64, 2048, 4096), (4, 16, 7168, 8192),
                             (64, 8, 7168, 4096), (48, 64, 1024, 8192)]}.items():
        assert [c for c in cases if rules.moe_decode_width(*c) != width] == []
    for pairs in range(1, 65):                     # the launcher has these
        for e in (1, 8, 64, 1024):
            for n in (8, 1000, 4096, 50000):
                for kb in (16, 4096, 28672):
                    assert rules.moe_decode_width(pairs, e, n, kb) in ((1, 2, 4) if pairs <= 32 else (2, 4))
