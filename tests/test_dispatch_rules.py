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
#include "gemm_ring.hpp"
using namespace bk;
extern "C" {
int64_t row_b_bytes(int K, int N, int64_t ld) { return mfma2::row_b_bytes(K, N, ld); }
int dma_extent_ok(int rows, int64_t ld) { return mfma2::dma_extent_ok(rows, ld); }
unsigned row_offset(int row, int64_t ld) { return (unsigned)mfma2::row_offset(row, ld); }
int last_rows_width(int N, int rem, int K) { return mfma2::last_rows_width(N, rem, K); }
int stages_fit(int K, int SB) { return mfma2::stages_fit(K, SB); }
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
