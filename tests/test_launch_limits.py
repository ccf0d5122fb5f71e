"""Host side of the row-wise launches, no GPU: no grid passes the 2^32 threads
that a launch can count (the rules, compiled here for the CPU)."""

import ctypes
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

SRC = r"""
#include "row_cfg.h"
extern "C" int norm_fwd_cfg(int64_t rows, int64_t H) { return oxi::norm_fwd_cfg(rows, H); }
extern "C" int block_threads(int tpr) { return oxi::row_block_threads(tpr); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("limits")
    (d / "limits.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'oxitorch_amd' / 'csrc'}", str(d / "limits.cpp"), "-o", str(d / "limits.so")], check=True)
    return ctypes.CDLL(str(d / "limits.so"))


@pytest.mark.parametrize("H", [3, 4, 1003, 4096, 8192, 8193, 12288, 16384, 16385])
def test_norm_forward(lib, H):
    """Up to 2^22 - 1 rows of 8193 to 16384 floats take 1024 threads each; 2^22
    of them (137 GB at 8193) go to the 256-thread kernel, which their grid fits."""
    for rows in (1, 1000, 2 ** 22 - 1, 2 ** 22, 2 ** 23, 2 ** 24 - 1):
        cfg = lib.norm_fwd_cfg(ctypes.c_int64(rows), ctypes.c_int64(H))
        assert (cfg == 10244) == (8192 < H <= 16384 and rows < 2 ** 22)
        threads = cfg // 10 if cfg else 256
        block = lib.block_threads(threads)
        assert -(-rows // (block // threads)) * block < 2 ** 32, (rows, H, cfg)
