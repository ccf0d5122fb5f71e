"""Host side of the launches, no GPU (the rules, compiled here for the CPU): no
grid of the row-wise kernels passes the 2^32 threads that a launch can count,
and which tiles transposed elementwise calls take."""

import ctypes
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

SRC = r"""
#include "map_route.h"
#include "row_cfg.h"
#include "softmax_mid.h"
extern "C" int norm_fwd_cfg(int64_t rows, int64_t H) { return oxi::norm_fwd_cfg(rows, H); }
extern "C" int block_threads(int tpr) { return oxi::row_block_threads(tpr); }
extern "C" int through_lds(int unary, int op, int64_t J, int64_t D, int64_t blocks, int cus) {
  return oxi::map_through_lds(unary < 0 ? oxi::OP_LONG : unary ? oxi::unary_length(op) : oxi::binary_length(op), J, D,
                              blocks, cus);
}
extern "C" int64_t mid_outer_max(int64_t len, int64_t inner) { return oxi::mid_outer_max(len, inner); }
extern "C" void mid_shape(int64_t outer, int64_t len, int64_t inner, int64_t* v) {
  const oxi::MidShape m = oxi::mid_shape(outer, len, inner);
  const int64_t q[] = {m.nt, m.tx, m.ty, m.nv, m.units, m.total, m.blocks};
  for (int i = 0; i < 7; ++i) v[i] = q[i];
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("limits")
    (d / "limits.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'oxitorch_amd' / 'csrc'}", str(d / "limits.cpp"), "-o", str(d / "limits.so")], check=True)
    lib = ctypes.CDLL(str(d / "limits.so"))
    lib.mid_outer_max.restype = ctypes.c_int64
    return lib


def mid_shape(lib, outer, length, inner):
    v = (ctypes.c_int64 * 7)()
    lib.mid_shape(ctypes.c_int64(outer), ctypes.c_int64(length), ctypes.c_int64(inner), v)
    return dict(zip(("nt", "tx", "ty", "nv", "units", "total", "blocks"), v))


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


@pytest.mark.parametrize("length", [1, 2, 16, 17, 32, 33, 128, 150, 256, 257, 512, 513, 1024, 2048, 2049, 100000])
@pytest.mark.parametrize("inner", [2, 3, 4, 5, 4096, 10 ** 6])
def test_middle_dim_softmax(lib, length, inner):
    """A launch takes as many outer indices as its grid holds: 2^30 of (17, 2)
    (146 GB) ran on a thread a column, and take several threads a column now."""
    most = lib.mid_outer_max(ctypes.c_int64(length), ctypes.c_int64(inner))
    for outer in (1, most, min(most, 2 ** 31)):
        m = mid_shape(lib, outer, length, inner)
        assert m["blocks"] < 2 ** 31 and m["blocks"] * m["nt"] < 2 ** 32, m
        assert m["blocks"] * m["tx"] >= m["total"] == outer * m["units"] and m["tx"] * m["ty"] == m["nt"]
    # one more outer index than that would pass the limit, or nearly (a block's worth)
    m = mid_shape(lib, most + 2 * m["tx"] + 1, length, inner)
    assert m["blocks"] * m["nt"] >= 2 ** 32 - 2 * m["nt"]


def test_middle_dim_softmax_kernels(lib):
    """The shapes whose kernels exist: streamed on 1024 threads, few positions on 256."""
    for inner, few, most in ((2, 4, 16), (3, 4, 16), (4, 2, 8), (5, 2, 8), (1000, 2, 8)):
        got = {(m["nv"], m["nt"]) for m in (mid_shape(lib, 1, n, inner) for n in [*range(1, 5000), 10 ** 5, 10 ** 9])}
        assert got == {(0, 1024), (few, 256), (most, 256), (most, 1024)}


def test_transposed_tiles(lib):
    """Long operations on tiny odd extents go through LDS while few; short ones never."""
    UN = ["neg", "abs", "sqrt", "rsqrt", "exp", "log", "log2", "log10", "sin", "cos", "tanh", "relu", "sigmoid"]

    def lds(op, B, J, D):
        kind, code = {"act": (-1, 0), "add": (0, 0), "pow": (0, 4)}.get(op) or (1, UN.index(op))
        blocks = B * -(-J // 64) * -(-D // 64)
        return bool(lib.through_lds(kind, code, *(ctypes.c_int64(v) for v in (J, D, blocks)), 256))

    for op in ("act", "tanh", "sin", "sigmoid", "pow"):
        assert all(lds(op, B, J, D) for B in (1, 25, 100, 1000) for J, D in ((4, 5), (7, 7), (11, 4), (4, 11))), op
        assert not any(lds(op, B, J, D) for B in (1, 100) for J, D in ((31, 33), (33, 5), (1001, 5), (50, 63))), op
        assert not lds(op, 100_000, 7, 7) and not lds(op, 5000, 11, 11), op
    assert lds("act", 100, 11, 11) and not lds("act", 1000, 11, 11) and not lds("act", 1, 5, 1001)
    assert lds("pow", 100, 5, 1001) and not lds("pow", 1000, 5, 1001) and lds("pow", 10_000, 4, 11)
    assert not any(lds(op, B, 7, 7) for op in ("add", "neg", "abs", "relu") for B in (1, 100, 10_000))
