"""Host side of the dim reductions, no GPU: the plan's strides and which
launch a call takes (csrc/reduce_route.h, compiled here for the CPU)."""

import ctypes
import itertools
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
CUS = 256

SRC = r"""
#include "reduce_route.h"
using namespace oxi;
static RPlan plan(const int64_t* shape, const int64_t* st, int nd, int dim, int64_t* nout) {
  RPlan p{};
  *nout = 1;
  for (int d = 0; d < nd; ++d) {
    if (d == dim) continue;
    p.size[p.nd] = shape[d];
    p.st[p.nd++] = st[d];
    *nout *= shape[d];
  }
  p.len = shape[dim];
  p.rst = st[dim];
  simplify(p);
  return p;
}
// r: kernel, threads, blocks, part, parts, inner, groups, vec
extern "C" void route(const int64_t* shape, const int64_t* st, int nd, int dim, int kind, int64_t x, int cus,
                      int64_t* r) {
  int64_t nout;
  const RPlan p = plan(shape, st, nd, dim, &nout);
  const ReduceRoute q = reduce_route(kind, p, nout, reinterpret_cast<const float*>(x), nullptr, cus);
  const int64_t v[] = {(int64_t)q.kernel, q.threads, q.blocks, q.part, q.parts, q.inner, q.groups, q.vec};
  for (int i = 0; i < 8; ++i) r[i] = v[i];
}
// the offset of every output's strip
extern "C" void offsets(const int64_t* shape, const int64_t* st, int nd, int dim, int64_t* out) {
  int64_t nout;
  const RPlan p = plan(shape, st, nd, dim, &nout);
  for (int64_t e = 0; e < nout; ++e) {
    int64_t off = 0, q = e;
    for (int d = p.nd - 1; d >= 0; --d) {
      off += q % p.size[d] * p.st[d];
      q /= p.size[d];
    }
    out[e] = off;
  }
}
"""
KERNELS = ["parts", "strips", "cols", "vec", "threads"]
KINDS = ["sum", "mean", "max", "min", "argmax", "argmin", "norm"]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "route.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", "-Werror", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'oxitorch_amd' / 'csrc'}", str(d / "route.cpp"), "-o", str(d / "route.so")], check=True)
    return ctypes.CDLL(str(d / "route.so"))


def _arr(v):
    return (ctypes.c_int64 * len(v))(*v)


def row_major(shape):
    st = [1] * len(shape)
    for d in range(len(shape) - 2, -1, -1):
        st[d] = st[d + 1] * shape[d + 1]
    return st


def route(lib, shape, dim, kind="sum", strides=None, x=0):
    r = (ctypes.c_int64 * 8)()
    lib.route(_arr(shape), _arr(strides or row_major(shape)), len(shape), dim, KINDS.index(kind), ctypes.c_int64(x), CUS, r)
    return dict(zip(("kernel", "threads", "blocks", "part", "parts", "inner", "groups", "vec"), [KERNELS[r[0]], *r[1:]]))


@pytest.mark.parametrize("shape", [(1,), (5,), (3, 1), (1, 3, 1, 4), (2, 3, 4), (4, 1, 1, 5, 2), (2, 1, 2, 1, 3, 2)])
def test_simplified_plans_keep_every_output(lib, shape):
    """Row-major, transposed, broadcast and cut views: the strips start where
    the view's own strides say, in the same order."""
    n = len(shape)
    views = [row_major(shape), [0 if d % 2 else s for d, s in enumerate(row_major(shape))], [2 * s for s in row_major(shape)],
             row_major([s + 1 for s in shape]), [-s for s in row_major(shape)]]
    for perm in itertools.islice(itertools.permutations(range(n)), 24):
        rm = row_major([shape[p] for p in perm])
        views.append([rm[perm.index(d)] for d in range(n)])
    for st in views:
        for dim in range(n):
            rest = [d for d in range(n) if d != dim]
            want = np.zeros([shape[d] for d in rest], np.int64)
            for k, d in enumerate(rest):
                want += (np.arange(shape[d]) * st[d]).reshape([-1 if q == k else 1 for q in range(len(rest))])
            got = (ctypes.c_int64 * max(want.size, 1))()
            lib.offsets(_arr(shape), _arr(st), n, dim, got)
            assert list(got) == want.ravel().tolist(), (shape, st, dim)


@pytest.mark.parametrize("kind", KINDS)
def test_outputs_that_do_not_lie_side_by_side(lib, kind):
    """Short strips of many narrow rows of outputs: a thread each. Size-1 and
    adjacent dims count as one row of outputs."""
    for shape, dim in [((8192, 64, 2), 1), ((4096, 64, 3), 1), ((4096, 64, 4), 1), ((16384, 64, 1), 1)]:
        st = row_major(shape)
        if shape[2] == 1:
            st = [2 * s for s in st]  # every other float: strips are not contiguous
        r = route(lib, shape, dim, kind, st)
        assert r["kernel"] == "threads" and r["blocks"] == -(-shape[0] * shape[2] // 256), (shape, r)
    for shape in ((1000, 16384, 1), (1000, 4096, 4), (1000, 1, 64, 256)):
        r = route(lib, shape, 0, kind)
        assert (r["kernel"], r["inner"], r["blocks"]) == ("cols", 16384, 1024), (shape, r)
        assert r == route(lib, (1000, 16384), 0, kind)
    for shape, dim in [((64, 128, 2), 1), ((16, 256, 2), 1), ((1, 5000, 3), 1), ((512, 100, 8), 1)]:
        assert route(lib, shape, dim, kind)["kernel"] == "cols", shape


def test_columns_route_is_bounded(lib):
    """Its blocks stay within 8 rounds of the chip (of max and min within a
    block an output), whatever the shape."""
    for inner, length, kind in itertools.product((1, 2, 3, 4, 15, 16, 17, 1000), (64, 500, 4096, 10 ** 6), KINDS):
        for rows in (1, 100, 600, 5000, 16384):
            r = route(lib, (rows, length, inner), 1, kind, [length * inner * 2, inner * 2, 1])
            if r["kernel"] == "cols":
                assert r["blocks"] <= (16384 if kind in ("max", "min") else 16 * CUS)
                assert r["blocks"] == rows * r["groups"] and rows * inner <= 16384


@pytest.mark.parametrize("length", [32, 2048, 2049, 50257])
def test_grids_stay_below_the_thread_limit(lib, length):
    """A launch counts its threads in 32 bits: from 2^24 long strips on a wave
    takes each, and strips that do not fit so go a thread each."""
    for n in (2 ** 20, 2 ** 24 - 1, 2 ** 24, 2 ** 24 + 1, 2 ** 26 - 4, 2 ** 26, 2 ** 33):
        r = route(lib, (n, length), 1)
        block = max(r["threads"], 256)
        assert r["blocks"] < 2 ** 31 and r["blocks"] * block < 2 ** 32, (n, r)
        if n < 2 ** 26:
            assert r["kernel"] == "strips" and r["threads"] == (64 if length <= 2048 or n >= 2 ** 24 else 256), (n, r)
            assert r["blocks"] * (block // r["threads"]) >= n
        else:
            assert r["kernel"] == "threads"


@pytest.mark.parametrize("kind", KINDS)
def test_four_outputs_a_thread(lib, kind):
    """From 2048 outputs a CU on, with aligned rows of a multiple of 4; not for argmax and argmin."""
    arg = kind in ("argmax", "argmin")
    for length in (2, 29, 1000):
        for shape, dim in (((length, 2048 * CUS), 0), ((length, 512, 4 * CUS), 0), ((2048 * CUS // 64, length, 64), 1)):
            assert route(lib, shape, dim, kind)["kernel"] == ("threads" if arg else "vec"), shape
            assert route(lib, shape, dim, kind, x=4)["kernel"] == "threads"
    for shape in ((29, 2048 * CUS - 4), (29, 2048 * CUS + 2), (29, 12596, 1, 6), (1000, 20000)):
        assert route(lib, shape, 0, kind)["kernel"] == "threads", shape


def test_parts_of_a_strip(lib):
    """They cover it, none empty, and their states fit a block's LDS."""
    for n, length in itertools.product((1, 2, 3, 17, 255), (65536, 65537, 1048583, 10 ** 8, 2 ** 31)):
        r = route(lib, (n, length), 1)
        part = r["part"]
        assert r["kernel"] == "parts" and r["blocks"] == n * r["parts"] and r["parts"] <= 1024
        assert part % 4096 == 0 and (r["parts"] - 1) * part < length <= r["parts"] * part
