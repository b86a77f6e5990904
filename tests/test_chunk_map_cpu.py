"""The window -> chunk arithmetic of the suffix kernels, the fix-up and the
cascade epilogue (`ChunkMap` in csrc/chunk_map.h), checked on the host.

The kernels take floor(x / d) as the truncated IEEE double quotient
(`div_nonneg`) for 0 <= x <= W P and 1 <= d < 2^31, where W < 2^31 windows (the
int32 prefix sums) and P <= 2^20 chunks (the ABI's limit). numpy's float64
division is the same correctly rounded IEEE operation, so these tests pin the
identity on random and adversarial operands (quotients just below an integer,
the largest operands), show that a single-precision quotient fails them, and
check the chunk map built on it: chunk c covers [lo(c), lo(c + 1)) and owner(p)
is the chunk whose range holds window p. The header itself is compiled for the host
and checked too: it is the code the kernels run."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

X_MAX = (2 ** 31 - 1) * 2 ** 20  # W P at the limits


def _div(x, d, dtype=np.float64):
    return (x.astype(dtype) / d.astype(dtype)).astype(np.int64)


def _operands(rng, n):
    d = np.concatenate([rng.integers(1, 2 ** 31, n), rng.integers(1, 5000, n)])
    q = rng.integers(0, X_MAX // d + 1)
    x = np.concatenate([
        rng.integers(0, X_MAX + 1, 2 * n),                  # anywhere
        np.minimum(q * d + d - 1, X_MAX),                   # just below the next integer
        q * d,                                              # exact quotients
        np.maximum(q * d - 1, 0),
    ])
    return x, np.concatenate([d, d, d, d])


def test_double_quotient_is_the_integer_floor():
    rng = np.random.default_rng(0)
    for _ in range(8):
        x, d = _operands(rng, 250_000)
        assert ((x >= 0) & (x <= X_MAX)).all()
        np.testing.assert_array_equal(_div(x, d), x // d)
    # the extremes
    x = np.array([X_MAX, X_MAX - 1, 2 ** 31 - 2, 0, (2 ** 31 - 1) * (2 ** 20 - 1)], dtype=np.int64)
    d = np.array([2 ** 31 - 1, 2 ** 31 - 1, 2 ** 31 - 1, 1, 2 ** 20], dtype=np.int64)
    np.testing.assert_array_equal(_div(x, d), x // d)


def test_single_precision_quotient_would_fail():
    # the check has teeth: a float32 quotient misses the floor on these operands
    rng = np.random.default_rng(1)
    x, d = _operands(rng, 50_000)
    assert (_div(x, d, np.float32) != x // d).any()


def _lo(c, W, P, split):
    if split == 0:
        return _div(c * W, np.full_like(c, P))
    h, j = P // 2, c // 2
    a = _div(j * W, np.full_like(j, h))
    b = _div((j + 1) * W, np.full_like(j, h))
    return np.where(c % 2 == 0, a, a + (((b - a) * split) >> 8))


def _owner(p, W, P, split):
    if split == 0:
        return _div((p + 1) * P - 1, np.full_like(p, W))
    j = _div((p + 1) * (P // 2) - 1, np.full_like(p, W))
    return 2 * j + (p >= _lo(2 * j + 1, W, P, split))


@pytest.mark.parametrize("W,P,split", [
    (1, 1, 0), (7, 512, 0), (1088, 64, 0), (1088, 64, 192), (5, 64, 192), (33787, 512, 0),
    (2 ** 31 - 1, 2 ** 20, 0), (2 ** 31 - 1, 512, 192), (123457, 1000, 128), (2 ** 30 + 3, 2 ** 20, 255),
])
def test_chunk_map_ranges_and_owner(W, P, split):
    c = np.arange(P + 1, dtype=np.int64)
    lo = _lo(c, W, P, split)
    # exact integer restatement of the ranges
    if split == 0:
        ref = c * W // P
    else:
        h, j = P // 2, c // 2
        a, b = j * W // h, (j + 1) * W // h
        ref = np.where(c % 2 == 0, a, a + (b - a) * split // 256)
    np.testing.assert_array_equal(lo, ref)
    assert lo[0] == 0 and lo[-1] == W and (np.diff(lo) >= 0).all()
    # owner(p) is the chunk holding window p: every window of a small map, a sample of a large one
    p = np.arange(W, dtype=np.int64) if W <= 1 << 16 else np.unique(np.concatenate([
        np.random.default_rng(2).integers(0, W, 1 << 16), lo[1:-1] - 1, lo[1:-1], [0, W - 1]]))
    p = p[(p >= 0) & (p < W)]
    own = _owner(p, W, P, split)
    assert ((own >= 0) & (own < P)).all()
    assert (lo[own] <= p).all() and (p < lo[own + 1]).all()


def _few_lo(c, W, P, split):
    """lo(c) below one window per chunk: one each for the first chunks, or the last (split > 0)."""
    return np.minimum(c, W) if split == 0 else np.maximum(c - (P - W), 0)


def _few_owner(p, W, P, split):
    return p if split == 0 else p + P - W


@pytest.mark.parametrize("P,split", [(64, 0), (512, 0), (64, 208), (2, 208), (64, 128), (64, 255)])
def test_no_empty_chunk_inside_a_cut_sequence(P, split):
    """Below and at one window per chunk: every window has one owner, and every chunk
    between the owners of two windows holds windows (the fold reads them all)."""
    for W in sorted({1, 2, 3, 5, P - 2, P - 1, P, P + 1, 3 * P + 1} - {0}):
        c, p = np.arange(P + 1, dtype=np.int64), np.arange(W, dtype=np.int64)
        few = W < P
        lo = _few_lo(c, W, P, split) if few else _lo(c, W, P, split)
        own = _few_owner(p, W, P, split) if few else _owner(p, W, P, split)
        assert lo[0] == 0 and lo[-1] == W
        size = np.diff(lo)
        assert (size >= 0).all()
        np.testing.assert_array_equal(np.repeat(np.arange(P), size), own)
        assert (size[own.min():own.max() + 1] >= 1).all()


CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-hust-cascade-kernel_amd", "csrc")


@pytest.fixture(scope="module")
def header(tmp_path_factory):
    """lo and owner of csrc/chunk_map.h, compiled for the host"""
    d = tmp_path_factory.mktemp("chunk_map")
    src = d / "chunk_map.cpp"
    src.write_text("""#include "chunk_map.h"
extern "C" void lo(int64_t W, int P, int split, const int64_t *c, int64_t n, int64_t *out) {
    const ck::ChunkMap m{W, P, split};
    for (int64_t i = 0; i < n; ++i) out[i] = m.lo((int)c[i]);
}
extern "C" void owner(int64_t W, int P, int split, const int64_t *p, int64_t n, int64_t *out) {
    const ck::ChunkMap m{W, P, split};
    for (int64_t i = 0; i < n; ++i) out[i] = m.owner(p[i]);
}
""")
    lib = d / "chunk_map.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, str(src), "-o", str(lib)], check=True)
    handle = ctypes.CDLL(str(lib))

    def call(name, x, W, P, split):
        x = np.ascontiguousarray(x, dtype=np.int64)
        out = np.empty_like(x)
        ptr = ctypes.POINTER(ctypes.c_int64)
        getattr(handle, name)(ctypes.c_int64(W), ctypes.c_int(P), ctypes.c_int(split), x.ctypes.data_as(ptr),
                              ctypes.c_int64(x.size), out.ctypes.data_as(ptr))
        return out
    return call


@pytest.mark.parametrize("P,split", [(1, 0), (64, 0), (512, 0), (73, 0), (2, 208), (64, 208), (64, 224), (512, 224),
                                     (64, 128), (64, 255)])
def test_compiled_header(header, P, split):
    """Every window has one owner, every chunk between the owners of two windows holds
    windows, and from one window per chunk on the ranges are the exact shares."""
    for W in sorted({1, 2, 3, 4, 5, P // 2, P - 2, P - 1, P, P + 1, 3 * P + 1, 20011, 2 ** 31 - 1}):
        if W < 1:
            continue
        c = np.arange(P + 1, dtype=np.int64)
        lo = header("lo", c, W, P, split)
        assert lo[0] == 0 and lo[-1] == W and (np.diff(lo) >= 0).all(), (W, lo)
        if W < P:  # one window a chunk, in the fused kernel the last ones: no stage-1 unit is there
            np.testing.assert_array_equal(np.flatnonzero(np.diff(lo)), np.arange(W) + (P - W if split else 0))
        if W >= P:
            h = max(P // 2, 1)
            a, b = c // 2 * W // h, (c // 2 + 1) * W // h
            np.testing.assert_array_equal(lo, c * W // P if split == 0 else
                                          np.where(c % 2 == 0, a, a + (b - a) * split // 256))
        p = np.arange(W, dtype=np.int64) if W <= 1 << 16 else np.unique(np.r_[
            np.random.default_rng(3).integers(0, W, 1 << 14), lo[1:-1] - 1, lo[1:-1], 0, W - 1])
        own = header("owner", p, W, P, split)
        assert (own >= 0).all() and (own < P).all()
        assert (lo[own] <= p).all() and (p < lo[own + 1]).all()
        assert (np.diff(lo)[own.min():own.max() + 1] >= 1).all(), W
