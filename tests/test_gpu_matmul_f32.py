"""GPU parity of the F32 product (matmul_f32.hip) against float64, at the
edges of its tiles and of the rules that choose between its kernels."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from gpu_util import Arena, capi, check, lib
from synapse_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arena():
    a = Arena(256 << 20)
    yield a
    a.close()


# Few rows (one wave per weight row; any column count, row starts on any
# dword), the last such and the first on the matrix cores (8 rows and
# n rows >= 40000), then 32 x 32, 32 x 64 and 64 x 64 tiles: whole, one row or
# one column chunk over, one stage, a partial last stage, the longest row the
# interface takes, columns that are no
# whole chunks; with and without bias.
@pytest.mark.parametrize("n,rows,cols", [(1, 1, 1), (1, 5, 3), (1, 70, 1025), (1, 33, 2048), (2, 9, 64), (7, 70, 65),
                                         (1, 9, 256), (5, 9, 257), (3, 6, 512), (4, 6, 513), (2, 9, 300), (3, 9, 257),
                                         (4, 40, 768), (7, 6000, 36), (15, 34, 5632), (8, 4999, 64), (8, 5000, 64),
                                         (40, 1000, 4), (40, 1000, 130), (52, 770, 132), (64, 768, 3072),
                                         (257, 768, 768), (100, 9000, 36), (385, 2050, 260), (1000, 1030, 128),
                                         (1024, 2048, 100), (1025, 2049, 64), (1, 3, 119167), (64, 640, 20000)])
def test_matmul_f32(arena, n, rows, cols):
    g = wl.rng(7 * n + rows + cols)
    w, x, b = wl.normal(g, (rows, cols)), wl.normal(g, (n, cols)), wl.normal(g, (rows,))
    exact = x.astype(np.float64) @ w.T.astype(np.float64)
    mark = arena.top
    arena.alloc(4, 4)  # w starts 4 bytes past a 256-byte line
    wo, xo, bo = arena.put(w, 4), arena.put(x, 4), arena.put(b, 4)
    guard = np.full(rows * n + 64, 7.0, np.float32)
    oo = arena.put(guard, 4)
    for bias in (False, True):
        d = capi.MatmulDesc(w_offset=wo, x_offset=xo, bias_offset=bo if bias else capi.NO_OFFSET, out_offset=oo, n=n,
                            rows=rows, cols=cols)
        check(lib().syn_hip_matmul(arena.handle, ctypes.byref(d)))
        got = arena.download(oo, (rows * n + 64,), np.float32)
        assert (got[rows * n:] == 7.0).all()
        want = exact + b.astype(np.float64) if bias else exact
        # Each product passes through at most 32 sums of its stage (of 32 to
        # 128 columns), then one per stage, 3 across the waves and the bias.
        depth = 36 + (cols + 31) // 32
        bound = depth * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + np.abs(b)).astype(np.float64) * 1.01
        assert (np.abs(got[:rows * n].reshape(n, rows) - want) <= bound).all()
    arena.top = mark
