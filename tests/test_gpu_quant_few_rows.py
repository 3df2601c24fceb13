"""GPU parity of quantized products with few activation rows or few tiles: the
matrix-core kernels whose waves split the columns (gemm_r16_kernel up to 32
rows, gemm_ks_kernel above), at the edges of their tiles, units and rules."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import quant_host as qh
from gpu_util import Arena, capi, check, lib
from synapse_amd.gguf import BLOCK, Q4_0, Q4_K, Q5_0, Q6_K, Q8_0
from test_gpu_quant import matmul_q, random_blocks

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arena():
    a = Arena(256 << 20)
    yield a
    a.close()


# Rows: the last GEMV (2) and the first tile (3), one and two tiles of 16
# activation rows whole and cut, then 32 x 32 tiles (33 on). Weight rows: one,
# a tile less one, whole and one over; odd counts start rows off a dword
# (Q6_K). Columns: one unit (seven waves idle), one per wave, one more, and
# for the 32-block formats a last unit of two to six blocks, and one of 25
# blocks (odd: the kernels that copy whole units do not take it). Long rows of
# few weight rows, which the GEMV keeps in some formats, and their 16-row tiles.
CASES = [(2, 17, 512), (3, 1, 256), (3, 15, 2048), (5, 33, 2304), (15, 16, 768), (16, 31, 4096), (17, 16, 256),
         (24, 65, 14336), (31, 5, 2560), (32, 130, 1024), (33, 31, 256), (40, 33, 1280), (64, 65, 1024), (65, 32, 2048),
         (96, 7, 768), (3, 17, 64), (16, 15, 320), (20, 33, 448), (33, 9, 64), (40, 33, 192), (31, 20, 800),
         (33, 20, 800), (3, 40, 4352), (3, 1040, 4352), (16, 9, 6400), (16, 600, 6400), (31, 9, 8192)]


@pytest.mark.parametrize("t", [Q4_0, Q5_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("n,rows,cols", CASES)
def test_few_rows(arena, t, n, rows, cols):
    """Activation bytes are ggml's bit for bit; every output is within 1e-5 of
    sum |w| |x^| of the exact product (the block integers are exact: at most
    cols / 32 + 10 float combines, each of 3 roundings of 6e-8)."""
    if cols % BLOCK[t][0]:
        pytest.skip("cols not whole blocks")
    _check(arena, t, n, rows, cols)


# Around the counts of 32 x 32 tiles from which gemm_ks_kernel asks for more
# columns or gives way to the larger tiles (test_quant_plan.cpp pins which
# kernel each takes).
@pytest.mark.parametrize("t,rows,cols", [(Q4_K, 16384, 1024), (Q4_K, 16385, 1024), (Q6_K, 16384, 1024),
                                         (Q6_K, 16385, 1024), (Q4_K, 16, 768),
                                         (Q8_0, 32768, 64), (Q8_0, 32769, 64), (Q4_K, 12288, 1024),
                                         (Q4_K, 12289, 1024), (Q4_K, 12289, 3072), (Q8_0, 12288, 64),
                                         (Q8_0, 12289, 64), (Q8_0, 12289, 192), (Q5_0, 24576, 192),
                                         (Q5_0, 24576, 256)])
def test_tile_count_rule(arena, t, rows, cols):
    _check(arena, t, 33, rows, cols)


# 32 activation rows of many weight rows: the larger tiles, half of them empty.
@pytest.mark.parametrize("t,rows,cols", [(Q4_0, 32768, 64), (Q4_K, 32768, 256), (Q6_K, 131072, 256)])
def test_thirty_two_rows_of_many(arena, t, rows, cols):
    _check(arena, t, 32, rows, cols)


# The larger tiles (gemm_q4k_kernel, gemm_q6k_kernel, gemm_qb32_kernel), past
# the tile counts that gemm_ks_kernel takes: ten stages of 256 columns, or five
# of 64, so that both stage buffers are filled and read again; the last tiles
# hold one activation row and 104 (40) weight rows.
@pytest.mark.parametrize("t,n,cols", [(Q4_0, 2049, 320), (Q5_0, 2049, 320), (Q8_0, 2049, 320), (Q4_K, 1025, 2560),
                                      (Q6_K, 1025, 2560)])
def test_large_tiles(arena, t, n, cols):
    _check(arena, t, n, 1000, cols)


def _check(arena, t, n, rows, cols):
    rng = np.random.default_rng(100000 * t + 1000 * n + rows + cols)
    raw = random_blocks(t, rows, cols, rng)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    x[1, :64] = 0.0
    if n > 2:
        x[2] = 0.0  # zero blocks only
    bias = rng.standard_normal(rows).astype(np.float32)
    want_act = np.concatenate([qh.quantize_act(x[r], t) for r in range(n)])
    w = qh.dequantize(raw, t).reshape(rows, cols).astype(np.float64)
    xa = np.stack([qh.dequantize_act(a, qh.act_type(t)) for a in want_act.reshape(n, -1)]).astype(np.float64)
    exact, scale = xa @ w.T, np.abs(xa) @ np.abs(w).T
    for b in (None, bias):
        out, act = matmul_q(arena, raw, t, x, rows, cols, b) if b is not None else matmul_q(arena, raw, t, x, rows, cols)
        assert np.array_equal(act, want_act)
        got = out.astype(np.float64) - (0 if b is None else b)
        err = np.abs(got - exact)
        assert np.all(err <= 1e-5 * np.maximum(scale, 1.0)), float((err / np.maximum(scale, 1.0)).max())


@pytest.mark.parametrize("n", [24, 48])
def test_extreme_weights(arena, n):
    """Q6_K and Q4_K blocks whose quants and scales sit at the ends of their
    ranges against activations at +-127: the largest integers the folded
    weight planes and their sums can reach."""
    rows, cols = 32, 512
    rng = np.random.default_rng(n)
    for t in (Q6_K, Q4_K):
        blocks = random_blocks(t, rows, cols, rng).reshape(rows * cols // 256, -1)
        for i, blk in enumerate(blocks):
            if t == Q6_K:
                blk[:192] = 0xFF if i % 2 else 0x00     # q = 63 or 0
                blk[192:208] = 0x80 if i % 3 else 0x7F  # scale -128 or 127
            else:
                blk[4:] = 0xFF  # scale, min and quants all ones
        x = np.where(rng.random((n, cols)) < 0.5, -1.0, 1.0).astype(np.float32)
        x[: n // 2] = np.abs(x[: n // 2])
        raw = blocks.reshape(-1)
        out, _ = matmul_q(arena, raw, t, x, rows, cols)
        act = np.stack([qh.quantize_act(r, t) for r in x])
        w = qh.dequantize(raw, t).reshape(rows, cols).astype(np.float64)
        xa = np.stack([qh.dequantize_act(a, qh.act_type(t)) for a in act]).astype(np.float64)
        err = np.abs(out - xa @ w.T)
        assert np.all(err <= 1e-5 * np.maximum(np.abs(xa) @ np.abs(w).T, 1.0))


def test_more_rows_than_one_launch():
    """16-row tiles take 32 threads per weight row, which 2^27 rows are too
    many for: the GEMV does them."""
    t, n, rows, cols, last = Q4_0, 3, 1 << 27, 64, 40
    rng = np.random.default_rng(27)
    raw = random_blocks(t, last, cols, rng)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    wbytes = rows * (cols // 32) * BLOCK[t][1]
    with Arena(wbytes + n * rows * 4 + (1 << 20)) as a:
        wo = a.alloc(wbytes)
        a.fill(wo, 0, wbytes)
        a.upload(wo + wbytes - raw.nbytes, raw)
        xo, act = a.put(x), a.alloc(4096)
        oo = a.alloc(n * rows * 4)
        d = capi.MatmulQDesc(w_offset=wo, x_offset=xo, act_offset=act, bias_offset=capi.NO_OFFSET, out_offset=oo,
                             w_type=t, n=n, rows=rows, cols=cols)
        check(lib().syn_hip_matmul_q(a.handle, ctypes.byref(d)))
        w = qh.dequantize(raw, t).reshape(last, cols).astype(np.float64)
        for r in range(n):
            xa = qh.dequantize_act(qh.quantize_act(x[r], t), qh.act_type(t)).astype(np.float64)
            got = a.download(oo + 4 * ((r + 1) * rows - 2 * last), (2 * last,), np.float32)
            assert not got[:last].any()
            assert np.all(np.abs(got[last:] - w @ xa) <= 1e-5 * np.maximum(np.abs(w) @ np.abs(xa), 1.0))
