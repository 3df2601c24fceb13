"""GPU parity of RMSNorm and the element-wise ops at the edges of their vector
forms: row lengths at each form's limit, lengths and offsets that are not
whole 16-byte chunks, in place."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from gpu_util import Arena, capi, check, lib
from synapse_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arena():
    a = Arena(128 << 20)
    yield a
    a.close()


def _put(arena, x, shift):
    """x at an offset `shift` floats past a 256-byte line."""
    off = arena.alloc(x.nbytes + 4 * shift + 256) + 4 * shift
    arena.upload(off, x)
    return off


@pytest.mark.parametrize("n,size", [(1, 1), (1, 4), (3, 7), (1, 896), (2, 1024), (2, 1028), (1, 4096), (2, 4100),
                                    (1, 16384), (1, 16388), (300, 4096), (5, 4095)])
@pytest.mark.parametrize("shift", [0, 1])
def test_rms_norm(arena, n, size, shift):
    g = wl.rng(n + size)
    x, gamma = wl.normal(g, (n, size)), wl.normal(g, (size,))
    eps = 1e-5
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 * x64).mean(-1, keepdims=True) + eps) * gamma
    mark = arena.top
    for in_place in (False, True):
        xo = _put(arena, x, shift)
        oo = xo if in_place else _put(arena, np.full((n, size), 9.0, np.float32), shift)
        d = capi.NormDesc(in_offset=xo, weight_offset=_put(arena, gamma, shift), out_offset=oo, n=n, size=size, eps=eps)
        check(lib().syn_hip_rms_norm(arena.handle, ctypes.byref(d)))
        got = arena.download(oo, (n, size), np.float32)
        # Six f32 roundings on the way (square, mean, + eps, root, quotient
        # and two products; the square's and mean's count half).
        assert np.all(np.abs(got - want) <= 6 * 2.0 ** -24 * np.abs(want))
    arena.top = mark


OPS = {"add": capi.SYN_ADD, "mul": capi.SYN_MUL, "silu_mul": capi.SYN_SILU_MUL, "scale": capi.SYN_SCALE,
       "gelu": capi.SYN_GELU, "silu": capi.SYN_SILU, "add_bias": capi.SYN_ADD_BIAS}


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("rows,period", [(1, 1), (1, 3), (3, 4), (7, 6), (5, 1024), (1, 14336), (301, 4096)])
@pytest.mark.parametrize("shift", [0, 1])
def test_elementwise(arena, op, rows, period, shift):
    _check_elementwise(arena, op, rows, period, shift, shift, shift)


# One operand alone off a 16-byte offset (a, b or the result), then more than
# 4096 blocks of four floats a thread: a second trip of the vector form's grid,
# with a bias period that is no power of two.
@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("rows,period,shifts", [(9, 1028, (1, 0, 0)), (9, 1028, (0, 1, 0)), (9, 1028, (0, 0, 1)),
                                                (301, 14340, (0, 0, 0))])
def test_elementwise_offsets_and_second_trip(arena, op, rows, period, shifts):
    _check_elementwise(arena, op, rows, period, *shifts)


def _check_elementwise(arena, op, rows, period, shift_a, shift_b, shift_out):
    g = wl.rng(rows + period)
    a = wl.normal(g, (rows, period), 3.0)
    b = wl.normal(g, (period,) if op == "add_bias" else (rows, period))
    mark = arena.top
    ao, bo = _put(arena, a, shift_a), _put(arena, b, shift_b)
    oo = _put(arena, np.full(rows * period + 8, 7.0, np.float32), shift_out)
    d = capi.ElementwiseDesc(a_offset=ao, b_offset=bo, out_offset=oo, count=rows * period, op=OPS[op], scalar=1.7,
                             period=period)
    check(lib().syn_hip_elementwise(arena.handle, ctypes.byref(d)))
    got = arena.download(oo, (rows * period + 8,), np.float32)
    arena.top = mark
    assert (got[rows * period:] == 7.0).all()
    got = got[:rows * period].reshape(rows, period)
    a64 = a.astype(np.float64)
    sig = a64 / (1 + np.exp(-a64))
    if op in ("add", "add_bias", "mul", "scale"):
        want = a + b if op[:3] == "add" else (a * b if op == "mul" else a * np.float32(1.7))
        assert np.array_equal(got, want)
    elif op == "gelu":
        h = a.astype(np.float16).astype(np.float64)
        want = 0.5 * h * (1 + np.tanh(0.79788456080286535588 * h * (1 + 0.044715 * h * h)))
        # rounded to binary16, from f32 arithmetic that cancels near -4
        assert np.all(np.abs(got - want) <= 2.0 ** -10 * np.abs(want) + 1e-6)
    else:
        want = sig * b if op == "silu_mul" else sig
        # expf within 2 ulp, then a sum, a quotient and a product
        assert np.all(np.abs(got - want) <= 6 * 2.0 ** -24 * np.abs(want) + 1e-37)
