"""GPU parity of image-encoder attention on f32 rows: the f32 matrix-core
kernel (flash_f32.hip) at the edges of its tiles, and the row-per-wave kernel
(generic.hip) for head sizes that are not whole 16-byte chunks, against the
oracle."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import binding as orc
from gpu_util import SYN_F32, Arena, SelfDesc, check, lib, self_attention
from synapse_amd import workloads as wl

pytestmark = pytest.mark.gpu

# Of the largest output: both sides sum in f32 (hd terms, then n), and each
# f32 rounding of a random sum's partial is at most 6e-8 of it.
BOUND = 2e-6


@pytest.fixture(scope="module")
def arena():
    a = Arena(256 << 20)
    yield a
    a.close()


# Keys go to the four waves in whole 16-row tiles, two per step: rows below,
# at and above 1, 4 and 8 tiles, and a wave left without keys (n = 130 with 3
# tiles a wave). Head sizes: one chunk, each group of the output's tiles (16,
# 32, 64 dims) whole and cut, both ends of every compiled size, and 6 (the
# row-per-wave kernel). The last line: either side of what that kernel keeps of
# the tiny heads (160 floats of a head, 1536 rows in all).
@pytest.mark.parametrize("n,batch,heads,hd", [(1, 1, 1, 64), (15, 2, 3, 64), (16, 1, 1, 64), (17, 3, 1, 64),
                                              (63, 1, 2, 64), (65, 2, 2, 64), (128, 1, 3, 64), (130, 1, 3, 64),
                                              (257, 2, 9, 64), (729, 1, 2, 72), (40, 1, 2, 4), (40, 1, 2, 12),
                                              (40, 2, 2, 32), (70, 1, 2, 36), (70, 1, 3, 80), (70, 1, 2, 84),
                                              (70, 1, 2, 96), (70, 1, 2, 100), (70, 1, 2, 128), (70, 1, 2, 132),
                                              (70, 1, 2, 192), (70, 1, 2, 196), (70, 1, 2, 256), (70, 1, 2, 6),
                                              (40, 2, 16, 4), (41, 2, 16, 4), (32, 3, 16, 4),
                                              (33, 3, 16, 4), (20, 1, 3, 8), (21, 1, 3, 8), (13, 4, 2, 12),
                                              (14, 4, 2, 12), (8, 1, 2, 16)])
def test_image_f32(arena, n, batch, heads, hd):
    g = wl.rng(1000 * hd + n)
    q, k, v = (wl.normal(g, (batch * n, heads * hd)) for _ in range(3))
    scale = float(np.float32(1) / np.sqrt(np.float32(hd)))
    got = self_attention(arena, q, k, v, n, batch, heads, scale, SYN_F32)
    for b in range(batch):
        sl = slice(b * n, (b + 1) * n)
        want = orc.self_attention(q[sl], k[sl], v[sl], heads, scale, threads=8)
        assert np.abs(got[sl] - want).max() <= BOUND * np.abs(want).max(), b


def test_image_f32_extreme_scores(arena):
    """Scores far apart and rising along the keys (every step moves the max),
    one key that outweighs the rest, and a row of NaN: as the oracle."""
    n, heads, hd = 150, 2, 64
    g = wl.rng(5)
    q, k, v = (wl.normal(g, (n, heads * hd)) for _ in range(3))
    k *= np.linspace(0.1, 30, n, dtype=np.float32)[:, None]
    q[3] *= 100
    q[7] = np.nan
    got = self_attention(arena, q, k, v, n, 1, heads, 0.125, SYN_F32)
    want = orc.self_attention(q, k, v, heads, 0.125, threads=8)
    assert np.isnan(got[7]).all()
    rows = np.arange(n) != 7
    # A score of size s carries an error of s * 2^-24 * sqrt(hd) at most,
    # which its exponential shows as a relative error: each row and head is
    # held to its own largest score.
    heads_of = lambda x: x[rows].reshape(-1, heads, hd)  # noqa: E731
    top = np.abs(np.einsum("qhd,khd->qhk", heads_of(q).astype(np.float64), k.reshape(n, heads, hd)) * 0.125).max(-1)
    err = np.abs(heads_of(got) - heads_of(want)).max(-1)
    assert np.all(err <= np.maximum(BOUND, top * 2.0 ** -24 * 8) * np.abs(heads_of(want)).max(-1))


@pytest.mark.parametrize("at", range(4))
def test_image_f32_offsets(arena, at):
    """Rows of 12-dim heads on 4-byte offsets, as the interface takes them."""
    n, heads, hd = 40, 2, 12
    g = wl.rng(at)
    rows = [wl.normal(g, (n, heads * hd)) for _ in range(3)]
    mark = arena.top
    offs = [arena.alloc(n * heads * hd * 4 + 256) for _ in range(4)]
    offs[at] += 4
    for off, x in zip(offs, rows):
        arena.upload(off, x)
    d = SelfDesc(q_offset=offs[0], k_offset=offs[1], v_offset=offs[2], out_offset=offs[3], n=n, batch=1, n_heads=heads,
                 head_dim=hd, scale=0.25, in_dtype=SYN_F32)
    check(lib().syn_hip_self_attention(arena.handle, ctypes.byref(d)))
    got = arena.download(offs[3], (n, heads * hd), np.float32)
    want = orc.self_attention(*rows, heads, 0.25, threads=8)
    assert np.abs(got - want).max() <= BOUND * np.abs(want).max()
    arena.top = mark


def test_image_f32_many_small_images():
    """More 16-row tiles than one launch dimension takes in blocks of 256
    threads: one key each, so the output is v."""
    batch, heads, hd = 65535, 257, 4
    assert batch * heads >= 2 ** 24
    x = np.arange(batch * heads * hd, dtype=np.float32).reshape(batch, heads * hd) % 8191
    with Arena(3 * x.nbytes) as a:
        off, out = a.put(x), a.alloc(x.nbytes)
        d = SelfDesc(q_offset=off, k_offset=off, v_offset=off, out_offset=out, n=1, batch=batch, n_heads=heads,
                     head_dim=hd, scale=2.0 ** -30, in_dtype=SYN_F32)
        check(lib().syn_hip_self_attention(a.handle, ctypes.byref(d)))
        assert np.array_equal(a.download(out, x.shape, np.float32), x)
