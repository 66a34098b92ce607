"""Batched matvec on the matrix cores (2-32 activation rows per pass).

Bound: x is rounded once, by at most 2^-31 of its 32-element block's largest
magnitude rounded up to a power of two (at most twice that magnitude); all sums
are integers or double, and the result is rounded once to fp32:
|y - exact| <= 2^-24 |exact| + 2^-30 sum_blocks max|x_b| sum|w_b|.  The exact sum
here is of the reference's element values, which are rounded to fp32 (2^-24 of
each); the kernel's are not: 2^-24 sum |w x| more, which also covers the double
sums' own rounding.  Q6_K rows of an odd block count take the byte-addressed
kernel, whose sums are fp32: chains of 16 elements, of at most K / 1024 + 1 such
groups a lane and of 6 steps across the lanes, each step rounding by at most
2^-24 sum |w x|.
"""
import numpy as np
import pytest
import torch

import ssdq
import ssdq_oracle as o
from helpers import announce, empty_dev, from_dev, to_dev
from ssdq import synth

pytestmark = pytest.mark.gpu

Q4_0, Q8_0, Q4_K, Q6_K = ssdq.Q4_0, ssdq.Q8_0, ssdq.Q4_K, ssdq.Q6_K

CASES = [  # (dtype, out_dim, in_dim, batch)
    # one unit; a partial group of 16 rows; both sides of every row count the kernel is built for
    (Q4_K, 1, 256, 2), (Q6_K, 15, 256, 4), (Q4_0, 17, 256, 5), (Q8_0, 33, 256, 8),
    (Q4_K, 300, 1024, 9), (Q6_K, 300, 1024, 16), (Q4_0, 300, 1024, 17), (Q8_0, 300, 1024, 32),
    # odd numbers of Q6_K blocks, which stay on the byte-addressed kernel
    (Q6_K, 7, 768, 3), (Q6_K, 1001, 1280, 6),
    # few rows: one slice below 64 row units, more from there on (Q6_K: from 16 units on)
    (Q4_K, 500, 4096, 3), (Q4_K, 500, 4096, 4), (Q6_K, 500, 3840 + 256, 2), (Q6_K, 500, 3584, 2), (Q4_0, 20, 2048, 16),
    # uneven units per wave and uneven K slices (9 and 33 units, 43 units at 8 / 32 rows)
    (Q4_K, 4097, 2304, 8), (Q4_0, 100, 8448, 4), (Q8_0, 100, 8448, 2), (Q4_K, 513, 11008, 7), (Q6_K, 129, 11008, 31),
    # more groups than waves (one wave walks several groups), chunks of 32 and a rest, a last single row
    (Q4_K, 70000, 512, 4), (Q8_0, 50001, 256, 32), (Q4_0, 64, 512, 33), (Q6_K, 64, 512, 42),
    # a row length that is not whole K-quant blocks
    (Q4_K, 64, 1024 + 64, 8),
]


def close_to_exact(y, dtype, w, x, out_dim, in_dim):
    e, _ = o.matvec_elements(dtype, w, out_dim, in_dim)
    e = e.astype(np.float64)
    k = e.shape[1]
    x = x.astype(np.float64)[:, :k]
    exact = x @ e.T
    mx = np.repeat(np.abs(x).reshape(len(x), k // 32, 32).max(axis=2), 32, axis=1)
    bound = 2.0 ** -24 * np.abs(exact) + 2.0 ** -30 * (mx @ np.abs(e).T) + 2.0 ** -24 * (np.abs(x) @ np.abs(e).T)
    if dtype == Q6_K and k // 256 % 2:
        bound += 2.0 ** -24 * (16 + k // 1024 + 1 + 6) * (np.abs(x) @ np.abs(e).T)
    err = np.abs(y.astype(np.float64).reshape(exact.shape) - exact)
    assert np.all(err <= bound), f"worst error / bound {np.nanmax(err / np.maximum(bound, 1e-300))}"


@pytest.mark.parametrize("dtype,out_dim,in_dim,batch", CASES)
def test_batch(dtype, out_dim, in_dim, batch):
    w = synth.quant_weights(dtype, out_dim, in_dim, 7000 + out_dim + batch)
    g = synth.rng(7001 + in_dim)
    x = g.standard_normal((batch, in_dim)).astype(np.float32)
    x[:, g.integers(0, in_dim, 4)] *= 100  # units of different ranges
    x[0, :256] = 0
    announce("batch", dtype, out_dim, in_dim, batch)
    y = empty_dev(out_dim * batch, torch.float32)
    assert ssdq.matvec(dtype, to_dev(w), to_dev(x), y, out_dim, in_dim, batch) == 0
    close_to_exact(from_dev(y), dtype, w, x, out_dim, in_dim)


@pytest.mark.parametrize("dtype,lo,hi", [(Q4_K, 4, 16), (Q6_K, 192, 208)])
def test_batch_extreme_scales(dtype, lo, hi):
    # every scale byte at its ends: the products s q reach the ends of the signed bytes they are split into
    out_dim, in_dim, batch = 48, 1024, 8
    w = synth.quant_weights(dtype, out_dim, in_dim, 7100).reshape(-1, synth.BLOCK[dtype][1])
    ends = np.array([0x80, 0x7F, 0xFF, 0x00, 0x3F, 0xC0], np.uint8)
    w[:, lo:hi] = ends[synth.rng(7101).integers(0, len(ends), (len(w), hi - lo))]
    w[::3, 16 if dtype == Q4_K else 0:144 if dtype == Q4_K else 192] = 0xFF
    w[1::3, 16 if dtype == Q4_K else 0:144 if dtype == Q4_K else 192] = 0
    w = w.ravel()
    x = np.where(synth.rng(7102).random((batch, in_dim)) < 0.5, -1.0, 1.0).astype(np.float32) * np.float32(1.99)
    announce("batch extreme scales", dtype)
    y = empty_dev(out_dim * batch, torch.float32)
    assert ssdq.matvec(dtype, to_dev(w), to_dev(x), y, out_dim, in_dim, batch) == 0
    close_to_exact(from_dev(y), dtype, w, x, out_dim, in_dim)


def without_weight(dtype, w):
    """w with a zero weight for the first element of every 256 (and, Q4_K, no minima)."""
    b = w.reshape(-1, synth.BLOCK[dtype][1]).copy()
    if dtype == Q4_0:
        b[::8, 2] = (b[::8, 2] & 0xF0) | 8
    elif dtype == Q8_0:
        b[::8, 2] = 0
    elif dtype == Q4_K:
        b[:, 2:4] = 0
        b[:, 16] &= 0xF0
    else:
        b[:, 0] &= 0xF0
        b[:, 128] = (b[:, 128] & 0xFC) | 2
    return b.ravel()


@pytest.mark.parametrize("dtype", [Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("batch", [2, 8, 13, 32])
@pytest.mark.parametrize("large", [3e7, 1e20])
def test_batch_large_channel_without_weight(dtype, batch, large):
    # a channel far above the rest of its 256 elements, and of no weight: the blocks it is not in keep their precision
    out_dim, in_dim = 100, 1024
    w = without_weight(dtype, synth.quant_weights(dtype, out_dim, in_dim, 7400))
    x = synth.normal_f32((batch, in_dim), 7401).reshape(batch, in_dim).copy()
    x[:, ::256] = large
    x[:, 1:32] = x[:, 257:288] = x[:, 513:544] = x[:, 769:800] = 0  # its own block
    announce("batch large channel", dtype, batch, large)
    y = empty_dev(out_dim * batch, torch.float32)
    assert ssdq.matvec(dtype, to_dev(w), to_dev(x), y, out_dim, in_dim, batch) == 0
    x[:, ::256] = 0
    close_to_exact(from_dev(y), dtype, w, x, out_dim, in_dim)


def test_batch_nonfinite_rows():
    out_dim, in_dim, batch = 40, 512, 6
    w = synth.quant_weights(Q4_K, out_dim, in_dim, 7200)
    x = synth.normal_f32((batch, in_dim), 7201)
    x[1, 300], x[3, 5], x[4, 511] = np.nan, np.inf, -np.inf
    x[5] *= np.float32(1e-37)
    announce("batch non-finite rows")
    y = empty_dev(out_dim * batch, torch.float32)
    assert ssdq.matvec(Q4_K, to_dev(w), to_dev(x), y, out_dim, in_dim, batch) == 0
    y = from_dev(y).reshape(batch, out_dim)
    assert np.isnan(y[[1, 3, 4]]).all()
    ok = [0, 2]
    close_to_exact(y[ok], Q4_K, w, x[ok], out_dim, in_dim)
    exact = x[5:].astype(np.float64) @ o.matvec_elements(Q4_K, w, out_dim, in_dim)[0].astype(np.float64).T
    assert np.all(np.abs(y[5] - exact[0]) <= 1e-3 * np.abs(exact).max())


def test_batch_captured_without_workspace():
    # 32 rows of K = 4096 want K slices; a stream that is captured before it has a
    # workspace takes chunks of 8 rows, which need none
    out_dim, in_dim, batch = 256, 4096, 32
    w = synth.quant_weights(Q8_0, out_dim, in_dim, 7300)
    x = synth.normal_f32((batch, in_dim), 7301)
    wd, xd, y = to_dev(w), to_dev(x), empty_dev(out_dim * batch, torch.float32)
    ssdq.matvec(Q8_0, wd, xd, y, out_dim, in_dim, 2)  # the kernel is loaded
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    announce("batch captured without workspace")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        ssdq.matvec(Q8_0, wd, xd, y, out_dim, in_dim, batch, stream=side)
    for rep in range(3):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        close_to_exact(from_dev(y), Q8_0, w, x, out_dim, in_dim)
