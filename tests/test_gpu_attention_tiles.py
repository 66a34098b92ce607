"""Edges of the decode-attention tiles and splits against the oracle.

Paged: 32-token tiles, two in flight, splits of whole tiles.  Flat f32: 16
tokens per wave and step, 8 waves per workgroup, up to 8 query heads together.
"""
import numpy as np
import pytest
import torch

import ssdq
import ssdq_oracle as o
from helpers import announce, assert_close, empty_dev, from_dev, to_dev
from test_gpu_attention import paged_case, run_paged

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_head,n_kv,hd,ctx", [
    (32, 8, 128, [1, 31, 32, 33, 63, 64, 65, 96, 97, 129]),
    (16, 4, 64, [2, 95, 1, 160, 161]),
    (8, 4, 256, [33, 64, 127]),
    (5, 1, 128, [40, 700]),        # five heads: two chunks, the second of one head
    (4, 4, 128, [1500, 20, 1037]),  # one head per KV head, several splits, ragged
    (32, 8, 128, [3000, 100, 1, 2999, 640]),  # halved splits, empty ones past the short sequences
])
def test_paged_tiles(n_head, n_kv, hd, ctx):
    bs, n = 16, len(ctx)
    mb = -(-max(ctx) // bs)
    announce("paged tiles", n_head, n_kv, hd, ctx)
    q, kc, ks, vc, vs, tables, cl = paged_case(n, n_head, n_kv, hd, bs, ctx, mb, 31 + n_head)
    got, rc = run_paged(q, kc, ks, vc, vs, tables, cl, n, n_head, n_kv, hd, bs, mb)
    assert rc == 0
    ref = o.paged_attention_int8(q, kc, ks, vc, vs, tables, cl, n, n_head, n_kv, hd, bs, mb, threads=8)
    assert_close(got, ref, "paged tiles")


def test_paged_value_scales_of_all_sizes():
    # rows of very different scales in one tile
    n_head, n_kv, hd, bs, ctx = 8, 2, 128, 16, [100]
    q, kc, ks, vc, vs, tables, cl = paged_case(1, n_head, n_kv, hd, bs, ctx, 7, 77)
    vs = np.asarray(vs) * np.float32(10.0) ** np.resize(np.arange(-6, 3), np.asarray(vs).shape).astype(np.float32)
    vs = vs.astype(np.float32)
    announce("paged value scales")
    got, _ = run_paged(q, kc, ks, vc, vs, tables, cl, 1, n_head, n_kv, hd, bs, 7)
    ref = o.paged_attention_int8(q, kc, ks, vc, vs, tables, cl, 1, n_head, n_kv, hd, bs, 7)
    assert_close(got, ref, "paged value scales")


def paged_softmax(q, kc, ks, tables, bs, ctx, n_kv):
    """Weights of sequence 0's tokens [n_head, ctx] and their pool rows, in float64."""
    hd = q.shape[2]
    rows = tables.reshape(-1)[np.arange(ctx) // bs] * bs + np.arange(ctx) % bs
    k = (kc.reshape(-1, n_kv, hd)[rows].astype(np.float64) * ks[rows].astype(np.float64)[:, None, None])
    s = np.stack([k[:, h * n_kv // q.shape[1]] @ q[0, h].astype(np.float64) for h in range(q.shape[1])]) / np.sqrt(hd)
    p = np.exp(s - s.max(axis=1, keepdims=True))
    return p / p.sum(axis=1, keepdims=True), rows


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("ctx", [31, 64, 200])
def test_paged_dimensions_of_low_weight_tokens(hd, ctx):
    """Dimensions in which every token of more than 2^-35 of the largest weight has
    value code 0 keep fp32's relative precision.  Bound, relative to sum p |v| of
    the dimension: scores of magnitude up to 64 take four fp32 roundings (and so
    does the largest, subtracted from them), which the exponential turns into
    2 x 64 x 4 x 2^-24 = 3.1e-5; its own error, the sums' and the final division's
    add less than 2e-6."""
    n_head, n_kv, bs, mb = 4, 1, 16, 13
    q, kc, ks, vc, vs, tables, cl = paged_case(1, n_head, n_kv, hd, bs, [ctx], mb, 90 + hd)
    q[0, 1:] = q[0, :1] * np.array([0.9, 1.05, 1.1], np.float32)[:, None]  # one order of the tokens for all heads
    p, rows = paged_softmax(q, kc, ks, tables, bs, ctx, n_kv)
    q *= np.float32(40 / (np.log(p[0].max()) - np.log(np.median(p[0]))))
    p, rows = paged_softmax(q, kc, ks, tables, bs, ctx, n_kv)
    v = vc.reshape(-1, hd)
    heavy = (p > 2.0 ** -35 * p.max(axis=1, keepdims=True)).any(axis=0)
    assert 0 < heavy.sum() < ctx
    dims = np.arange(0, hd, 3)
    v[np.ix_(rows[heavy], dims)] = 0
    announce("paged dimensions of low-weight tokens", hd, ctx)
    got, _ = run_paged(q, kc, ks, v.reshape(-1), vs, tables, cl, 1, n_head, n_kv, hd, bs, mb)
    vf = v[rows].astype(np.float64) * vs[rows].astype(np.float64)[:, None]
    exact, size = p @ vf, p @ np.abs(vf)
    assert size[:, dims].max() < 1e-6 and size[:, dims].min() > 0
    err = np.abs(got.reshape(n_head, hd) - exact) / size
    assert err.max() < 3.3e-5, err.max()


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("ctx,at", [(70, 3), (70, 69), (64, 63), (33, 32)])
def test_paged_infinite_value_scale(hd, ctx, at):
    # an infinite scale gives its token's codes their infinities, also where a ragged tile repeats the last token
    n_head, n_kv, bs, mb = 4, 1, 16, 5
    q, kc, ks, vc, vs, tables, cl = paged_case(1, n_head, n_kv, hd, bs, [ctx], mb, 95)
    row = int(tables.reshape(-1)[at // bs]) * bs + at % bs
    v = vc.reshape(-1, hd)
    v[row] = np.where(np.arange(hd) % 2, 100, -7)
    vs = vs.copy()
    vs[row] = np.inf
    announce("paged infinite value scale", hd, ctx, at)
    got, _ = run_paged(q, kc, ks, v.reshape(-1), vs, tables, cl, 1, n_head, n_kv, hd, bs, mb)
    want = np.where(np.arange(hd) % 2, np.inf, -np.inf)
    assert (got.reshape(n_head, hd) == want).all()


@pytest.mark.parametrize("ctx", [[3000, 100, 1, 0], [20000, 30, 6000]])
def test_paged_records_of_an_earlier_call(ctx):
    # short sequences have no records for the later splits: what an earlier call left there (infinities and NaN) is
    # loaded with the rest and must not count
    n_head, n_kv, hd, bs, n = 8, 2, 128, 16, len(ctx)
    mb = -(-max(ctx) // bs)
    q, kc, ks, vc, vs, tables, cl = paged_case(n, n_head, n_kv, hd, bs, ctx, mb, 98)
    announce("paged records of an earlier call", ctx)
    bad = np.where(np.arange(vs.size) % 2, np.nan, np.inf).astype(np.float32)
    run_paged(q, kc, ks, vc, bad, tables, np.full(n, max(ctx), np.int32), n, n_head, n_kv, hd, bs, mb)
    got, _ = run_paged(q, kc, ks, vc, vs, tables, cl, n, n_head, n_kv, hd, bs, mb)
    ref = o.paged_attention_int8(q, kc, ks, vc, vs, tables, cl, n, n_head, n_kv, hd, bs, mb, threads=8)
    assert_close(got, ref, "paged records of an earlier call")


@pytest.mark.parametrize("n_head,n_kv,hd", [(4, 4, 128), (32, 8, 128), (10, 2, 128), (16, 1, 64), (3, 3, 256), (8, 2, 256)])
@pytest.mark.parametrize("lo,hi", [(0, 1), (0, 127), (0, 128), (0, 129), (5, 20), (17, 1500), (700, 700)])
def test_flash_tiles(n_head, n_kv, hd, lo, hi):
    seq = max(hi, 1)
    g = np.random.default_rng(hd + hi)
    q = g.standard_normal((n_head, hd), dtype=np.float32)
    k = g.standard_normal((seq, n_kv, hd), dtype=np.float32)
    v = g.standard_normal((seq, n_kv, hd), dtype=np.float32)
    out = empty_dev(n_head * hd, torch.float32)
    announce("flash tiles", n_head, n_kv, hd, lo, hi)
    ssdq.flash_attention_f32(to_dev(q), to_dev(k), to_dev(v), out, n_head, n_kv, hd, seq, lo, hi)
    assert_close(from_dev(out), o.flash_attention_f32(q, k, v, n_head, n_kv, hd, seq, lo, hi), "flash tiles")


@pytest.mark.parametrize("n_head,n_kv,hd,seq", [(8, 2, 128, 5), (4, 4, 64, 130), (8, 2, 256, 31)])
def test_flash_infinite_value_of_the_last_token(n_head, n_kv, hd, seq):
    # ragged steps repeat the last token, the combine the last split, with weight 0: an infinity in them must not
    # turn into NaN
    g = np.random.default_rng(seq)
    q = g.standard_normal((n_head, hd), dtype=np.float32)
    k = g.standard_normal((seq, n_kv, hd), dtype=np.float32)
    v = g.standard_normal((seq, n_kv, hd), dtype=np.float32)
    v[-1, :, 3], v[-1, :, hd - 1] = np.inf, -np.inf
    out = empty_dev(n_head * hd, torch.float32)
    announce("flash infinite value", n_head, n_kv, hd, seq)
    ssdq.flash_attention_f32(to_dev(q), to_dev(k), to_dev(v), out, n_head, n_kv, hd, seq, 0, seq)
    got = from_dev(out).reshape(n_head, hd)
    assert (got[:, 3] == np.inf).all() and (got[:, hd - 1] == -np.inf).all()
    rest = [d for d in range(hd) if d not in (3, hd - 1)]
    v[-1, :, 3] = v[-1, :, hd - 1] = 0
    ref = o.flash_attention_f32(q, k, v, n_head, n_kv, hd, seq, 0, seq).reshape(n_head, hd)
    assert_close(got[:, rest], ref[:, rest], "flash infinite value")
