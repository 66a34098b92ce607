"""The launch shapes of the extra types' matvec: groups requested ahead or not,
workgroups of 4, 8 and 16 waves, with ragged row counts.

A row's sum runs over its own groups in one order whatever the launch, so every
row of the whole call must equal, bit for bit, the same row from a call of 64
rows, and those are held to the exact sum of the oracle's element values with the
matvec tolerance of the other files (1e-4 + 1e-3 |exact|: about 16 times the
rounding of 28672 fp32 products of this size summed over 64 lanes, 2^-24 * sqrt(K)
* 0.5 being 5e-6).
"""
import numpy as np
import pytest
import torch

import ssdq
import ssdq_oracle as o
from helpers import ATOL, RTOL, announce, empty_dev, from_dev, to_dev
from ssdq import synth

pytestmark = pytest.mark.gpu


def call(dtype, w, x, out_dim, in_dim, batch):
    y = empty_dev(out_dim * batch, torch.float32)
    ssdq.matvec(dtype, w, x, y, out_dim, in_dim, batch)
    return from_dev(y).reshape(batch, out_dim)


@pytest.mark.parametrize("dtype,out_dim,in_dim,batch", [
    (ssdq.IQ4_XS, 10243, 4096, 1),   # eight workgroups per CU, one group at a time
    (ssdq.IQ4_XS, 1021, 4096, 1),    # few rows: requested ahead
    (ssdq.IQ4_XS, 3, 4352, 1),       # 136 groups: a last walk of 8 lanes
    (ssdq.IQ4_XS, 8201, 14336, 1),   # two workgroups of 8 waves per CU
    (ssdq.IQ4_XS, 8200, 28672, 1),   # one of 16 waves
    (ssdq.IQ4_XS, 4099, 4096, 8),    # 8 waves, one row each
    (ssdq.BF16, 8195, 14336, 1),
    (ssdq.IQ4_NL, 8195, 14336, 1),   # paired groups, 8 waves
    (ssdq.IQ3_S, 8195, 14336, 1),
    (ssdq.F16, 2051, 4096, 8),
    (ssdq.BF16, 4601, 4096, 4),      # 5 waves, 9 rows a place
    (ssdq.IQ3_S, 7001, 4096, 4),     # 7 waves
    (ssdq.IQ4_XS, 9001, 14336, 1),   # 5 waves of two rows, 18 rows a place
    (ssdq.BF16, 1021, 4096, 2),      # two rows: requested ahead
    (ssdq.BF16, 4099, 4096, 2),      # too many rows for that
    (ssdq.IQ4_XS, 1021, 4352, 2),    # lanes stop at their own last group, 136 groups
])
def test_rows_do_not_depend_on_the_launch(dtype, out_dim, in_dim, batch):
    announce("matvec ext rows", ssdq.TYPE_NAMES[dtype], out_dim, in_dim, batch)
    rng = np.random.default_rng(out_dim)
    rb = ssdq.row_bytes(dtype, in_dim)
    some = synth.quant_weights(dtype, min(out_dim, 64), in_dim, out_dim)
    w = np.resize(some.reshape(-1, rb), (out_dim, rb))       # rows repeat every 64
    x = rng.standard_normal((batch, in_dim)).astype(np.float32)
    wd, xd = to_dev(w.reshape(-1)), to_dev(x.reshape(-1))
    y = call(dtype, wd, xd, out_dim, in_dim, batch)
    n = min(out_dim, 64)
    few = call(dtype, wd[: n * rb].clone(), xd, n, in_dim, batch)
    assert np.array_equal(y, few[:, np.arange(out_dim) % n])
    exact = np.stack([o.matvec_exact(dtype, some, x[b], n, in_dim) for b in range(batch)])
    assert np.all(np.abs(few - exact) <= ATOL + RTOL * np.abs(exact))
