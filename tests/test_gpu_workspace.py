"""The library's per-stream workspace under HIP graph capture.

A graph captured on a stream keeps the workspace address it saw.  A later,
larger eager call on the same stream grows the workspace; the old buffer must
stay valid (it is retired, not freed), so replays of the graph still read and
write live memory and still produce the oracle's result.  Tolerance: the
matvec bar, |gpu - ref| <= 1e-4 + 1e-3 |ref| (with the exact-sum substitution
of helpers.assert_close_attributed).
"""
import ctypes

import numpy as np
import pytest
import torch

import ssdq
import ssdq_oracle as o
from helpers import announce, assert_close_attributed, to_dev
from ssdq import synth

pytestmark = pytest.mark.gpu


def test_graph_replay_after_workspace_growth():
    dev = torch.device("cuda")
    side = torch.cuda.Stream()
    # K-sliced Q4_K matvec (4096 x 14336): its slice partials live in the
    # workspace, summed by a second kernel
    out_dim, in_dim = 4096, 14336
    w = synth.quant_weights(ssdq.Q4_K, out_dim, in_dim, 901)
    x = synth.normal_f32(in_dim, 902)
    wd, xd = to_dev(w), to_dev(x)
    yd = torch.empty(out_dim, dtype=torch.float32, device=dev)
    ref = o.matvec(ssdq.Q4_K, w, x, out_dim, in_dim, threads=16)[0]
    exact = o.matvec_exact(ssdq.Q4_K, w, x, out_dim, in_dim)

    announce("workspace: eager warm-up and capture of a K-sliced matvec")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        ssdq.matvec(ssdq.Q4_K, wd, xd, yd, out_dim, in_dim, stream=side)
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        ssdq.matvec(ssdq.Q4_K, wd, xd, yd, out_dim, in_dim, stream=side)
    torch.cuda.synchronize()

    # a larger eager call on the same stream: the prefill GEMM's prepared X
    # (512 x 4096 fp16 plus sums, ~4 MB) outgrows the matvec's partials
    announce("workspace: larger eager GEMM on the captured stream")
    M, N, K = 512, 1024, 4096
    gw = synth.quant_weights(ssdq.Q4_K, N, K, 903)
    gx = synth.f32_to_bf16_bits(synth.normal_f32((M, K), 904))
    gy = torch.empty(M * N, dtype=torch.float32, device=dev)
    with torch.cuda.stream(side):
        ssdq.gemm_q4k_bf16(to_dev(gw), to_dev(gx), gy, M, N, K, stream=side)
    side.synchronize()

    # replays, with eager work and synchronizations between them
    for rep in range(4):
        announce("workspace: graph replay", rep)
        yd.fill_(np.nan)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = yd.cpu().numpy()
        assert_close_attributed(got, ref, exact, f"replay {rep}")
        # unrelated eager work on the side stream between replays
        with torch.cuda.stream(side):
            ssdq.matvec(ssdq.Q4_K, wd, xd, torch.empty_like(yd), out_dim, in_dim, stream=side)
        side.synchronize()

    # a reservation larger than anything so far also leaves the graph valid
    announce("workspace: reserve, then replay")
    ssdq.reserve_workspace(64 << 20, stream=side)
    yd.fill_(np.nan)
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    assert_close_attributed(yd.cpu().numpy(), ref, exact, "after reserve")
    del g
    torch.cuda.synchronize()
    ssdq.release_workspaces()


def own_stream():
    """A stream that had no call before (torch hands out streams of a pool); kept,
    so that no later stream gets its handle, and with it its workspace."""
    hip = ctypes.CDLL("libamdhip64.so")
    handle = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
    return torch.cuda.ExternalStream(handle.value)


def test_batch_workspace_is_bounded():
    # 32 rows of a wide matrix with K slices: the partial sums of at most 32 MiB of
    # rows at a time (43680 here), whole groups of 16, the last piece ragged
    dtype, out_dim, in_dim, batch = ssdq.Q4_0, 90005, 2304, 32
    w = synth.quant_weights(dtype, out_dim, in_dim, 920)
    x = synth.normal_f32((batch, in_dim), 921).reshape(batch, in_dim)
    wd, xd = to_dev(w), to_dev(x)
    y = torch.empty(batch * out_dim, dtype=torch.float32, device="cuda")
    ssdq.matvec(dtype, wd, xd, y, 16, in_dim, 2)  # code loaded
    y.fill_(float("nan"))
    torch.cuda.synchronize()
    side = own_stream()
    announce("workspace: bounded", out_dim, in_dim, batch)
    free = torch.cuda.mem_get_info()[0]
    ssdq.matvec(dtype, wd, xd, y, out_dim, in_dim, batch, stream=side)
    side.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 34 << 20
    y = y.cpu().numpy().reshape(batch, out_dim)
    rows = np.r_[0:40, 43660:43700, 87340:87380, 89990:out_dim]
    wr = w.reshape(out_dim, -1)[rows].ravel()
    for b in (0, 31):
        ref = o.matvec(dtype, wr, x[b], rows.size, in_dim)[0]
        assert_close_attributed(y[b, rows], ref, o.matvec_exact(dtype, wr, x[b], rows.size, in_dim), f"row {b}")
    assert np.isfinite(y).all()


def test_no_workspace_for_calls_that_use_none():
    # Q6_K rows of an odd block count run on the byte-addressed kernel, 2-8 rows of
    # Q8_0 at K = 4096 in one launch: neither has K slices, so a stream of its own
    # gets no workspace for them
    side = own_stream()
    for dtype, out_dim, in_dim, batch in ((ssdq.Q6_K, 4096, 11008, 32), (ssdq.Q8_0, 256, 4096, 8)):
        w = to_dev(synth.quant_weights(dtype, out_dim, in_dim, 910))
        x = to_dev(synth.normal_f32((batch, in_dim), 911))
        y = torch.empty(batch * out_dim, dtype=torch.float32, device="cuda")
        ssdq.matvec(dtype, w, x, y, 16, in_dim, 2)  # code loaded
        torch.cuda.synchronize()
        announce("workspace: none wanted", dtype, out_dim, in_dim, batch)
        free = torch.cuda.mem_get_info()[0]
        ssdq.matvec(dtype, w, x, y, out_dim, in_dim, batch, stream=side)
        side.synchronize()
        assert torch.cuda.mem_get_info()[0] == free
