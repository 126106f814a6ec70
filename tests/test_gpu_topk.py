"""The sampler's candidates on the GPU (w4a8_topk) against the oracle's
restatement of the reference's insertion sort (board/tp/tp_llama.cpp:894-909):
values bit for bit and indices, at the LM-head size and its ragged and
maximum sizes, with heavy ties, +-0, -1e30 / -inf (never admitted) and fewer
admitted values than k; the first candidate equals the fused argmax of the
same logits; bad arguments are refused before any launch."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

import c_oracle as C
from gpu_helpers import dev, host

pytestmark = pytest.mark.gpu

F32 = np.float32


def _logits(n, seed, grid=0):
    rng = np.random.default_rng(seed)
    y = (rng.standard_normal(n) * 3).astype(np.float32)
    if grid:
        y = (np.round(y * grid) / grid).astype(np.float32)
    return y


def _check(gpu, y, k, label):
    vals, idx = gpu.topk(dev(y), k)
    want_v, want_i = C.topk(y, k)
    got_v, got_i = host(vals), host(idx)
    assert np.array_equal(got_i, want_i), (label, got_i[:8], want_i[:8])
    assert np.array_equal(got_v.view(np.uint32), want_v.view(np.uint32)), label


@pytest.mark.parametrize("n,k,seed,grid", [(128256, 40, 0, 0), (128256, 64, 1, 0), (128256, 1, 2, 0),
                                           (128256, 64, 3, 2), (262144, 64, 4, 8), (1000, 17, 5, 1),
                                           (1025, 64, 6, 0), (64, 64, 7, 0)])
def test_topk_matches_the_oracle(gpu, n, k, seed, grid):
    print(f"topk n={n} k={k} seed={seed} grid={grid}", flush=True)
    _check(gpu, _logits(n, seed, grid), k, f"n={n} k={k}")


def test_special_values(gpu):
    y = _logits(5000, 11, 1)
    y[:50] = F32(-1e30)
    y[50:100] = -np.inf
    y[100:110] = 0.0
    y[110:120] = -0.0
    y[200] = np.inf
    _check(gpu, y, 64, "specials")
    z = np.full(3000, F32(-1e30), dtype=np.float32)        # fewer admitted values than k
    z[[7, 1500, 2999]] = [1.0, -2.0, 1.0]
    z[[3, 4]] = [-np.inf, -5e30]
    _check(gpu, z, 64, "few admitted")
    _check(gpu, np.zeros(4096, dtype=np.float32), 64, "all zero")


@pytest.mark.parametrize("n,k", [(65536, 64), (65536 - 1024, 64), (65537, 64), (66561, 1), (128256, 40), (8192, 8),
                                 (8192, 9), (1025, 2), (1024, 1), (262144, 64), (262143, 40)])
@pytest.mark.parametrize("how", ["one slice", "few slices", "every slice", "descending", "negative zeros",
                                 "few admitted", "six slices admitted"])
def test_topk_where_the_best_lie(gpu, n, k, how):
    """Lists (1,024 logits each) as many as are merged pairwise (64), one more, one, and k;
    candidates at or above the k-th list head from one list's 64 up to more than the 256 that
    are sorted by themselves."""
    y = _logits(n, n + k)
    rng = np.random.default_rng(k)
    if how == "one slice":
        y[n - 900:n - 700] += 100.0
    elif how == "few slices":               # 64 in each of k / 2 slices: past 256
        for c in range(max(k // 2, 1)):
            y[1024 * c:1024 * c + 64] += 50.0 + rng.standard_normal(64).astype(np.float32)
    elif how == "every slice":              # each slice a full list above the rest
        for c in range(n // 1024):
            y[1024 * c + 100:1024 * c + 164] += 50.0
    elif how == "few admitted":             # fewer lists with a candidate than k, mostly
        y = np.where(np.arange(n) % (n // 5) == 0, y, F32(-1e30))
    elif how == "six slices admitted":      # as few lists, and more than 256 candidates
        y = np.where(np.arange(n) // 1024 % max(n // 6144, 1) == 0, y, F32(-1e30))
    elif how == "descending":
        y = np.sort(y)[::-1].copy()
    else:                                   # ties of +0 and -0, their bits kept
        y = -np.abs(y)
        at = rng.choice(n, 200, replace=False)
        y[at] = np.where(np.arange(200) % 2, F32(0.0), F32(-0.0))
    _check(gpu, y, k, f"n={n} k={k} {how}")


def test_topk_time_where_the_bound_does_not_help(gpu):
    """A call of one list has nothing to sort by heads, and where hundreds of candidates tie
    only the lists that hold them are merged: measured 0.72 times a call of 128,256 logits, and
    1.15 times the same call on random logits."""
    import torch

    def time(y, k):
        y = dev(y)
        ws = torch.empty(gpu.lib().w4a8_topk_workspace_bytes(y.numel()), dtype=torch.uint8, device="cuda")
        vals, idx = torch.empty(k, device="cuda"), torch.empty(k, dtype=torch.int32, device="cuda")
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            s = torch.cuda.current_stream().cuda_stream
            for _ in range(40):
                gpu.check("w4a8_topk", gpu.lib().w4a8_topk(y.data_ptr(), y.numel(), k, vals.data_ptr(), idx.data_ptr(),
                                                           ws.data_ptr(), ws.numel(), s))
        best = float("inf")
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            g.replay()
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        return best

    large, small = time(_logits(128256, 2), 40), time(_logits(1000, 1), 1)
    assert small < 0.87 * large, f"{small / large:.2f}"
    spread, tied = time(_logits(262144, 3), 64), time(np.ones(262144, np.float32), 64)
    assert tied < 1.32 * spread, f"{tied / spread:.2f}"


def test_first_candidate_is_the_fused_argmax(gpu):
    import q4_0_oracle as O
    rows, k = 128256, 2048
    blocks = C.quantize_q4_0(O.normal_f32((rows, k), 21, 0.02))
    x = O.normal_f32(k, 22)
    ws = gpu.argmax_workspace()
    y, best = gpu.gemv_q4_0_f32_argmax(dev(blocks), k, dev(x), ws)
    vals, idx = gpu.topk(y, 40)
    assert int(host(idx)[0]) == int(host(best)[0])
    _check(gpu, host(y), 40, "lm head logits")


def test_rejections(gpu):
    import torch
    L = gpu.lib()
    y = torch.zeros(1000, dtype=torch.float32, device="cuda")
    v = torch.empty(64, dtype=torch.float32, device="cuda")
    i = torch.empty(64, dtype=torch.int32, device="cuda")
    ws = torch.empty(L.w4a8_topk_workspace_bytes(262144), dtype=torch.uint8, device="cuda")
    nbytes = ws.numel()
    call = lambda n, k, wsb=nbytes, yp=y.data_ptr(): L.w4a8_topk(yp, n, k, v.data_ptr(), i.data_ptr(),
                                                                 ws.data_ptr(), wsb, None)
    assert call(1000, 0) == -2 and call(1000, 65) == -2 and call(0, 8) == -2 and call(262145, 8) == -2
    assert call(1000, 8, wsb=L.w4a8_topk_workspace_bytes(1000) - 1) == -2
    assert call(1000, 8, yp=y.data_ptr() + 2) == -3
    assert L.w4a8_topk(None, 1000, 8, v.data_ptr(), i.data_ptr(), ws.data_ptr(), nbytes, None) == -1
    assert call(1000, 8) == 0
    torch.cuda.synchronize()


def _check_nan(gpu, y, k, label):
    """Indices equal, NaN slots in the same places, every other value bit for bit."""
    vals, idx = gpu.topk(dev(y), k)
    want_v, want_i = C.topk(y, k)
    got_v, got_i = host(vals), host(idx)
    assert np.array_equal(got_i, want_i), (label, got_i[:8], want_i[:8])
    assert np.array_equal(np.isnan(got_v), np.isnan(want_v)), label
    ok = ~np.isnan(want_v)
    assert np.array_equal(got_v[ok].view(np.uint32), want_v[ok].view(np.uint32)), label
    # A NaN slot holds y's own NaN, bit for bit.
    for j in np.flatnonzero(~ok):
        assert got_v[j:j + 1].view(np.uint32)[0] == y[got_i[j]:got_i[j] + 1].view(np.uint32)[0], label


@pytest.mark.parametrize("n,k,seed,where", [(128256, 40, 20, "spread"), (128256, 64, 21, "last"),
                                            (128256, 1, 22, "spread"), (5000, 17, 23, "runs"),
                                            (1025, 64, 24, "first"), (64, 64, 25, "spread"),
                                            (262144, 40, 26, "late")])
def test_nan_logits_follow_the_reference_loop(gpu, n, k, seed, where):
    """NaN logits take the last slot and let the next logit in, as the
    reference's loop does (tp_llama.cpp:902-908), wherever they stand."""
    print(f"topk NaN n={n} k={k} seed={seed} where={where}", flush=True)
    rng = np.random.default_rng(seed)
    y = _logits(n, seed, grid=2 if where == "runs" else 0)
    if where == "spread":
        y[rng.integers(0, n, 12)] = np.nan
        y[rng.integers(0, n, 6)] = -np.inf
    elif where == "last":
        y[-1] = np.nan
    elif where == "first":
        y[0] = np.nan
        y[1] = -np.inf
    elif where == "runs":
        y[100:104] = np.nan
        y[2000:2002] = [np.nan, -np.inf]
        y[4999] = np.nan
    else:
        y[n - 5000] = np.nan
        y[n - 4999] = F32(-3e30)
    y[rng.integers(0, n, 2)] = F32(np.frombuffer(np.uint32(0xFFC00123).tobytes(), np.float32)[0])  # a payload
    _check_nan(gpu, y, k, f"n={n} k={k} {where}")
    clean = y.copy()
    clean[np.isnan(clean)] = 0.0
    _check(gpu, clean, k, f"n={n} k={k} without NaN")          # the parallel path again afterwards
