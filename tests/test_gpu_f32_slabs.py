"""The f32 GEMM's split operands and K slabs (nf4_gemm_f32.hip): forward and
dX at the edges of its row tiles (64 and 128 rows), K steps (32) and slabs
(eight steps), magnitudes at both ends of f32, and infinities beside slabs,
against the float64 product at the f32 bar (1e-5 of the sum of |products|);
and the slabs taken in turn, to the same bits, where the workspace cannot hold their partials
(the least workspace, a stream under capture).
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from unifur_amd import _lib as L
from unifur_amd import quantize as Q

from test_gpu_gemm import lora_parts
from test_gpu_linear import TOL_F32, acts, make_linear

pytestmark = pytest.mark.gpu


def worst(got, ref, bound):
    return float(np.max(np.abs(np.asarray(got, np.float64) - ref) / np.maximum(bound, 1e-300)))


# (rows, d_in, d_out): one step and less; a slab boundary with a partial last
# step; sixteen slabs; rows around the 64- and 128-row tiles
SHAPES = [(1, 4, 64), (33, 36, 64), (64, 2052, 192), (65, 4096, 128), (128, 544, 4096), (129, 4100, 256),
          (300, 2048, 320)]


@pytest.mark.parametrize("striped", [True, False])
@pytest.mark.parametrize("shape", SHAPES)
def test_backward_dx(device, oracle, shape, striped):
    M, K, N = shape
    lin, wdeq = make_linear(oracle, K, N, 0xB0 + M, device, striped=striped)
    dy, dyt = acts(oracle, M, N, 0xB1, torch.float32, device)
    w = wdeq.astype(np.float64)
    dx = lin.backward(dyt).cpu().numpy()
    assert worst(dx, dy.astype(np.float64) @ w.T, np.abs(dy) @ np.abs(w).T) <= TOL_F32


@pytest.mark.parametrize("striped", [True, False])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[0] > 32])
def test_forward(device, oracle, shape, striped):
    M, K, N = shape
    lin, wdeq = make_linear(oracle, K, N, 0xB2 + M, device, dq=striped, striped=striped)
    x, xt = acts(oracle, M, K, 0xB3, torch.float32, device)
    y = lin.forward(xt).cpu().numpy()
    w = wdeq.astype(np.float64)
    assert worst(y, x.astype(np.float64) @ w, np.abs(x) @ np.abs(w)) <= TOL_F32


@pytest.mark.parametrize("scale", [1e-30, 1e30, 3.0e38])
def test_magnitudes(device, oracle, scale):
    """The largest f32 values round to an infinite first term, which leads to
    the f32 instruction, and so do values that the scaling before the cut
    takes past it."""
    M, K, N = 96, 512, 128
    lin, wdeq = make_linear(oracle, K, N, 0xB4, device)
    x, _ = acts(oracle, M, K, 0xB5, torch.float32, device)
    x = (x / np.abs(x).max() * scale).astype(np.float32)
    if scale > 1e38:
        x[:, np.arange(K) % 64 != 0] = 0.0  # eight products a sum, so that none overflows
    w = wdeq.astype(np.float64)
    ref = x.astype(np.float64) @ w
    ok = np.abs(x).astype(np.float64) @ np.abs(w) < 3.4e38  # no partial sum can overflow
    got = lin.forward(torch.from_numpy(x).to(device)).cpu().numpy()
    assert ok.any()
    assert worst(got[ok], ref[ok], (np.abs(x).astype(np.float64) @ np.abs(w))[ok]) <= TOL_F32


def test_infinities_beside_slabs(device, oracle):
    M, K, N = 70, 4096, 192
    lin, wdeq = make_linear(oracle, K, N, 0xB6, device)
    x, _ = acts(oracle, M, K, 0xB7, torch.float32, device)
    x = x.copy()
    x[0, 5], x[3, 4000], x[69, 77] = np.inf, -np.inf, np.nan
    x[5, 1], x[5, 4090] = np.inf, np.inf  # in two slabs: one sign or NaN per column
    w = wdeq.astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w
    got = lin.forward(torch.from_numpy(x).to(device)).cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
    fin = np.isfinite(ref)
    clean = np.where(np.isfinite(x), x, 0.0)
    assert worst(got[fin], ref[fin], (np.abs(clean) @ np.abs(w))[fin]) <= TOL_F32


def test_least_workspace_and_capture_take_the_slabs_in_turn(device, oracle):
    M, K, N, r = 130, 4096, 1024, 8
    lin, wdeq = make_linear(oracle, K, N, 0xB8, device)
    x, xt = acts(oracle, M, K, 0xB9, torch.float32, device)
    a, b, ad = lora_parts(oracle, K, N, r, 0xBA, device)
    w = wdeq.astype(np.float64)
    ref = x.astype(np.float64) @ w + oracle.lora_ref_f64(x, a, b, 2.0)
    bound = np.abs(x) @ np.abs(w) + (np.abs(x) @ np.abs(a)) @ np.abs(b) * 2.0
    lib = L.lib()
    least = lib.unifur_nf4_linear_min_workspace_size(M, K, N, L.F32, r)
    assert least < lib.unifur_nf4_linear_workspace_size(M, K, N, L.F32, r)
    ws = torch.zeros(least, dtype=torch.uint8, device=device)
    y = torch.empty(M, N, device=device)
    ww, lo = lin.weight_struct(), ad.struct()
    L.check(lib.unifur_nf4_linear_forward(xt.data_ptr(), L.F32, M, ctypes.byref(ww), None, ctypes.byref(lo),
                                          y.data_ptr(), L.F32, ws.data_ptr(), least,
                                          torch.cuda.current_stream().cuda_stream))
    assert worst(y.cpu().numpy(), ref, bound) <= TOL_F32
    assert torch.equal(y, Q.QloraLinear(lin, ad).forward(xt))
    # a stream whose internal workspace a small call sized, then under capture
    layer = Q.QloraLinear(lin, ad)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        layer.forward(xt[:2])
        s.synchronize()
        with torch.cuda.graph(graph, stream=s):
            out = layer.forward(xt)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y)


def call(lin, xt, need, adapter=None):
    y = torch.empty(xt.shape[0], lin.d_output(), device=xt.device)
    ws = torch.zeros(need, dtype=torch.uint8, device=xt.device)
    w, lo = lin.weight_struct(), adapter.struct() if adapter is not None else None
    L.check(L.lib().unifur_nf4_linear_forward(xt.data_ptr(), L.F32, xt.shape[0], ctypes.byref(w), None,
                                              ctypes.byref(lo) if lo is not None else None, y.data_ptr(), L.F32,
                                              ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
    return y


def in_skinny_launches(lin, xt, adapter=None):
    """What launches of at most 32 rows give, each by a call of its own."""
    layer = Q.QloraLinear(lin, adapter) if adapter is not None else lin
    return torch.cat([layer.forward(xt[m:m + 32]) for m in range(0, xt.shape[0], 32)])


@pytest.mark.parametrize("rows", [40, 64])
@pytest.mark.parametrize("K,N,r", [(4096, 4096, 0), (2048, 8192, 8), (11008, 256, 0)])
def test_without_room_33_to_64_rows_take_the_skinny_kernel(device, oracle, rows, K, N, r):
    """One workgroup a tile taking the slabs in turn is several times slower
    there than two skinny launches."""
    lin, wdeq = make_linear(oracle, K, N, 0xBB, device)
    x, xt = acts(oracle, rows, K, 0xBC, torch.float32, device)
    w = wdeq.astype(np.float64)
    ref, bound, ad = x.astype(np.float64) @ w, np.abs(x) @ np.abs(w), None
    if r:
        a, b, ad = lora_parts(oracle, K, N, r, 0xBD, device)
        ref = ref + oracle.lora_ref_f64(x, a, b, 2.0)
        bound = bound + (np.abs(x) @ np.abs(a)) @ np.abs(b) * 2.0
    lib = L.lib()
    y = call(lin, xt, lib.unifur_nf4_linear_min_workspace_size(rows, K, N, L.F32, r), ad)
    assert torch.equal(y, in_skinny_launches(lin, xt, ad))
    assert worst(y.cpu().numpy(), ref, bound) <= TOL_F32
    full = call(lin, xt, lib.unifur_nf4_linear_workspace_size(rows, K, N, L.F32, r), ad)
    assert worst(full.cpu().numpy(), ref, bound) <= TOL_F32


@pytest.mark.parametrize("rows", [40, 64])
@pytest.mark.parametrize("K,N", [(8192, 256), (16384, 896), (2048, 8192)])
def test_narrow_and_one_round_shapes_stay_on_the_skinny_kernel(device, oracle, rows, K, N):
    lin, wdeq = make_linear(oracle, K, N, 0xBE, device)
    x, xt = acts(oracle, rows, K, 0xBF, torch.float32, device)
    w = wdeq.astype(np.float64)
    y = lin.forward(xt)
    assert torch.equal(y, in_skinny_launches(lin, xt))
    assert worst(y.cpu().numpy(), x.astype(np.float64) @ w, np.abs(x) @ np.abs(w)) <= TOL_F32
