"""The bf16 GEMM of batches just past the skinny kernel's (nf4_gemm_mid.hip)
at the edges of its row tiles (96 and 128 rows), column tiles (a last tile of
64 of its 128 columns) and d_in slabs (one that is shorter, one step), both
scale kinds, output types and alignments, with a bias and an adapter, against
the float64 product at the bf16 bar; and its slabs taken in turn, to the same
bits, where the workspace has no room for their partials.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from unifur_amd import _lib as L
from unifur_amd import quantize as Q

from test_gpu_capture_workspace import captured, stream  # noqa: F401 (a fixture)
from test_gpu_gemm import lora_parts, zero_linear
from test_gpu_linear import TOL_BF16, TOL_F32, acts, check, make_linear

pytestmark = pytest.mark.gpu


def forward(lin, xt, rows, adapter, bias, y, need):
    w = lin.weight_struct()
    lo = adapter.struct() if adapter is not None else None
    ws = torch.zeros(need, dtype=torch.uint8, device=xt.device)
    L.check(L.lib().unifur_nf4_linear_forward(
        xt.data_ptr(), L.BF16, rows, ctypes.byref(w), bias.data_ptr() if bias is not None else None,
        ctypes.byref(lo) if lo is not None else None, y.data_ptr(), L.F32 if y.dtype == torch.float32 else L.BF16,
        ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
    assert int(ws[:65536].count_nonzero()) == 0
    return y


# 2^24 weights or more: d_in of 64-row steps that the slabs divide and not, a
# long d_in, a d_out of half a column tile
@pytest.mark.parametrize("K,N", [(4096, 4096), (4160, 4032 + 64), (16448, 1088), (1024, 16448)])
@pytest.mark.parametrize("rows,r,dq", [(65, 0, True), (96, 16, True), (97, 3, False), (128, 0, False), (129, 16, True),
                                       (192, 5, True)])
def test_mid_rows(device, oracle, K, N, rows, r, dq):
    lin, wdeq = make_linear(oracle, K, N, 0xC0 + rows, device, dq=dq)
    x, xt = acts(oracle, rows, K, 0xC1, torch.bfloat16, device)
    bias = oracle.fill_normal(0xC2, 0.1, N)
    bt = torch.from_numpy(bias).to(device)
    ref = oracle.linear_ref_f64(x, wdeq, bias)
    ad = None
    if r:
        a, b, ad = lora_parts(oracle, K, N, r, 0xC3, device)
        ref = ref + oracle.lora_ref_f64(x, a, b, 2.0)
    lib = L.lib()
    full = lib.unifur_nf4_linear_workspace_size(rows, K, N, L.BF16, r)
    least = lib.unifur_nf4_linear_min_workspace_size(rows, K, N, L.BF16, r)
    y = forward(lin, xt, rows, ad, bt, torch.empty(rows, N, device=device), full)
    check(y, ref, x, wdeq, TOL_BF16, f"mid {rows} x {K} -> {N} rank {r}")
    # a least workspace without room for the partials: the slabs in turn, the
    # same bits (with an adapter where it holds x A, else the fused kernel)
    y2 = forward(lin, xt, rows, ad, bt, torch.empty(rows, N, device=device), least)
    if least >= 65536 + (4 * rows * r + 255) // 256 * 256:
        assert torch.equal(y, y2)
    else:
        check(y2, ref, x, wdeq, TOL_BF16, f"mid {rows} x {K} -> {N} rank {r} least")
    # bf16 outputs are the same sums rounded, at an output off 16 bytes too
    buf = torch.full((rows * N + 8,), float("nan"), dtype=torch.bfloat16, device=device)
    y3 = buf[1:1 + rows * N].view(rows, N)
    forward(lin, xt, rows, ad, bt, y3, full)
    assert torch.equal(y3, y.to(torch.bfloat16))
    assert torch.isnan(buf[0]) and torch.isnan(buf[1 + rows * N:]).all()


# x A in slabs of d_in (2^18 factor elements or more): two and four rows a
# group with a last group that is not full, four columns a lane and one, a rank
# whose eights the GEMM's slabs do not share evenly
@pytest.mark.parametrize("K,N,rows,r", [(8192, 2048, 65, 32), (8192, 2048, 130, 64), (8192, 2048, 99, 33),
                                        (8192, 2112, 191, 45), (4096, 4096, 128, 64), (8256, 4096, 255, 64)])
def test_wide_adapters(device, oracle, K, N, rows, r):
    lin, wdeq = make_linear(oracle, K, N, 0xC6, device)
    x, xt = acts(oracle, rows, K, 0xC7, torch.bfloat16, device)
    a, b, ad = lora_parts(oracle, K, N, r, 0xC8, device)
    ref = oracle.linear_ref_f64(x, wdeq) + oracle.lora_ref_f64(x, a, b, 2.0)
    lib = L.lib()
    full = lib.unifur_nf4_linear_workspace_size(rows, K, N, L.BF16, r)
    least = lib.unifur_nf4_linear_min_workspace_size(rows, K, N, L.BF16, r)
    y = forward(lin, xt, rows, ad, None, torch.empty(rows, N, device=device), full)
    check(y, ref, x, wdeq, TOL_BF16, f"mid {rows} x {K} -> {N} rank {r}")
    assert torch.equal(y, forward(lin, xt, rows, ad, None, torch.empty(rows, N, device=device), least))
    # the adapter's term alone, over a weight of zeros, is f32 throughout
    zero = zero_linear(K, N, device, True)
    t = forward(zero, xt, rows, ad, None, torch.empty(rows, N, device=device), full).cpu().numpy()
    bound = (np.abs(x) @ np.abs(a)) @ np.abs(b) * 2.0
    assert float(np.max(np.abs(t - oracle.lora_ref_f64(x, a, b, 2.0)) / bound)) <= TOL_F32
    fresh = Q.LoraAdapter.new(Q.LoraConfig.new(K, N, r), device=device)
    assert torch.equal(Q.QloraLinear(lin, fresh).forward(xt), lin.forward(xt))


def test_an_adapter_of_zeros_adds_nothing(device, oracle):
    K = N = 4096
    lin, _ = make_linear(oracle, K, N, 0xC4, device)
    _, xt = acts(oracle, 100, K, 0xC5, torch.bfloat16, device)
    fresh = Q.LoraAdapter.new(Q.LoraConfig.new(K, N, 16), device=device)
    assert torch.equal(Q.QloraLinear(lin, fresh).forward(xt), lin.forward(xt))


# 2^25 weights and more: up to 256 rows
@pytest.mark.parametrize("rows,K,N", [(193, 4096, 8192), (256, 4096, 8192), (224, 11008, 4096)])
def test_rows_past_192(device, oracle, rows, K, N):
    lin, wdeq = make_linear(oracle, K, N, 0xC9, device)
    x, xt = acts(oracle, rows, K, 0xCA, torch.bfloat16, device)
    ref = oracle.linear_ref_f64(x, wdeq)
    lib = L.lib()
    full = lib.unifur_nf4_linear_workspace_size(rows, K, N, L.BF16, 0)
    y = forward(lin, xt, rows, None, None, torch.empty(rows, N, device=device), full)
    check(y, ref, x, wdeq, TOL_BF16, f"mid {rows} x {K} -> {N}")
    least = lib.unifur_nf4_linear_min_workspace_size(rows, K, N, L.BF16, 0)
    assert torch.equal(y, forward(lin, xt, rows, None, None, torch.empty(rows, N, device=device), least))


# the SwiGLU block's down projection takes this kernel over a striped weight of
# 2^24 values or more; its slabs lie in the block's partials
@pytest.mark.parametrize("hidden,inter", [(4096, 11008), (2048, 8192)])
@pytest.mark.parametrize("dq", [True, False])
@pytest.mark.parametrize("rows", [65, 129, 192, 256])
def test_swiglu_down(device, hidden, inter, dq, rows):
    g = torch.Generator(device)
    g.manual_seed(0xCB)
    lins = []
    for k, n in ((hidden, inter), (hidden, inter), (inter, hidden)):
        p = Q.PackedNf4Tensor.quantize(torch.randn(k * n, generator=g, device=device) * 0.02)
        lins.append(Q.Nf4Linear.from_packed(p.with_double_quantization() if dq else p, k, n, striped=True))
    x = torch.randn(rows, hidden, generator=g, device=device).bfloat16()
    wg, wu, wd = [m.dequantized_weight().double().view(m.d_input(), m.d_output()) for m in lins]
    a = x.double() @ wg
    h = a * torch.sigmoid(a) * (x.double() @ wu)
    ref, bound = h @ wd, h.abs() @ wd.abs()
    ws3 = [m.weight_struct() for m in lins]
    lib = L.lib()
    full = lib.unifur_nf4_swiglu_workspace_size(rows, hidden, inter, L.BF16)
    least = lib.unifur_nf4_swiglu_min_workspace_size(rows, hidden, inter, L.BF16)
    buf = torch.full((rows * hidden + 8,), float("nan"), device=device)
    for need, shift in ((full, 0), (least, 0), (full, 1)):  # shift: an output off 16 bytes
        y = buf[shift:shift + rows * hidden].view(rows, hidden)
        ws = torch.zeros(need, dtype=torch.uint8, device=device)
        L.check(lib.unifur_nf4_swiglu_forward(x.data_ptr(), L.BF16, rows, *[ctypes.byref(w) for w in ws3],
                                              y.data_ptr(), L.F32, ws.data_ptr(), need,
                                              torch.cuda.current_stream().cuda_stream))
        e = (y.double() - ref).abs()
        assert float((e / bound).max()) <= TOL_BF16 and float(e.max() / ref.abs().max()) <= TOL_BF16
        assert int(ws[:65536].count_nonzero()) == 0
        assert torch.isnan(buf[shift + rows * hidden:]).all()
        buf.fill_(float("nan"))


@pytest.mark.parametrize("K,N", [(4096, 4096), (8192, 2048)])
def test_a_workspace_between_takes_the_fused_slabs(device, oracle, stream, K, N):
    """128 rows in 16 MiB: the fused kernel's slabs fit where this kernel's
    just do not; a split launch and its reduction, not one launch of workgroups
    that take the slabs in turn (two to three times slower)."""
    h, s = stream
    rows, need = 128, 16 << 20
    lin, wdeq = make_linear(oracle, K, N, 0xCC, device)
    x, xt = acts(oracle, rows, K, 0xCD, torch.bfloat16, device)
    y = forward(lin, xt, rows, None, None, torch.empty(rows, N, device=device), need)
    check(y, oracle.linear_ref_f64(x, wdeq), x, wdeq, TOL_BF16, f"{rows} x {K} -> {N} in 16 MiB")
    ws, w = torch.zeros(need, dtype=torch.uint8, device=device), lin.weight_struct()
    torch.cuda.synchronize()
    for room, launches in ((need, 2), (L.lib().unifur_nf4_linear_min_workspace_size(rows, K, N, L.BF16, 0), 1)):
        st, text, nodes = captured(h, s, lambda: L.lib().unifur_nf4_linear_forward(
            xt.data_ptr(), L.BF16, rows, ctypes.byref(w), None, None, y.data_ptr(), L.F32, ws.data_ptr(), room, s))
        assert (st, nodes) == (L.OK, launches), (st, nodes, text)
