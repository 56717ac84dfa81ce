"""The adapter term of decode-sized calls, (x A) B s (LoraAdapter::forward,
src/quantize.rs:619-624), alone over an all-zero base weight: the x A kernel
at one row per workgroup and, past 256 rows, at four with a last row group that
is not full, every lane split of the rank (powers of two, ranks between them,
factors that are not four-float aligned), d_in below and past one step of the
workgroup, and the epilogue's batches of sixteen ranks with a remainder.

x is exact in its dtype and everything after it is f32, so both activation
types are held to the f32 bar (1e-5 of the sum of |products|).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from unifur_amd import quantize as Q

from test_gpu_gemm import lora_parts, zero_linear
from test_gpu_linear import TOL_F32, acts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 3, 4, 5, 33])
@pytest.mark.parametrize("K,r", [(64, 1), (64, 64), (200, 3), (1032, 4), (4104, 16), (896, 20), (4096, 33)])
def test_adapter_term_of_decode_rows(device, oracle, dt, rows, K, r):
    N, s = 192, 0.5
    lin = zero_linear(K, N, device, True)
    x, xt = acts(oracle, rows, K, 0x91 + K, dt, device)
    a, b, ad = lora_parts(oracle, K, N, r, 0x92 + r, device, scaling=s, sigma=0.05)
    got = Q.QloraLinear(lin, ad).forward(xt, out_dtype=torch.float32).cpu().numpy().astype(np.float64)
    ref = oracle.lora_ref_f64(x, a, b, s)
    bound = (np.abs(x) @ np.abs(a)) @ np.abs(b) * s
    assert float(np.max(np.abs(got - ref) / bound)) <= TOL_F32


@pytest.mark.parametrize("shift", [1, 2])
def test_adapter_term_with_a_factor_off_sixteen_bytes(device, oracle, shift):
    """A rank of a multiple of four whose A starts off a 16-byte boundary
    takes the one-column loads."""
    K, N, r, s = 640, 128, 8, 2.0
    lin = zero_linear(K, N, device, True)
    x, xt = acts(oracle, 2, K, 0x93, torch.float32, device)
    a, b, _ = lora_parts(oracle, K, N, r, 0x94, device, scaling=s, sigma=0.05)
    buf = torch.empty(K * r + shift, dtype=torch.float32, device=device)
    at = buf[shift:].view(K, r)
    at.copy_(torch.from_numpy(np.asarray(a, np.float32)))
    ad = Q.LoraAdapter(at, torch.from_numpy(np.asarray(b, np.float32)).to(device), s)
    got = Q.QloraLinear(lin, ad).forward(xt).cpu().numpy().astype(np.float64)
    bound = (np.abs(x) @ np.abs(a)) @ np.abs(b) * s
    assert float(np.max(np.abs(got - oracle.lora_ref_f64(x, a, b, s)) / bound)) <= TOL_F32


# past 256 rows, where no other kernel takes x A: a dense f32 linear (f32 and
# bf16 x), and a d_in the row products refuse (no multiple of 8) through the f32 GEMM
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [257, 259, 260])
@pytest.mark.parametrize("K,r", [(12, 4), (300, 16), (1032, 7)])
def test_four_rows_a_workgroup(device, oracle, dt, rows, K, r):
    N, s = 192, 0.5
    x, xt = acts(oracle, rows, K, 0x96 + K, dt, device)
    a, b, ad = lora_parts(oracle, K, N, r, 0x97 + r, device, scaling=s, sigma=0.05)
    ref = oracle.lora_ref_f64(x, a, b, s)
    bound = (np.abs(x) @ np.abs(a)) @ np.abs(b) * s
    layers = [Q.QLoRALinear(Q.DenseLinear(torch.zeros(K, N, device=device)), ad, K * N, False)]
    if dt == torch.float32 and K % 8:
        layers.append(Q.QloraLinear(zero_linear(K, N, device, True), ad))
    for layer in layers:
        got = layer.forward(xt, out_dtype=torch.float32).cpu().numpy().astype(np.float64)
        assert float(np.max(np.abs(got - ref) / bound)) <= TOL_F32


def test_rows_past_one_launch(device):
    """2^24 + 3 rows through an adapted f32 linear of 4 inputs: a launch of a
    1024-thread workgroup per four rows would pass 2^32 work items, which wrap."""
    K, N, r, s, M = 4, 4, 1, 2.0, (1 << 24) + 3
    g = torch.Generator(device)
    g.manual_seed(0x95)
    w, a, b = [torch.randn(*d, generator=g, device=device) for d in ((K, N), (K, r), (r, N))]
    x = torch.randn(M, K, generator=g, device=device)
    layer = Q.QLoRALinear(Q.DenseLinear(w), Q.LoraAdapter.from_parts(a, b, s), K * N, False)
    y = layer.forward(x)
    # f32 sums of K products and of one more: 1e-5 of the sum of |products|
    for m in range(0, M, 1 << 22):
        xm = x[m:m + (1 << 22)].double()
        ref = xm @ w.double() + (xm @ a.double()) @ b.double() * s
        bound = xm.abs() @ w.double().abs() + (xm.abs() @ a.double().abs()) @ b.double().abs() * s
        assert float(((y[m:m + (1 << 22)].double() - ref).abs() / bound).max()) <= TOL_F32, m
