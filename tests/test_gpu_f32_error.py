"""Rounding error of the f32 GEMM's split products (nf4_gemm_f32.hip) against
the float64 product of the same operands (the layer's own dequantized f32
weight, which the codec tests hold to the reference bit for bit): no larger
than that of f32 products summed in order by the f32 matrix instruction, also
where the terms of a sum share a sign and its rounding errors add up.
"""
from __future__ import annotations

import pytest
import torch

from unifur_amd import quantize as Q

pytestmark = pytest.mark.gpu


def normal(device, seed, *shape, sigma=1.0):
    g = torch.Generator(device)
    g.manual_seed(seed)
    return torch.randn(*shape, generator=g, device=device) * sigma


def layer(values, striped=None):
    lin = Q.Nf4Linear.from_values(values.contiguous(), values.shape[0], values.shape[1], striped=striped)
    return lin, lin.dequantized_weight().view(values.shape).double()


def rel(y, ref):
    return float((y.double() - ref).norm() / ref.norm())


# 512 rows x 8320 outputs are 260 tiles: one slab over all of the reduction,
# the longest chain of additions.  The bounds are what the f32 instruction
# shows at these shapes for operands of one sign.
ONE_SIGN = {4096: 8.8e-7, 11008: 1.45e-6, 11000: 1.45e-6}


@pytest.mark.parametrize("shift", [False, True])
@pytest.mark.parametrize("K", [4096, 11008])
def test_sums_of_one_sign_forward(device, K, shift):
    w, x = normal(device, 1, K, 8320, sigma=0.02), normal(device, 2, 512, K)
    lin, wd = layer(w + 0.005 if shift else w.abs())
    x = x + 1.0 if shift else x.abs()
    assert rel(lin.forward(x), x.double() @ wd) <= ONE_SIGN[K]


@pytest.mark.parametrize("N", [4096, 11008])
def test_sums_of_one_sign_dx(device, N):
    lin, wd = layer(normal(device, 3, 8320, N, sigma=0.02).abs())
    dy = normal(device, 4, 512, N, sigma=1e-3).abs()
    assert rel(lin.backward(dy), dy.double() @ wd.t()) <= ONE_SIGN[N]


def test_sums_of_one_sign_bf16_activations(device):
    K = 11000  # no multiple of 64: the f32 GEMM with bf16 activations
    lin, wd = layer(normal(device, 5, K, 8320, sigma=0.02).abs())
    x = normal(device, 6, 512, K).abs().bfloat16()
    assert rel(lin.forward(x, out_dtype=torch.float32), x.double() @ wd) <= ONE_SIGN[K]


def test_sums_of_one_sign_in_turn(device):
    """The slabs taken in turn (no room for partials) to the same bits."""
    K, N = 11008, 2048
    lin, wd = layer(normal(device, 7, K, N, sigma=0.02).abs())
    x = normal(device, 8, 300, K).abs()
    y = lin.forward(x)
    assert rel(y, x.double() @ wd) <= ONE_SIGN[K]


@pytest.mark.parametrize("dq", [True, False])
@pytest.mark.parametrize("striped", [True, False])
def test_rows_of_the_identity_give_the_dequantized_weight(device, striped, dq):
    """One exact product a sum: the weight operand is the f32 value of the
    format (level * scale, rounded once), bit for bit."""
    K, N = 320, 448
    p = Q.PackedNf4Tensor.quantize(normal(device, 9, K * N, sigma=0.02))
    lin = Q.Nf4Linear.from_packed(p.with_double_quantization() if dq else p, K, N, striped=striped)
    w = lin.dequantized_weight().view(K, N)
    assert torch.equal(lin.forward(torch.eye(K, device=device)), w)
    assert torch.equal(lin.backward(torch.eye(N, device=device)), w.t())
    # d_in no multiple of 64: the same kernel with bf16 activations
    K = 328
    p = Q.PackedNf4Tensor.quantize(normal(device, 10, K * N, sigma=0.02))
    lin = Q.Nf4Linear.from_packed(p.with_double_quantization() if dq else p, K, N, striped=striped)
    y = lin.forward(torch.eye(K, device=device, dtype=torch.bfloat16), out_dtype=torch.float32)
    assert torch.equal(y, lin.dequantized_weight().view(K, N))


# (rows, d_in, d_out), and what f32 products summed in order show there for
# operands of either sign and of one: the f32 instruction, and at 64 rows f32
# FMA in slabs
SHORT = [(512, 4, 8320, 3.8e-8, 3.5e-8), (512, 8, 8320, 5.1e-8, 4.5e-8), (512, 64, 8320, 1.37e-7, 1.11e-7),
         (64, 4096, 8192, 2.8e-7, 6.9e-8), (64, 11008, 8192, 4.5e-7, 1.07e-7)]


@pytest.mark.parametrize("M,K,N,either,one", SHORT)
def test_short_sums(device, M, K, N, either, one):
    w, x = normal(device, 11, K, N, sigma=0.02), normal(device, 12, M, K)
    lin, wd = layer(w)
    assert rel(lin.forward(x), x.double() @ wd) <= either
    lin, wd = layer(w.abs())
    assert rel(lin.forward(x.abs()), x.abs().double() @ wd) <= one


def test_single_products(device):
    """One product a sum.  Rounding the result is off by at most 2^-24 of it
    and 2.5e-8 rms; the products left out add at most 2 x 2^-25 and 0.6e-8
    rms, of either sign alike."""
    M, K, N = 512, 4096, 8320
    lin, wd = layer(normal(device, 13, K, N, sigma=0.02))
    v, at = normal(device, 14, M), torch.arange(M, device=device) * 7 % K
    x = torch.zeros(M, K, device=device)
    x[torch.arange(M, device=device), at] = v
    ref = v.double()[:, None] * wd[at]
    e = ((lin.forward(x).double() - ref) / ref)[ref != 0]
    assert float(e.abs().max()) <= 2.0 ** -23
    assert float(e.square().mean().sqrt()) <= 2.7e-8
    assert abs(float(e.mean())) <= 2e-9


# f32 products summed in order show 3.9e-7 over these 512 terms, and 4.8e-7
# where the operands are subnormal
@pytest.mark.parametrize("scale", [1e-33, 1e-35, 1e-37, 1e-39])
def test_the_smallest_operands(device, scale):
    """x, dy and weights down to the subnormals: a bf16 term has no bits below
    2^-133, so operands are scaled before they are cut, or (weights) their sums
    taken with the f32 instruction."""
    M, K, N = 96, 512, 128
    bar = 4e-7 if scale > 1e-38 else 4.8e-7
    lin, wd = layer(normal(device, 15, K, N))
    x, dy = normal(device, 16, M, K) * scale, normal(device, 17, M, N) * scale
    assert rel(lin.forward(x), x.double() @ wd) <= bar
    assert rel(lin.backward(dy), dy.double() @ wd.t()) <= bar
    y = lin.forward(x)  # 32 rows and more of ordinary size beside them change nothing
    assert torch.equal(lin.forward(torch.cat([x, normal(device, 18, 40, K)]))[:M], y)
    for dq in (True, False):
        p = Q.PackedNf4Tensor.quantize(normal(device, 19, K * N) * scale)
        lin = Q.Nf4Linear.from_packed(p.with_double_quantization() if dq else p, K, N)
        wd, x = lin.dequantized_weight().view(K, N).double(), normal(device, 20, M, K)
        assert rel(lin.forward(x), x.double() @ wd) <= bar
    # bf16 activations (d_in no multiple of 64), small and beside small weights
    K = 520
    for xs, ws in ((scale, 1.0), (1.0, scale)):
        lin, wd = layer(normal(device, 21, K, N) * ws)
        x = (normal(device, 22, M, K) * xs).bfloat16()
        assert rel(lin.forward(x, out_dtype=torch.float32), x.double() @ wd) <= bar
