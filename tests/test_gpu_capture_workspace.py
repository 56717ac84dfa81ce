"""A captured call whose plan needs more than the stream's internal workspace
holds is refused with UNIFUR_NF4_ERR_WORKSPACE and records nothing, on the
bf16 paths whose workspace a caller has to size; the f32 GEMM, which needs no
more than its least form, is captured with its slabs in turn, and a call that
succeeds leaves no error text behind.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from unifur_amd import _lib as L
from unifur_amd import quantize as Q
from unifur_amd import qwennet as N

from test_gpu_graphs import _hip

pytestmark = pytest.mark.gpu

P = ctypes.c_void_p


@pytest.fixture
def stream():
    h = _hip()
    s = P()
    assert h.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0  # a new stream: no workspace yet
    yield h, s
    assert h.hipStreamSynchronize(s) == 0
    h.hipStreamDestroy(s)


def captured(h, s, call):
    """Status of a call under capture, the error text after it and the number
    of nodes it recorded."""
    graph, n = P(), ctypes.c_size_t(0)
    assert h.hipStreamBeginCapture(s, 2) == 0
    st = call()
    text = L.lib().unifur_nf4_last_error()
    assert h.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert h.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    h.hipGraphDestroy(graph)
    return st, text, n.value


def weight(device, k, n, seed):
    g = torch.Generator(device)
    g.manual_seed(seed)
    return Q.Nf4Linear.from_values(torch.randn(k, n, generator=g, device=device) * 0.02, k, n)


def size_workspace(lin, x1, y1, s):
    """An eager call of one row: the stream's internal workspace at its least."""
    w = lin.weight_struct()
    assert L.lib().unifur_nf4_linear_forward(x1.data_ptr(), L.F32, 1, ctypes.byref(w), None, None, y1.data_ptr(),
                                             L.F32, None, 0, s) == 0


def test_bf16_plans_are_refused(device, stream):
    h, s = stream
    lib = L.lib()
    K = 4096
    lin, gate, up, down = (weight(device, k, n, i) for i, (k, n) in
                           enumerate([(K, K), (K, 2048), (K, 2048), (2048, K)]))
    x1, y1 = torch.zeros(1, K, device=device), torch.empty(1, K, device=device)
    x = torch.randn(100, K, device=device).bfloat16()
    y = torch.empty(100, K, device=device, dtype=torch.bfloat16)
    torch.cuda.synchronize()
    size_workspace(lin, x1, y1, s)
    w, ws = lin.weight_struct(), [m.weight_struct() for m in (gate, up, down)]
    layer = N.QwenDecoderLayer(lin, lin, lin, lin, Q.QwenMlp(gate, up, down), torch.zeros(K, device=device),
                               torch.zeros(K, device=device), 1e-6)
    ls = layer.layer_struct()
    q = [torch.empty_like(x) for _ in range(3)]
    calls = {
        "linear": lambda: lib.unifur_nf4_linear_forward(x.data_ptr(), L.BF16, 100, ctypes.byref(w), None, None,
                                                        y.data_ptr(), L.BF16, None, 0, s),
        "swiglu": lambda: lib.unifur_nf4_swiglu_forward(x.data_ptr(), L.BF16, 100, *[ctypes.byref(m) for m in ws],
                                                        y.data_ptr(), L.BF16, None, 0, s),
        "attn_in": lambda: lib.unifur_nf4_decoder_attn_in(x.data_ptr(), L.BF16, 100, ctypes.byref(ls),
                                                          *[t.data_ptr() for t in q], None, 0, s),
        "attn_out": lambda: lib.unifur_nf4_decoder_attn_out_mlp(x.data_ptr(), q[0].data_ptr(), L.BF16, 100,
                                                                ctypes.byref(ls), y.data_ptr(), None, 0, s),
    }
    for name, call in calls.items():
        st, text, nodes = captured(h, s, call)
        assert (st, nodes) == (L.ERR_WORKSPACE, 0) and b"capturing" in text, (name, st, nodes, text)


def test_f32_slabs_in_turn_leave_no_error(device, stream):
    h, s = stream
    lib = L.lib()
    K = 4096
    lin = weight(device, K, 1024, 9)
    x1, y1 = torch.zeros(1, K, device=device), torch.empty(1, 1024, device=device)
    x, y = torch.randn(130, K, device=device), torch.empty(130, 1024, device=device)
    torch.cuda.synchronize()
    size_workspace(lin, x1, y1, s)
    w = lin.weight_struct()
    before = lib.unifur_nf4_last_error()
    st, text, nodes = captured(h, s, lambda: lib.unifur_nf4_linear_forward(
        x.data_ptr(), L.F32, 130, ctypes.byref(w), None, None, y.data_ptr(), L.F32, None, 0, s))
    assert st == 0 and nodes == 1 and text == before, (st, nodes, text)
