"""The host extension's matmul call against the general Python path: the same
bits, dtypes and shapes where it takes a call, the same errors where it does
not."""

from __future__ import annotations

import ctypes

import pytest
import torch

import pare_amd as P
from pare_amd import _lib
from pare_amd import kernels as KN
from pare_amd.config import QuantConfig
from pare_amd.linear import QuantizedLinear

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _layer(N, K, gs, bias=None, act_order=False, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randn(N, K, generator=g, device=DEV) * 0.02
    packed, s, z = P.rtn_quantize(w, gs)
    g_idx = None
    if act_order:
        g_idx = (torch.randperm(K, generator=g, device=DEV) // gs).to(torch.int32)
    return QuantizedLinear(packed, s, z, QuantConfig(bits=4, scheme="rtn", group_size=gs), bias, K, N,
                           use_kernel=True, g_idx=g_idx)


@pytest.mark.parametrize("shape", [(1,), (1, 1), (2, 3), (4, 1, 5), (70,), ()])
@pytest.mark.parametrize("dtype,native", [(torch.float16, False), (torch.bfloat16, False),
                                          (torch.bfloat16, True), (torch.float32, False)])
@pytest.mark.parametrize("N,K,gs,act_order", [(512, 1536, 128, False), (1028, 2048, 64, False),
                                              (260, 384, 128, True), (66, 256, 32, False)])
def test_module_forward_equals_the_general_path(N, K, gs, act_order, dtype, native, shape):
    for bias in (None, torch.randn(N, device=DEV).to(dtype)):
        layer = _layer(N, K, gs, bias, act_order)
        layer.native_bf16 = native
        x = torch.randn(*shape, K, device=DEV).to(dtype)
        with torch.no_grad():
            first = layer(x)                          # builds the copies: general path
            fast = layer._forward_host(x)
            want = layer._forward_kernel(x)
        assert fast is not None
        for y in (first, fast):
            assert y.dtype == want.dtype and y.shape == want.shape and y.is_contiguous()
            assert torch.equal(y, want)


@pytest.mark.parametrize("N,K,gs,M", [(1024, 4096, 256, 512), (516, 10240, 512, 70), (1024, 4096, 128, 512),
                                      (512, 2048, 64, 512)])
def test_native_bf16_does_not_depend_on_earlier_calls(N, K, gs, M):
    """The kernel (and so the bits) of a native bf16 forward: the same on a fresh
    layer as after a call of few rows that builds the tiled copy."""
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3)).bfloat16()
    outs = []
    for early in (False, True):
        layer = _layer(N, K, gs)
        layer.native_bf16 = True
        if early:
            layer(x[:8])
            assert layer._packed_weight_tiled is not None
        outs += [layer(x), layer(x)]
    for y in outs[1:]:
        assert torch.equal(y.view(torch.int16), outs[0].view(torch.int16))


@pytest.mark.parametrize("gs", [64, 128, 256])
def test_bf16_act_order_call_reads_the_copies_it_was_given(gs):
    """A bf16 call with a permutation and the tiled copy: with ``out`` (general
    path) and without (host extension) it is the same call, on the kernel that
    the copy allows."""
    N, K, M = 516, 2048, 225
    layer = _layer(N, K, gs, act_order=True)
    layer.native_bf16 = True
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3)).bfloat16()
    w, z, perm, sz = layer._kernel_buffers()
    layer(x[:8])                                     # the GEMV: no copy for it
    assert layer._packed_weight_tiled is None
    wt = P.tile_w4a16(w, gs)
    kw = {"perm": perm, "sz_gm": sz, "w_tiled": wt}
    assert KN.kernel_route(M, N, K, gs, torch.bfloat16, tiled=True, perm=True) == "bgemm"
    y = P.matmul_w4a16_bf16(x, w, layer.scale, z, gs, **kw)
    out = torch.empty_like(y)
    P.matmul_w4a16_bf16(x, w, layer.scale, z, gs, out=out, **kw)
    with KN.force_kernel("gemv"):
        gemv = P.matmul_w4a16_bf16(x, w, layer.scale, z, gs, **kw)
    for v in (out, layer(x), layer(x)):
        assert torch.equal(v.view(torch.int16), y.view(torch.int16))
    assert (y.double() - gemv.double()).norm() <= 4e-3 * gemv.double().norm()


def test_module_inputs_the_host_path_converts_or_leaves():
    layer = _layer(512, 1536, 128)
    x = torch.randn(6, 1536, device=DEV).half()
    want = layer(x)
    strided = torch.empty(6, 3072, device=DEV).half()[:, ::2].copy_(x)
    odd = torch.empty(6 * 1536 + 1, device=DEV).half()[1:].view(6, 1536).copy_(x)
    turned = x.t().contiguous().t()
    for v in (strided, odd, turned):
        assert torch.equal(layer._forward_host(v), want)
        assert torch.equal(layer(v), want)
    # left to the general path: empty inputs, other dtypes, changed weights
    assert layer._forward_host(x[:0]) is None and layer(x[:0]).shape == (0, 512)
    assert layer._forward_host(x.double()) is None and layer(x.double()).dtype == torch.float64
    layer.scale.mul_(2.0)
    assert layer._forward_host(x) is None
    assert torch.allclose(layer(x), 2 * want, rtol=2e-3, atol=1e-3)
    assert layer._forward_host(x) is not None
    with pytest.raises(RuntimeError, match="HIP device"):
        layer(x.cpu())
    with pytest.raises(RuntimeError):
        layer(torch.randn(2, 1000, device=DEV).half())


def test_bias_keeps_its_gradient_and_dtype():
    layer = _layer(256, 1536, 128, torch.randn(256, device=DEV))
    x = torch.randn(3, 1536, device=DEV).half()
    layer(x)
    y = layer(x)                                     # fp16 result + fp32 bias
    assert y.dtype == torch.float32 and y.requires_grad
    y.sum().backward()
    assert torch.equal(layer.bias.grad, torch.full((256,), 3.0, device=DEV))


def test_operator_errors_are_the_general_paths():
    layer = _layer(256, 1536, 128)
    w, z, _, sz = layer._kernel_buffers()
    s = layer.scale
    x = torch.randn(4, 1536, device=DEV).half()
    want = P.matmul_w4a16(x, w, s, z, 128)
    assert torch.equal(KN._matmul(x, w, s, z, 128, None, None, None, None, None), want)
    assert torch.equal(P.matmul_w4a16(x, w, s, z.float(), 128), want)   # fp32 zeros: general path
    out = torch.empty(4, 256, device=DEV, dtype=torch.float16)
    assert P.matmul_w4a16(x, w, s, z, 128, out=out) is out and torch.equal(out, want)
    bad = [dict(x=x[0]), dict(x=x.t()), dict(x=x.float()), dict(w=w[:, :-1]), dict(w=w.to(torch.int8)),
           dict(s=s[:-1]), dict(s=s.reshape(256, 1, 12)), dict(gs=100), dict(sz_gm=(sz[0].t(), sz[1].t())),
           dict(perm16=torch.zeros(1536, dtype=torch.int16, device=DEV)),
           dict(w_tiled=torch.zeros(16, dtype=torch.uint8, device=DEV)),
           dict(perm=torch.zeros(1536, dtype=torch.int64, device=DEV))]
    for kw in bad:
        args = {"x": x, "w": w, "s": s, "gs": 128, **kw}
        extra = {k: v for k, v in kw.items() if k not in ("x", "w", "s", "gs")}
        with pytest.raises((AssertionError, RuntimeError, IndexError)):
            P.matmul_w4a16(args["x"], args["w"], args["s"], z, args["gs"], **extra)


def test_buffers_that_the_general_path_converts_go_there_at_once(monkeypatch):
    """The reference's fp32 zeros, and scales of other types, are never the host
    extension's: it is not asked first (1.1-1.5 us of such a call)."""
    layer = _layer(256, 1536, 128)
    w, z, _, _ = layer._kernel_buffers()
    x = torch.randn(4, 1536, device=DEV).half()
    s16 = layer.scale.half()
    want = P.matmul_w4a16(x, w, layer.scale, z, 128)
    want16 = P.matmul_w4a16(x, w, s16.float(), z, 128)

    def asked(*args, **kw):
        raise AssertionError("asked the host extension")

    monkeypatch.setattr(KN, "host_matmul", asked)
    assert torch.equal(P.matmul_w4a16(x, w, layer.scale, z.float(), 128), want)
    assert torch.equal(P.matmul_w4a16(x, w, s16, z, 128), want16)
    xb = x.bfloat16()
    y = P.matmul_w4a16_bf16(xb, w, layer.scale, z.float(), 128)
    with pytest.raises(AssertionError, match="asked"):
        P.matmul_w4a16_bf16(xb, w, layer.scale, z, 128)
    assert y.dtype == torch.bfloat16


def test_vmap_and_subclasses_are_not_read_as_plain_tensors():
    layer = _layer(256, 1536, 128)
    x = torch.randn(4, 1536, device=DEV).half()
    want = layer(x)

    class Sub(torch.Tensor):
        pass

    sub = x.as_subclass(Sub)
    assert torch.equal(torch.as_tensor(layer(sub)).as_subclass(torch.Tensor), want)
    with pytest.raises(RuntimeError):
        torch.vmap(layer)(x)


def test_other_threads_run_during_the_library_call():
    """The library's entry points are called without the interpreter lock, as
    ctypes calls them: a launch on a full queue waits, and what it waits for may
    need the lock (a host callback in Python). In the place of the matmul: whether
    the calling thread holds it, where 0 counts as success."""
    layer = _layer(256, 1536, 128)
    x = torch.randn(4, 1536, device=DEV).half()
    layer(x)
    L, ext = _lib.lib(), _lib.host()
    fns = [ctypes.cast(getattr(L, f), ctypes.c_void_p).value for f in (
        "pmi_matmul_w4a16", "pmi_matmul_kernel_choice", "pmi_matmul_best_workspace_bytes",
        "pmi_matmul_route")]
    held = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    try:
        ext.bind(held, *fns[1:])
        y = layer._forward_host(x)
    finally:
        ext.bind(*fns)
    assert y is not None and y.shape == (4, 256)
    assert torch.equal(layer._forward_host(x), layer._forward_kernel(x))
