"""Host-side checks of the module layer that need no GPU: buffer validation and
fusion rules (pare/layers/linear.py:40-99 buffer contract)."""

from __future__ import annotations

import gc
import threading
import weakref

import pytest
import torch

import pare_amd as P


def _ql(N, K, gs=128, g_idx=None):
    packed = torch.zeros(N, K // 2, dtype=torch.uint8)
    scale = torch.ones(N, K // gs, 1)
    zero = torch.full((N, K // gs, 1), 8.0)
    return P.QuantizedLinear(packed, scale, zero, P.QuantConfig(group_size=gs), None, K, N,
                             use_kernel=True, g_idx=g_idx)


def test_quantized_linear_rejects_bad_packed_shape():
    with pytest.raises(ValueError, match="packed_weight"):
        P.QuantizedLinear(torch.zeros(8, 10, dtype=torch.uint8), torch.ones(8, 1, 1),
                          torch.zeros(8, 1, 1), P.QuantConfig(group_size=128), None, 128, 8)


def test_quantized_linear_cpu_forward_raises():
    with pytest.raises(RuntimeError, match="HIP device"):
        _ql(8, 128)(torch.zeros(1, 128))


def test_fused_concatenates_buffers():
    f = P.FusedQuantizedLinear([_ql(64, 256), _ql(16, 256), _ql(16, 256)])
    assert f.split_sizes == [64, 16, 16]
    assert tuple(f.fused.packed_weight.shape) == (96, 128)
    assert tuple(f.fused.scale.shape) == (96, 2, 1)
    assert f.in_features == 256 and f.fused.use_kernel


def test_fused_rejects_mismatched_layers():
    with pytest.raises(ValueError, match="in_features"):
        P.FusedQuantizedLinear([_ql(64, 256), _ql(64, 512)])
    with pytest.raises(ValueError, match="group size"):
        P.FusedQuantizedLinear([_ql(64, 256, gs=128), _ql(64, 256, gs=64)])
    g = torch.arange(256, dtype=torch.int32) // 128
    with pytest.raises(ValueError, match="g_idx"):
        P.FusedQuantizedLinear([_ql(64, 256, g_idx=g), _ql(64, 256)])
    with pytest.raises(ValueError, match="at least one"):
        P.FusedQuantizedLinear([])


def test_workspaces_of_captures_and_eager_calls_are_apart(monkeypatch):
    """A graph's replays may run beside eager calls on the stream it was captured
    on, and beside another graph captured there: none of them shares a workspace,
    and what a capture holds is let go once it has ended."""
    from pare_amd import kernels as KN

    capture = 0
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capture != 0)
    monkeypatch.setattr(KN, "_capture_id", lambda stream: capture, raising=False)
    dev, stream = torch.device("cpu", 0), 0x7007

    eager = KN._workspace(dev, stream, 1 << 20)
    capture = 11
    first = KN._workspace(dev, stream, 1 << 20)
    assert first is not eager and KN._workspace(dev, stream, 1 << 19) is first
    assert first[:64 * 1024].eq(0).all()
    assert KN._workspace(dev, stream, 8 << 20) is first      # one fill of the counters for small calls
    larger = KN._workspace(dev, stream, (8 << 20) + 1)
    assert larger is not first and KN._workspace(dev, stream, 1 << 20) is larger
    capture = 12
    second = KN._workspace(dev, stream, 1 << 20)
    capture = 0
    assert KN._workspace(dev, stream, 1 << 20) is eager
    assert len({t.data_ptr() for t in (eager, first, larger, second)}) == 4
    refs = [weakref.ref(t) for t in (first, larger, second)]
    del first, larger, second
    gc.collect()
    assert all(r() is None for r in refs)
    # another eager call of the stream that needs more replaces its workspace
    grown = KN._workspace(dev, stream, (1 << 20) + 1)
    assert grown is not eager and KN._workspace(dev, stream, 1 << 20) is grown


def test_threads_on_one_stream_have_workspaces_of_their_own(monkeypatch):
    """Two threads that launch on the same stream: the launches of their calls
    may interleave, so neither works in the other's scratch, and a thread that
    has ended keeps none."""
    from pare_amd import kernels as KN

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    dev, stream = torch.device("cpu", 0), 0x7107
    mine = KN._workspace(dev, stream, 1 << 20)
    other = []

    def work():
        ws = KN._workspace(dev, stream, 1 << 20)
        assert KN._workspace(dev, stream, 1 << 20) is ws
        other.append((ws.data_ptr(), weakref.ref(ws)))

    t = threading.Thread(target=work)
    t.start()
    t.join()
    assert other and other[0][0] != mine.data_ptr()
    gc.collect()
    assert other[0][1]() is None
    assert KN._workspace(dev, stream, 1 << 20) is mine


def test_kernel_available_needs_the_host_extension(monkeypatch):
    """matmul_w4a16 raises where the host extension does not load (not built, or
    built for another torch): the probe then says so."""
    from types import SimpleNamespace

    from pare_amd import _lib
    from pare_amd import kernels as KN

    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(pmi_device_supported=lambda d: 1))
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(_lib, "host", lambda: None)
    assert KN.kernel_available()

    def missing():
        raise RuntimeError("not built")

    monkeypatch.setattr(_lib, "host", missing)
    assert not KN.kernel_available()


def test_cache_of_a_module_saved_by_an_earlier_version():
    """A pickled module carries its kernel copies. One saved when the cache had no
    tiled_supported entry is left to the general path, which reads four entries."""
    layer = _ql(64, 256)
    layer._packed_weight_kernel, layer._packed_weight_tiled, layer._perm16 = layer.packed_weight, None, None
    layer._kernel_cache = (layer._stamp(), torch.zeros(64, 2, dtype=torch.uint8), None, None)
    assert layer._forward_host(torch.zeros(1, 256)) is None
    assert layer._kernel_buffers()[0] is layer.packed_weight
