"""The wide-load forms of the RTN, repack, dequantisation and group-major
kernels: bit for bit the oracle, and bit for bit the general kernels, which
take the same buffers when they start at an odd address."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import pare_amd as P
from oracle import pare_oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
SHAPES = [(1, 32, 32), (3, 64, 8), (5, 640, 64), (2, 96, 16), (37, 1536, 512), (513, 768, 128),
          (7, 2048, 256), (11, 1152, 384), (130, 4096, 32), (3, 2048, 1024)]


def _off_by_one(t: torch.Tensor) -> torch.Tensor:
    """A contiguous copy that starts one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    return out


def _weights(N, K, gs, dtype):
    w = torch.randn(N, K, generator=torch.Generator().manual_seed(N + K)) * 0.02
    w[0, :gs] = 0.0                      # an all-zero group
    w[-1, -gs:] = -w[-1, -gs:].abs()     # one without positive values
    w[N // 2, 0] = -0.0
    return w.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sym", [False, True, "offset8"])
@pytest.mark.parametrize("N,K,gs", SHAPES)
def test_rtn_wide(N, K, gs, sym, dtype):
    w = _weights(N, K, gs, dtype)
    if dtype != torch.float16:           # a weight that overflowed in training
        w[N // 2, gs // 2] = float("inf")
        w[0, K - 1] = float("nan")
    got = P.rtn_quantize(w.to(DEV), gs, sym)
    general = P.rtn_quantize(_off_by_one(w.to(DEV)), gs, sym)
    for a, b in zip(got, general):
        assert a.shape == b.shape
        assert np.array_equal(a.cpu().numpy().view(np.uint8), b.cpu().numpy().view(np.uint8))
    if sym != "offset8" and dtype == torch.float16:
        packed, s, z = O.rtn_quantize(w.float().numpy(), gs, sym=bool(sym))
        assert np.array_equal(got[0].cpu().numpy(), packed)
        assert np.array_equal(got[1].cpu().numpy().view(np.uint32), s.view(np.uint32))
        assert np.array_equal(got[2].cpu().numpy(), z)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rtn_quotients_of_16_bit_weights(dtype):
    """Codes over every magnitude of the type below the group's extremes, for
    many ranges (scales): each quotient has to be the correctly rounded one,
    since exact ties decide codes."""
    bits = torch.arange(0, 1 << 15, dtype=torch.int32).to(torch.int16)
    v = bits.view(dtype).float()
    v = v[torch.isfinite(v) & (v < 0.06)]
    v = torch.cat([v, -v])
    g = torch.Generator().manual_seed(3)
    rows = []
    for hi in torch.rand(24, generator=g) * 0.05 + 0.01:
        lo = -hi * torch.rand(1, generator=g)
        x = torch.minimum(torch.maximum(v, lo), hi).to(dtype)
        x = x[torch.randperm(x.numel(), generator=g)][: x.numel() // 128 * 128]
        x = x.view(-1, 128)
        x[:, 0], x[:, 1] = hi.to(dtype), lo.to(dtype)
        rows.append(x)
    n = min(r.shape[0] for r in rows)
    w = torch.cat([r[:n] for r in rows])
    for sym in (False, "offset8"):
        got = P.rtn_quantize(w.to(DEV), 128, sym)
        general = P.rtn_quantize(_off_by_one(w.to(DEV)), 128, sym)
        assert all(torch.equal(a, b) for a, b in zip(got, general))
    packed, _, _ = O.rtn_quantize(w.float().numpy(), 128)
    assert np.array_equal(P.rtn_quantize(w.to(DEV), 128)[0].cpu().numpy(), packed)


@pytest.mark.parametrize("N,K,gs", SHAPES)
def test_repack_and_dequant_wide(N, K, gs):
    rng = np.random.default_rng(N * K)
    packed = torch.from_numpy(rng.integers(0, 256, (N, K // 2), dtype=np.uint8))
    s = torch.from_numpy(rng.standard_normal((N, K // gs, 1)).astype(np.float32))
    z = torch.from_numpy(rng.integers(0, 16, (N, K // gs, 1)).astype(np.float32))
    pd, sd, zd = packed.to(DEV), s.to(DEV), z.to(DEV)
    po = _off_by_one(pd)
    if gs % 32 == 0:
        want = O.repack_int4_for_kernel(packed.numpy(), gs)
        assert np.array_equal(P.repack_int4_for_kernel(pd, gs).cpu().numpy(), want)
        assert np.array_equal(P.repack_int4_for_kernel(po, gs).cpu().numpy(), want)
    ref = O.dequantize_packed(packed.numpy(), s.numpy(), z.numpy())
    for zz in (zd, zd.reshape(N, -1).to(torch.uint8)):
        for dtype in (torch.float32, torch.float16, torch.bfloat16):
            got = P.dequantize_int4(pd, sd, zz, gs, dtype=dtype)
            general = P.dequantize_int4(po, sd, zz, gs, dtype=dtype)
            assert torch.equal(got, torch.from_numpy(ref).to(DEV).to(dtype))
            assert torch.equal(got, general)


@pytest.mark.parametrize("N,G", [(1, 1), (31, 33), (32, 32), (4100, 3), (70, 148)])
def test_sz_group_major_tiles(N, G):
    rng = np.random.default_rng(N + G)
    s = torch.from_numpy(rng.standard_normal((N, G)).astype(np.float32)).to(DEV)
    z = torch.from_numpy(rng.integers(0, 16, (N, G)).astype(np.float32)).to(DEV)
    for zz in (z, z.to(torch.uint8)):
        s_gm, z_gm = P.sz_group_major(s, zz)
        assert torch.equal(s_gm, s.t().contiguous())
        assert torch.equal(z_gm, z.t().contiguous().to(torch.uint8))
    bad = z.clone()
    bad[N - 1, G - 1] = 16.0   # the last element: counted once, whatever the padding
    with pytest.raises(ValueError, match="^1 zero points"):
        P.sz_group_major(s, bad)
