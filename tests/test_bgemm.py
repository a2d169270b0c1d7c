"""The big-tile GEMM beyond its fp16, 128-column-group, tiled-copy case (which
tests/test_tgemm.py covers): group sizes 32 and 64, bf16, callers without the
tiled or group-major copies, split K, act_order, ragged M, N and K.

Each case runs through the public operator, is compared with a float64 product
of the oracle's dequantised weights under a bound derived from the arithmetic,
and with the GEMV (the general path, forced) under twice that bound."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import pare_amd as P
from oracle import pare_oracle as O
from pare_amd import _lib
from pare_amd.kernels import force_kernel, kernel_route

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _case(N, K, gs, seed, act_order):
    w = (torch.randn(N, K, generator=torch.Generator().manual_seed(seed)) * 0.02).numpy()
    perm = None
    if act_order:
        packed, s, z, g_idx = O.rtn_quantize_act_order(
            w, np.random.default_rng(seed).permutation(K), gs)
        w_hat = O.dequantize_gidx(O.unpack_int4(packed), s, z, g_idx)
        perm = P.perm_from_g_idx(torch.from_numpy(g_idx).to(DEV), gs)
    else:
        packed, s, z = O.rtn_quantize(w, gs)
        w_hat = O.dequantize_packed(packed, s, z)
    wk = P.repack_int4_for_kernel(torch.from_numpy(packed).to(DEV), gs, perm=perm)
    return wk, torch.from_numpy(s).to(DEV), P.zeros_to_u8(torch.from_numpy(z).to(DEV)), perm, w_hat


def _bound(x, w_hat, s, gs, bf16):
    """Output rounding (half an ulp of 11 or 8 bits) plus the fp32 sums: at most
    K + G + 4 roundings of 2^-24 of the sum of the terms' sizes, |x| s 15 in fp16
    and, in bf16, |x| s (143 + 143) for the products with 128 + q and their
    correction by 128 + z."""
    K = x.shape[1]
    scale = np.repeat(s.cpu().numpy().reshape(w_hat.shape[0], -1), gs, axis=1)[:, :K]
    size = np.abs(x) @ np.abs(scale).T * (286.0 if bf16 else 15.0)
    ref = x @ w_hat.astype(np.float64).T
    return ref, np.abs(ref) * 2.0 ** (-8 if bf16 else -11) + size * (K + K // gs + 4) * 2.0 ** -24 + 2.0 ** -25


@pytest.mark.parametrize("M,N,K,gs,bf16,copies,act_order", [
    # gs 64 / 32 on the tiled copy: split K, one tile of rows and its edges, no split
    (205, 4096, 4096, 64, False, True, False), (224, 3844, 4096, 64, False, True, False),
    (400, 14300, 1536, 64, False, True, False), (385, 4100, 2048, 32, False, True, False),
    (90, 2560, 14336, 32, False, True, True),
    # bf16, every group size, tiled copy and row-major weights
    (25, 14000, 1536, 128, True, True, False), (113, 4100, 1536, 128, True, True, False),
    (225, 2060, 2048, 256, True, True, True), (97, 516, 1536, 64, True, True, False),
    (193, 260, 1536, 32, True, True, False), (112, 772, 384, 128, True, False, False),
    (130, 516, 1152, 64, True, False, True), (96, 68, 640, 32, True, False, False),
    (12, 16644, 2048, 128, True, False, False), (640, 14340, 256, 128, True, False, False),
    # fp16 without the copies: column counts and group sizes only the GEMV reads
    (25, 260, 384, 128, False, False, False), (60, 1028, 1408, 128, False, False, True),
    (33, 64, 128, 64, False, False, False), (225, 516, 1152, 64, False, False, False),
    (97, 900, 160 * 4, 32, False, False, False), (12, 16644, 2048, 32, False, False, True),
    # fp16 with the copies: few tiles, K split or not
    (639, 2060, 14336, 128, False, True, False), (1153, 4096, 4096, 128, False, True, True),
    # the fewest rows that leave the GEMV
    (17, 516, 1536, 128, True, False, False), (17, 1028, 1152, 64, False, False, True),
    # the edges of the 64-row tile: up to 64 rows, and past one taller tile up to 128
    (64, 772, 1408, 128, True, True, False), (65, 772, 1408, 128, True, True, False),
    (48, 4100, 1536, 32, True, True, True), (64, 516, 1536, 64, True, True, False),
    (113, 260, 1152, 64, True, False, False), (128, 516, 640, 32, True, False, False),
    (129, 516, 640, 32, True, False, False), (128, 17156, 256, 128, True, False, False),
    (64, 516, 1408, 128, False, False, False), (65, 516, 1408, 64, False, False, False),
    (128, 516, 1152, 64, False, False, False), (97, 4100, 14336, 32, False, True, False),
    # fp16 without the copies, large enough to leave the register-streamed GEMM
    (769, 5636, 4096, 128, False, False, False),
])
def test_bgemm_routes_against_fp64_and_the_gemv(M, N, K, gs, bf16, copies, act_order):
    wk, s, zu8, perm, w_hat = _case(N, K, gs, M + N % 101, act_order)
    kw = {"perm": perm}
    if copies:
        kw.update(sz_gm=P.sz_group_major(s, zu8), w_tiled=P.tile_w4a16(wk, gs))
    print(f"[case] bgemm M={M} N={N} K={K} gs={gs} bf16={bf16} copies={copies} act={act_order}", flush=True)
    assert kernel_route(M, N, K, gs, torch.bfloat16 if bf16 else torch.float16, tiled=copies,
                        perm=act_order) == "bgemm"
    op = P.matmul_w4a16_bf16 if bf16 else P.matmul_w4a16
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).to(
        torch.bfloat16 if bf16 else torch.float16)
    xd = x.to(DEV)
    y = op(xd, wk, s, zu8, gs, **kw)
    y2 = op(xd, wk, s, zu8, gs, **kw)
    with force_kernel("gemv"):
        yg = op(xd, wk, s, zu8, gs, **kw)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    # act_order: w_hat is in the original column order, so the scales of a row
    # are only bounded by their largest
    if act_order:
        s = s.reshape(N, -1).amax(1, keepdim=True).expand(N, K // gs)
    ref, bound = _bound(x.double().numpy(), w_hat, s, gs, bf16)
    err = np.abs(y.double().cpu().numpy() - ref)
    assert (err <= bound).all(), f"max {np.max(err / bound):.2f} of the bound"
    diff = np.abs(y.double().cpu().numpy() - yg.double().cpu().numpy())
    assert (diff <= 2 * bound).all(), f"against the GEMV: {np.max(diff / bound):.2f} of the bound"


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("what", ["mean", "outlier"])
def test_bgemm_bf16_under_cancellation(gs, what):
    """Activations with a large common offset, and outlier columns whose codes equal
    their zero points: products with 128 + q that cancel against the row sums.
    They are about 2^-24 143 max|x| s of error per rounding, a dozen roundings a
    group: against sums of sqrt(K) 4.6 s (offset 100: 100 times that) below 2e-4
    of y, where its rounding to bf16 is 1.7e-3 of it, so 2 % beside that."""
    M, N, K = 96, 516, 4096
    g = torch.Generator(device=DEV).manual_seed(1)
    q = torch.randint(0, 16, (N, K), generator=g, device=DEV, dtype=torch.uint8)
    z = torch.randint(0, 16, (N, K // gs), generator=g, device=DEV, dtype=torch.uint8)
    s = torch.rand(N, K // gs, generator=g, device=DEV) * 0.004 + 0.001
    x = torch.randn(M, K, generator=g, device=DEV)
    if what == "mean":
        x += 100.0
    else:
        for c in (5, gs + 3):
            q[:, c], x[:, c] = z[:, c // gs], 1000.0
    x = x.bfloat16()
    wk = P.repack_int4_for_kernel(q[:, 0::2] | (q[:, 1::2] << 4), gs)
    w = ((q.double().reshape(N, -1, gs) - z.double()[..., None]) * s.double()[..., None]).reshape(N, K)
    ref = x.double() @ w.t()
    assert kernel_route(M, N, K, gs, torch.bfloat16) == "bgemm"
    y = P.matmul_w4a16_bf16(x, wk, s, z, gs).double()
    rounding = (ref.bfloat16().double() - ref).norm()
    assert (y - ref).norm() <= 1.02 * rounding


def test_bgemm_route_needs_no_workspace_and_no_alignment_of_y():
    """With no workspace, or a y that is not 8-byte aligned, bf16 calls of many
    rows run on the GEMV as before, through the C ABI."""
    M, N, K, gs = 64, 512, 1536, 128
    wk, s, zu8, _, _ = _case(N, K, gs, 5, False)
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)).bfloat16()
    s2 = s.reshape(N, -1).contiguous()
    L = _lib.lib()
    buf = torch.zeros(M * N + 4, dtype=torch.bfloat16, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def call(y, ws):
        return L.pmi_matmul_w4a16(x.data_ptr(), _lib.PMI_BF16, wk.data_ptr(), s2.data_ptr(),
                                  zu8.data_ptr(), _lib.PMI_U8, None, None, None, None, None,
                                  y.data_ptr(), _lib.PMI_BF16, M, N, K, gs,
                                  ws.data_ptr() if ws is not None else None,
                                  ws.numel() if ws is not None else 0, stream)

    with force_kernel("gemv"):
        want = P.matmul_w4a16_bf16(x, wk, s, zu8, gs)
    ws = torch.zeros(L.pmi_matmul_best_workspace_bytes(M, N, K, gs, 0), dtype=torch.uint8, device=DEV)
    for y, w in ((buf[:M * N], None), (buf[1:M * N + 1], ws)):
        assert call(y, w) == 0, _lib.last_error()
        torch.cuda.synchronize()
        assert torch.equal(y.view(M, N).view(torch.int16), want.view(torch.int16))


def test_bgemm_split_without_its_workspace_runs_elsewhere():
    """Few tiles and no room for their split: the call runs on the kernel that
    it would run on without the tiled copy (same bits), through the C ABI."""
    M, N, K, gs = 639, 2060, 14336, 128
    L = _lib.lib()
    assert L.pmi_matmul_kernel_choice(M, N, K, gs, _lib.PMI_CHOICE_TILED) == 6
    assert L.pmi_matmul_kernel_choice(M, N, K, gs, 0) == 4
    g = torch.Generator(device=DEV).manual_seed(4)
    wk = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8, device=DEV)
    s = torch.rand(N, K // gs, generator=g, device=DEV) * 0.01 + 1e-3
    z = torch.randint(0, 16, (N, K // gs), generator=g, dtype=torch.uint8, device=DEV)
    x = torch.randn(M, K, generator=g, device=DEV).half()
    s_gm, z_gm = P.sz_group_major(s, z)
    wt = P.tile_w4a16(wk, gs)
    stream = torch.cuda.current_stream().cuda_stream
    out = []
    for tiled in (wt.data_ptr(), None):
        y = torch.full((M, N), float("nan"), dtype=torch.float16, device=DEV)
        rc = L.pmi_matmul_w4a16(x.data_ptr(), _lib.PMI_F16, wk.data_ptr(), s.data_ptr(), z.data_ptr(),
                                _lib.PMI_U8, None, None, s_gm.data_ptr(), z_gm.data_ptr(), tiled,
                                y.data_ptr(), _lib.PMI_F16, M, N, K, gs, None, 0, stream)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        out.append(y)
    assert torch.equal(out[0].view(torch.int16), out[1].view(torch.int16))


@pytest.mark.parametrize("M,N,K,gs,bf16,copies,kernel", [
    (301, 4096, 14336, 64, False, True, "tgemm"), (65, 4096, 14336, 64, False, True, "tgemm"),
    (193, 4100, 4096, 32, False, True, "tgemm"), (1024, 1024, 18944, 128, False, False, "gemm64"),
    (17, 512, 14336, 128, True, False, "gemv"), (28, 4096, 4096, 64, False, False, "gemv"),
])
def test_bgemm_leaves_few_tiles_whose_split_has_no_room(M, N, K, gs, bf16, copies, kernel):
    """With the workspace that pmi_matmul_workspace_bytes reports, or one that
    holds all but the partial tiles, such calls run on the kernel that took them
    before (same bits), through the C ABI: unsplit they would occupy 2-80 CUs."""
    L = _lib.lib()
    g = torch.Generator(device=DEV).manual_seed(4)
    wk = torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8, device=DEV)
    s = torch.rand(N, K // gs, generator=g, device=DEV) * 0.01 + 1e-3
    z = torch.randint(0, 16, (N, K // gs), generator=g, dtype=torch.uint8, device=DEV)
    dtype, code = (torch.bfloat16, _lib.PMI_BF16) if bf16 else (torch.float16, _lib.PMI_F16)
    x = torch.randn(M, K, generator=g, device=DEV).to(dtype)
    gm = P.sz_group_major(s, z) if copies else None
    wt = P.tile_w4a16(wk, gs) if copies else None
    stream = torch.cuda.current_stream().cuda_stream

    def call(nbytes):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=DEV) if nbytes else None
        y = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
        rc = L.pmi_matmul_w4a16(x.data_ptr(), code, wk.data_ptr(), s.data_ptr(), z.data_ptr(), _lib.PMI_U8,
                                None, None, gm[0].data_ptr() if gm else None, gm[1].data_ptr() if gm else None,
                                wt.data_ptr() if copies else None, y.data_ptr(), code, M, N, K, gs,
                                ws.data_ptr() if nbytes else None, nbytes, stream)
        assert rc == 0, _lib.last_error()
        torch.cuda.synchronize()
        return y

    base = L.pmi_matmul_workspace_bytes(M, N, K, gs, 0)
    print(f"[case] no room M={M} N={N} K={K} gs={gs} bf16={bf16} base={base}", flush=True)
    assert L.pmi_matmul_best_workspace_bytes(M, N, K, gs, 0) > max(base, 2 << 20)
    for nbytes in (base, 2 << 20):
        with force_kernel(kernel):
            want = call(nbytes)
        assert torch.equal(call(nbytes).view(torch.int16), want.view(torch.int16)), nbytes


@pytest.mark.parametrize("bf16,gs", [(True, 128), (False, 64)])
def test_bgemm_in_a_captured_graph(bf16, gs):
    """A captured call that no eager call warmed up (its workspace then belongs
    to the graph), replayed with eager work of the same shape in between."""
    M, N, K = 130, 1028, 1152
    wk, s, zu8, _, _ = _case(N, K, gs, 9, False)
    op = P.matmul_w4a16_bf16 if bf16 else P.matmul_w4a16
    x = torch.randn(M, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(2))
    x = x.bfloat16() if bf16 else x.half()
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        y = op(x, wk, s, zu8, gs)
    for k in range(3):
        x.add_(1.0)
        want = op(x, wk, s, zu8, gs)
        with torch.cuda.stream(side):
            eager = op(x, wk, s, zu8, gs)
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int16), want.view(torch.int16)), k
        assert torch.equal(eager.view(torch.int16), want.view(torch.int16)), k


def test_bgemm_graph_replays_beside_eager_work_on_its_capture_stream():
    """A graph captured on a stream whose eager calls use the same scratch,
    replayed on another stream while that one is busy: row sums and partial
    tiles of the two stay apart."""
    M, N, K, gs = 130, 1028, 4096, 128
    wk, s, zu8, _, _ = _case(N, K, gs, 9, False)
    g = torch.Generator(device=DEV).manual_seed(2)
    x, xe = (torch.randn(M, K, device=DEV, generator=g).bfloat16() for _ in range(2))
    want, want_e = (P.matmul_w4a16_bf16(v, wk, s, zu8, gs) for v in (x, xe))
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        P.matmul_w4a16_bf16(xe, wk, s, zu8, gs)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        y = P.matmul_w4a16_bf16(x, wk, s, zu8, gs)
    for _ in range(4):
        got, eager = [], []
        for _ in range(16):
            with torch.cuda.stream(side):
                eager.append(P.matmul_w4a16_bf16(xe, wk, s, zu8, gs))
            graph.replay()
            got.append(y.clone())
        torch.cuda.synchronize()
        for a, b in zip(got, eager):
            assert torch.equal(a.view(torch.int16), want.view(torch.int16))
            assert torch.equal(b.view(torch.int16), want_e.view(torch.int16))
