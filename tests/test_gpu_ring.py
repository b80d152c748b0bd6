"""GPU: the ring kernel of lx_gemm_w (up to 64 bf16 rows on wide matrices) against the tile kernels, bit for bit: two, three and four
slices, 32 and 64 weight rows a workgroup, ragged rows and columns, rows that end inside a stage and inside a slice; the epilogue's
operands and strides; from a graph as well."""

import ctypes

import pytest
import torch

import ops
from dromos_amd.abi import BF16, DTYPE, F32, FORMATS, MATH_BF16
from dromos_amd.formats import random_weight

pytestmark = pytest.mark.gpu
# N: 290 .. 1000 tiles; K: whole stages, and rows cut short in every format's way.
CASES = [("nvfp4", m, n, k) for m, n, k in [(17, 4625, 2048), (33, 8190, 2112), (48, 6400, 3136), (64, 14336, 4032), (49, 15999, 4096), (40, 8208, 11008)]]
CASES += [("bf16", m, n, k) for m, n, k in [(9, 6145, 4096), (16, 8190, 2056), (33, 12001, 4104), (48, 6400, 8200), (64, 14336, 3072)]]
CASES += [(f, m, n, k) for f in ("int8", "fp8") for m, n, k in [(17, 6145, 4096), (32, 8190, 4112), (48, 7008, 8192), (49, 8705, 4096), (33, 16127, 5136), (64, 14336, 8176)]]


@pytest.fixture(autouse=True)
def clear_table(hip):
    yield
    hip.lib.lx_tune_clear()


def tiles(hip, fmt, x, w, y, **kw):
    (M, K), N = x.shape, y.shape[1]
    assert hip.lib.lx_tune_force(f"gemm_w_{fmt}".encode(), M, N, K, 0) == 0
    try:
        return ops.gemm_w(hip, x, w, MATH_BF16, y=y.clone(), **kw)
    finally:
        hip.lib.lx_tune_clear()


@pytest.mark.parametrize("fmt,M,N,K", CASES)
def test_ring_gives_the_tile_kernels_bits(hip, fmt, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = random_weight(FORMATS[fmt], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), device="cuda")
    assert torch.equal(ops.gemm_w(hip, x, w, MATH_BF16, y=y.clone()), tiles(hip, fmt, x, w, y))
    y = torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    for kw in ({"alpha": 0.5}, {"bias": torch.randn(N, generator=g, device="cuda"), "alpha": 1.5, "beta": 0.25}):
        assert torch.equal(ops.gemm_w(hip, x, w, MATH_BF16, y=y.clone(), **kw), tiles(hip, fmt, x, w, y, **kw))


@pytest.mark.parametrize("fmt", ["bf16", "int8", "fp8", "nvfp4"])
def test_ring_strides_and_graph(hip, fmt):
    M, N, K, pad = 50, 8704, 4096, 8
    w = random_weight(FORMATS[fmt], N, K, 5).to("cuda")
    x = torch.randn(M, K + pad, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).cuda()
    want = tiles(hip, fmt, x[:, :K].contiguous(), w, torch.empty(M, N, device="cuda"))
    struct, stream, graph = w.lx(), ctypes.c_void_p(), ctypes.c_void_p()
    y = torch.full((M, N + 1), -3.0, device="cuda")
    torch.cuda.synchronize()
    assert hip.lib.lx_rt_stream_create(ctypes.byref(stream)) == 0
    try:
        assert hip.lib.lx_rt_capture_begin(stream) == 0
        assert hip.status("gemm_w", x, BF16, K + pad, ctypes.pointer(struct), MATH_BF16, None, F32, y, DTYPE[y.dtype], N + 1, M, N, K, 1.0, 0.0, None, stream.value) == 0
        assert hip.lib.lx_rt_capture_end(stream, ctypes.byref(graph)) == 0
        for _ in range(3):
            y.fill_(-3.0)
            torch.cuda.synchronize()
            assert hip.lib.lx_rt_graph_launch(graph, stream) == 0 and hip.lib.lx_rt_stream_sync(stream) == 0
            assert torch.equal(y[:, :N], want) and bool((y[:, N:] == -3.0).all())
        assert hip.lib.lx_rt_graph_destroy(graph) == 0
    finally:
        assert hip.lib.lx_rt_stream_destroy(stream) == 0


# An infinity among a bf16 row's last values: what lies past the row's end must not meet it.
def test_ring_infinite_weights_at_the_rows_end(hip):
    M, N, K = 20, 12008, 4104
    w = random_weight(FORMATS["bf16"], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16).cuda()
    clean = ops.gemm_w(hip, x, w, MATH_BF16, y=torch.empty(M, N, device="cuda"))
    w.data[3, K - 1], w.data[N - 1, K - 8] = float("inf"), float("-inf")
    got = ops.gemm_w(hip, x, w, MATH_BF16, y=torch.empty(M, N, device="cuda"))
    assert torch.equal(got[:, 3], x[:, K - 1].float() * float("inf")) and torch.equal(got[:, N - 1], x[:, K - 8].float() * -float("inf"))
    got[:, [3, N - 1]] = clean[:, [3, N - 1]]
    assert torch.equal(got, clean)
