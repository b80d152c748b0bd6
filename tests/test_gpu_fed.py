"""GPU: the ring kernel of lx_gemm_w with loader wavefronts (NVFP4 weights) against the tile kernels, bit for bit: every kernel that is built
(row tiles, one to four slices), ragged rows and columns, rows that end inside a stage, a slice and before the last slice; the epilogue's
operands, strides and activation scales; from a graph as well. Every case asks the library first whether the kernel takes it."""

import ctypes

import pytest
import torch

import ops
from dromos_amd.abi import BF16, DTYPE, F32, FORMATS, MATH_BF16, MATH_FP4, MATH_FP8
from dromos_amd.formats import random_weight

pytestmark = pytest.mark.gpu
NVFP4 = FORMATS["nvfp4"]
# Rows, columns, K; slices. The last three: one slice of many stages, where the other slice's wavefronts have none, and of 64 x 30001 x 4096's loaders of activations
# the one without stages asks for lines ahead (70 a workgroup, the first 64 are the other's).
CASES = [(9, 8209, 1088, 2), (16, 8250, 4416, 3), (17, 8241, 3200, 4), (32, 8211, 6464, 4), (20, 16401, 4096, 2), (25, 16433, 1088, 2), (33, 12301, 6464, 4), (48, 8207, 8704, 3),
         (40, 8225, 4416, 3), (34, 30001, 1024, 1), (49, 30001, 1088, 1), (64, 14336, 4096, 4), (63, 14330, 4160, 3), (50, 12301, 2176, 3), (64, 17003, 2176, 2), (57, 16385, 1024, 1),
         (64, 8197, 10304, 4), (17, 29003, 3392, 1), (49, 28977, 6208, 1), (64, 30001, 4096, 1)]


def plan(hip, M, N, K):
    return hip.lib.dromos_plan_fed(NVFP4, M, N, K, 0, 1)


@pytest.fixture(autouse=True)
def clear_table(hip):
    yield
    hip.lib.lx_tune_clear()


def tiles(hip, x, w, y, math=MATH_BF16, **kw):
    (M, K), N = x.shape, y.shape[1]
    assert hip.lib.lx_tune_force(b"gemm_w_nvfp4", M, N, K, 0) == 0
    try:
        return ops.gemm_w(hip, x, w, math, y=y.clone(), **kw)
    finally:
        hip.lib.lx_tune_clear()


@pytest.mark.parametrize("M,N,K,slices", CASES)
def test_gives_the_tile_kernels_bits(hip, M, N, K, slices):
    assert plan(hip, M, N, K) == slices
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = random_weight(NVFP4, N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), device="cuda")
    assert torch.equal(ops.gemm_w(hip, x, w, MATH_BF16, y=y.clone()), tiles(hip, x, w, y))
    y = torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    for kw in ({"alpha": 0.5}, {"bias": torch.randn(N, generator=g, device="cuda"), "alpha": 1.5, "beta": 0.25}):
        assert torch.equal(ops.gemm_w(hip, x, w, MATH_BF16, y=y.clone(), **kw), tiles(hip, x, w, y, **kw))


def test_strides_and_graph(hip):
    M, N, K, pad = 50, 8712, 4416, 64
    assert plan(hip, M, N, K) > 0
    w = random_weight(NVFP4, N, K, 5).to("cuda")
    x = torch.randn(M, K + pad, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).cuda()
    want = tiles(hip, x[:, :K].contiguous(), w, torch.empty(M, N, device="cuda"))
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


# The activations' scales in the epilogue.
@pytest.mark.parametrize("math", [MATH_FP8, MATH_FP4])
@pytest.mark.parametrize("M,N,K", [(17, 8241, 3200), (64, 14336, 4096)])
def test_under_the_maths_of_activation_images(hip, math, M, N, K):
    assert plan(hip, M, N, K) > 0
    g = torch.Generator(device="cuda").manual_seed(M)
    w = random_weight(NVFP4, N, K, N + K).to("cuda")
    x = (torch.randn(M, K, generator=g, device="cuda") * torch.rand(M, 1, generator=g, device="cuda")).to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), device="cuda")
    assert torch.equal(ops.gemm_w(hip, x, w, math, y=y.clone()), tiles(hip, x, w, y, math=math))


# An infinity and a NaN among one row's activations reach that row only, at the row's end as well.
def test_activations_that_are_not_finite(hip):
    M, N, K = 33, 8250, 4416
    assert plan(hip, M, N, K) > 0
    w = random_weight(NVFP4, N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16).cuda()
    clean = ops.gemm_w(hip, x, w, MATH_BF16, y=torch.empty(M, N, device="cuda"))
    x[3, K - 1], x[32, 0] = float("nan"), float("inf")
    got = ops.gemm_w(hip, x, w, MATH_BF16, y=torch.empty(M, N, device="cuda"))
    assert bool(got[3].isnan().all()) and not bool(got[32].isfinite().all())
    got[[3, 32]] = clean[[3, 32]]
    assert torch.equal(got, clean)
