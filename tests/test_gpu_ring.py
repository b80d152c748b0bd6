"""GPU: the ring kernel of lx_gemm_w (up to 64 bf16 rows on wide matrices) against the tile kernels, bit for bit: every kernel that is
built (row tiles, two to four slices, 32 and 64 weight rows a workgroup), ragged rows and columns, rows that end inside a stage and inside a slice;
the epilogue's operands, strides and activation scales; from a graph as well. Every case asks the library first whether the ring takes it."""

import ctypes

import pytest
import torch

import ops
from dromos_amd.abi import BF16, DTYPE, F32, FORMATS, MATH_BF16, MATH_FP4, MATH_FP8
from dromos_amd.formats import random_weight

pytestmark = pytest.mark.gpu
# Row tiles 1 .. 4; 8 * columns a workgroup + slices.
CASES = [("nvfp4", *c) for c in [(17, 4625, 2048, 258), (33, 7190, 2048, 258), (63, 7001, 2048, 258), (25, 16007, 2112, 514), (35, 10274, 2048, 514), (51, 11853, 2048, 514),
                                 (50, 12000, 2112, 259), (40, 8208, 2112, 515), (17, 5201, 3136, 260), (33, 5762, 3136, 260), (64, 8209, 4032, 260), (48, 6400, 4096, 260),
                                 (24, 11047, 3392, 516), (40, 11047, 3392, 516), (40, 10288, 11008, 516)]]
CASES += [("bf16", *c) for c in [(9, 7345, 4608, 260), (30, 7414, 6144, 260), (33, 8001, 4104, 260), (64, 7001, 2056, 259), (16, 12293, 2560, 516), (17, 13930, 3072, 516),
                                 (34, 10109, 3072, 516), (64, 11697, 5120, 516)]]
CASES += [(f, *c) for f in ("int8", "fp8") for c in [(17, 5182, 4096, 260), (32, 5937, 6144, 260), (33, 7990, 4112, 259), (51, 7442, 4976, 260), (36, 12922, 5120, 516), (52, 11697, 5120, 516)]]


def plan(hip, fmt, M, N, K):
    return hip.lib.dromos_plan_ring(FORMATS[fmt], M, N, K, 0, 1, None)


@pytest.fixture(autouse=True)
def clear_table(hip):
    yield
    hip.lib.lx_tune_clear()


def tiles(hip, fmt, x, w, y, math=MATH_BF16, **kw):
    (M, K), N = x.shape, y.shape[1]
    assert hip.lib.lx_tune_force(f"gemm_w_{fmt}".encode(), M, N, K, 0) == 0
    try:
        return ops.gemm_w(hip, x, w, math, y=y.clone(), **kw)
    finally:
        hip.lib.lx_tune_clear()


@pytest.mark.parametrize("fmt,M,N,K,taken", CASES)
def test_ring_gives_the_tile_kernels_bits(hip, fmt, M, N, K, taken):
    assert plan(hip, fmt, M, N, K) == taken
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
    M, N, K, pad = 50, 8704, 4096, 64
    assert plan(hip, fmt, M, N, K) > 0
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
    M, N, K = 33, 8008, 4104
    assert plan(hip, "bf16", M, N, K) == 260
    w = random_weight(FORMATS["bf16"], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16).cuda()
    clean = ops.gemm_w(hip, x, w, MATH_BF16, y=torch.empty(M, N, device="cuda"))
    w.data[3, K - 1], w.data[N - 1, K - 8] = float("inf"), float("-inf")
    got = ops.gemm_w(hip, x, w, MATH_BF16, y=torch.empty(M, N, device="cuda"))
    assert torch.equal(got[:, 3], x[:, K - 1].float() * float("inf")) and torch.equal(got[:, N - 1], x[:, K - 8].float() * -float("inf"))
    got[:, [3, N - 1]] = clean[:, [3, N - 1]]
    assert torch.equal(got, clean)


# The activations' scales in the epilogue.
@pytest.mark.parametrize("math", [MATH_FP8, MATH_FP4])
@pytest.mark.parametrize("M,N,K", [(17, 4625, 2048), (40, 11047, 3392), (64, 8209, 4032)])
def test_ring_under_the_maths_of_activation_images(hip, math, M, N, K):
    assert plan(hip, "nvfp4", M, N, K) > 0
    g = torch.Generator(device="cuda").manual_seed(M)
    w = random_weight(FORMATS["nvfp4"], N, K, N + K).to("cuda")
    x = (torch.randn(M, K, generator=g, device="cuda") * torch.rand(M, 1, generator=g, device="cuda")).to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), device="cuda")
    assert torch.equal(ops.gemm_w(hip, x, w, math, y=y.clone()), tiles(hip, "nvfp4", x, w, y, math=math))


# A table entry keeps a call from the ring kernel, so the tuner stores none where the ring is faster than every variant (here about
# half of the best one's time), and still stores the fastest where another kernel takes the call.
def test_the_tuner_leaves_the_rings_calls_to_it(hip):
    from dromos_amd import tune

    M, N, K = 40, 8192, 2048
    assert plan(hip, "nvfp4", M, N, K) > 0
    got = tune.tune(hip, "gemm_w_nvfp4", M, N, K, repeats=5)
    assert got["pick"] is None and hip.lib.lx_tune_get(b"gemm_w_nvfp4", M, N, K) == -1 and plan(hip, "nvfp4", M, N, K) > 0
    assert tune.time_own_rule(hip, "gemm_w_nvfp4", M, 2048, K) is None and tune.time_own_rule(hip, "gemv_w_fp8", 4, N, K) is None
