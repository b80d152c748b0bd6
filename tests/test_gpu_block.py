"""GPU: the block kernels (more rows than a decode step has) against the kernels for up to 64 rows, bit for bit: the same
rows in calls of 32 at most. Row counts, output counts and row lengths around the edges of blocks, K tiles, slices and
load steps; every format and math; the epilogue's operands; a stream with and without the partial-tile buffer."""

import ctypes

import pytest
import torch

import checks
import ops
from dromos_amd.abi import BF16, DTYPE, F32, FORMATS, MATH_BF16, MATH_FP4, MATH_FP8, MATH_INT8
from dromos_amd.formats import random_stack, random_weight

pytestmark = pytest.mark.gpu
MATHS = [("bf16", MATH_BF16), ("int8", MATH_BF16), ("fp8", MATH_BF16), ("nvfp4", MATH_BF16), ("int8", MATH_INT8), ("fp8", MATH_FP8),
         ("nvfp4", MATH_FP8), ("nvfp4", MATH_FP4)]


def chunks_of_32(hip, x, w, math, y, **kw):
    return torch.cat([ops.gemm_w(hip, x[m : m + 32].contiguous(), w, math, y=y[m : m + 32].clone(), **kw) for m in range(0, x.shape[0], 32)])


def on_a_stream(hip, buffer, x, w, math, y):
    """lx_gemm_w on a stream of the library's with or without its partial-tile buffer."""
    stream, struct = ctypes.c_void_p(), w.lx()
    (M, K), N = x.shape, y.shape[1]
    ws = torch.empty(max(256, int(hip.size("gemm_workspace_bytes", M, K, math))), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    assert hip.lib.lx_rt_stream_create(ctypes.byref(stream)) == 0
    assert buffer or hip.lib.lx_rt_stream_release(stream) == 0
    try:
        assert hip.status("gemm_w", x, DTYPE[x.dtype], x.shape[1], ctypes.pointer(struct), math, None, F32, y, DTYPE[y.dtype], y.shape[1], M, N, K, 1.0,
                          0.0, ws, stream.value) == 0
        assert hip.lib.lx_rt_stream_sync(stream) == 0
    finally:
        assert hip.lib.lx_rt_stream_destroy(stream) == 0
    return y


# Every block shape in every mode that the rule takes it in ("one slice a row", "added" in registers, "part": a slice a workgroup),
# each near the smallest product that it is taken for.
PLANS = ["one", "added", "part"]
SHAPES = ["64x64", "64x128", "128x128", "128x256"]
COVER = [("bf16", MATH_BF16, "one", "64x64", 66, 131, 224), ("bf16", MATH_BF16, "one", "64x128", 1605, 598, 224), ("bf16", MATH_BF16, "one", "128x128", 2312, 849, 256),
         ("bf16", MATH_BF16, "added", "64x64", 66, 129, 520), ("bf16", MATH_BF16, "added", "64x128", 1605, 598, 512), ("bf16", MATH_BF16, "added", "128x128", 2312, 849, 1064),
         ("bf16", MATH_BF16, "part", "64x64", 67, 139, 1184), ("bf16", MATH_BF16, "part", "64x128", 520, 132, 2336), ("bf16", MATH_BF16, "part", "128x128", 1097, 134, 2368),
         ("int8", MATH_BF16, "one", "64x64", 76, 139, 512), ("int8", MATH_BF16, "one", "64x128", 2086, 454, 512), ("int8", MATH_BF16, "one", "128x128", 2559, 806, 512),
         ("int8", MATH_BF16, "added", "64x64", 68, 131, 544), ("int8", MATH_BF16, "added", "64x128", 2368, 422, 544), ("int8", MATH_BF16, "added", "128x128", 2547, 789, 544),
         ("int8", MATH_BF16, "part", "64x64", 75, 130, 1344), ("int8", MATH_BF16, "part", "64x128", 782, 201, 2144), ("int8", MATH_BF16, "part", "128x128", 611, 513, 2592),
         ("fp8", MATH_BF16, "one", "64x64", 77, 131, 512), ("fp8", MATH_BF16, "one", "64x128", 2120, 470, 512), ("fp8", MATH_BF16, "one", "128x128", 2055, 1009, 512),
         ("fp8", MATH_BF16, "added", "64x64", 68, 136, 544), ("fp8", MATH_BF16, "added", "64x128", 2719, 330, 544), ("fp8", MATH_BF16, "added", "128x128", 1703, 1156, 544),
         ("fp8", MATH_BF16, "part", "64x64", 76, 133, 1312), ("fp8", MATH_BF16, "part", "64x128", 1124, 131, 2080), ("fp8", MATH_BF16, "part", "128x128", 901, 350, 2592),
         ("nvfp4", MATH_BF16, "one", "64x64", 68, 134, 512), ("nvfp4", MATH_BF16, "one", "64x128", 1843, 520, 512), ("nvfp4", MATH_BF16, "one", "128x128", 3014, 643, 512),
         ("nvfp4", MATH_FP4, "one", "128x256", 1719, 2384, 512), ("nvfp4", MATH_BF16, "added", "64x64", 129, 257, 1056),
         ("nvfp4", MATH_FP8, "added", "64x128", 1129, 897, 1056), ("nvfp4", MATH_BF16, "added", "128x128", 2181, 905, 1056),
         ("nvfp4", MATH_BF16, "added", "128x256", 1667, 2413, 1088), ("nvfp4", MATH_BF16, "part", "64x64", 95, 130, 2048), ("nvfp4", MATH_BF16, "part", "64x128", 802, 264, 3264),
         ("nvfp4", MATH_FP4, "part", "128x128", 1603, 195, 4640), ("nvfp4", MATH_BF16, "part", "128x256", 643, 743, 7264),
         ("int8", MATH_INT8, "one", "64x64", 68, 133, 512), ("int8", MATH_INT8, "one", "64x128", 1497, 641, 512), ("int8", MATH_INT8, "one", "128x128", 2411, 847, 512),
         ("int8", MATH_INT8, "one", "128x256", 2404, 1702, 528), ("int8", MATH_INT8, "part", "64x64", 71, 136, 1408), ("int8", MATH_INT8, "part", "64x128", 782, 194, 2112),
         ("int8", MATH_INT8, "part", "128x128", 1606, 195, 2368), ("int8", MATH_INT8, "part", "128x256", 2883, 130, 3648),
         ("fp8", MATH_FP8, "one", "64x64", 85, 137, 512), ("fp8", MATH_FP8, "one", "64x128", 783, 4663, 512), ("fp8", MATH_FP8, "one", "128x128", 1311, 1548, 512),
         ("fp8", MATH_FP8, "one", "128x256", 2255, 10704, 512), ("fp8", MATH_FP8, "added", "64x64", 73, 132, 608), ("fp8", MATH_FP8, "added", "64x128", 1073, 3631, 544),
         ("fp8", MATH_FP8, "added", "128x128", 2065, 1001, 560), ("fp8", MATH_FP8, "added", "128x256", 2749, 8363, 576), ("fp8", MATH_FP8, "part", "64x64", 82, 130, 1376),
         ("fp8", MATH_FP8, "part", "64x128", 777, 258, 6240), ("fp8", MATH_FP8, "part", "128x128", 773, 464, 2240)]


@pytest.mark.parametrize("fmt,math,mode,shape,M,N,K", COVER)
def test_every_shape_and_mode(hip, fmt, math, mode, shape, M, N, K):
    buffer = mode == "part"
    assert hip.lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, 0, buffer) == 4 * PLANS.index(mode) + SHAPES.index(shape)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = random_weight(FORMATS[fmt], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    y = torch.full((M, N), float("nan"), device="cuda")
    assert torch.equal(on_a_stream(hip, buffer, x, w, math, y.clone()), chunks_of_32(hip, x, w, math, y))


# The INT8 math's sums are whole numbers, so K is cut as is estimated fastest: slices that are not the row's own, the last of them shorter, rows
# that end inside a K tile, on every block shape; and where no number of slices fits the partial-tile buffer, none.
@pytest.mark.parametrize("M,N,K,plan", [(193, 2703, 6528, 10), (515, 4096, 11008, 11), (437, 2608, 10016, 10), (585, 608, 4992, 9), (545, 576, 2752, 8), (133, 1968, 5136, 10),
                                        (430, 5216, 13344, 11), (4000, 4096, 4096, None)])
def test_int8_math_in_slices_of_its_own(hip, M, N, K, plan):
    got = hip.lib.dromos_plan_gemm(FORMATS["int8"], MATH_INT8, M, N, K, 0, 1)
    assert got == plan if plan else got // 4 != 2
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = random_weight(FORMATS["int8"], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    for y in (torch.full((M, N), float("nan"), device="cuda"), torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16)):
        want = on_a_stream(hip, False, x, w, MATH_INT8, y.clone())
        assert torch.equal(on_a_stream(hip, True, x, w, MATH_INT8, y.clone()), want)
    assert torch.equal(chunks_of_32(hip, x[:64].contiguous(), w, MATH_INT8, y[:64].clone()), want[:64])



# The wide block (128 x 256, plan shape 16): blocks cut short in rows and columns, odd and even numbers of columns, rows that end
# inside a stage of K and inside its pieces, two stages past a slice, the epilogue's operands.
WIDE = [("int8", MATH_BF16, 20, 834, 7039, 1568, 0), ("int8", MATH_BF16, 20, 1921, 3332, 1600, 1), ("fp8", MATH_BF16, 20, 2731, 2203, 1568, 2), ("fp8", MATH_BF16, 20, 769, 7668, 1600, 0),
        ("nvfp4", MATH_BF16, 20, 518, 7603, 1856, 0), ("nvfp4", MATH_BF16, 20, 897, 4612, 1984, 1), ("nvfp4", MATH_FP4, 20, 3896, 1033, 1856, 2), ("nvfp4", MATH_FP8, 20, 1512, 2703, 1856, 0),
        ("int8", MATH_INT8, 16, 2691, 1491, 2336, 0), ("int8", MATH_INT8, 16, 477, 8257, 2416, 2), ("fp8", MATH_FP8, 20, 2049, 7169, 4112, 0)]


@pytest.mark.parametrize("fmt,math,plan,M,N,K,epilogue", WIDE)
def test_wide_block(hip, fmt, math, plan, M, N, K, epilogue):
    assert hip.lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, 0, 0) == plan
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    w = random_weight(FORMATS[fmt], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    y = torch.randn(M, N, generator=g, device="cuda").to([torch.float32, torch.bfloat16, torch.bfloat16][epilogue])
    bias = torch.randn(N, generator=g, device="cuda")
    kw = [{}, {"alpha": 0.5}, {"bias": bias, "alpha": 1.5, "beta": 0.25}][epilogue]
    assert torch.equal(ops.gemm_w(hip, x, w, math, y=y.clone(), **kw), chunks_of_32(hip, x, w, math, y, **kw))


# Few blocks (a slice a workgroup), one block past a multiple of 64 / 128 rows and columns, an odd N, many blocks of each shape;
# K of one slice, of slices whose last is short, of a last step and a last K tile cut short.
@pytest.mark.parametrize("fmt,math", MATHS)
@pytest.mark.parametrize("M,N,K", [(65, 300, 4096), (129, 257, 1056), (128, 1000, 544), (191, 2064, 8224), (515, 4096, 1056), (1030, 3001, 2080),
                                   (2050, 4112, 1024), (66, 30000, 544)])
def test_rows_are_those_of_calls_of_32(hip, fmt, math, M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    w = random_weight(FORMATS[fmt], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    y = torch.full((M, N), float("nan"), device="cuda")
    assert torch.equal(ops.gemm_w(hip, x, w, math, y=y.clone()), chunks_of_32(hip, x, w, math, y))


@pytest.mark.parametrize("fmt,math", [("fp8", MATH_BF16), ("nvfp4", MATH_FP4), ("int8", MATH_INT8)])
@pytest.mark.parametrize("y_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bias,alpha,beta", [(None, 0.5, 0.0), (torch.float32, 1.0, 0.0), (torch.bfloat16, 1.5, 0.25)])
@pytest.mark.parametrize("M,N,K", [(70, 132, 4096), (300, 1001, 1056)])
def test_epilogue_operands(hip, fmt, math, y_dtype, bias, alpha, beta, M, N, K):
    g = torch.Generator().manual_seed(N)
    w = random_weight(FORMATS[fmt], N, K, N).to("cuda")
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    y = torch.randn(M, N, generator=g).to(y_dtype).cuda()
    kw = dict(bias=None if bias is None else torch.randn(N, generator=g).to(bias).cuda(), alpha=alpha, beta=beta)
    assert torch.equal(ops.gemm_w(hip, x, w, math, y=y.clone(), **kw), chunks_of_32(hip, x, w, math, y, **kw))


@pytest.mark.parametrize("fmt", checks.FMT_NAMES)
def test_strides_and_a_stream_without_the_partial_buffer(hip, fmt):
    M, N, K, pad = 130, 264, 4096, 8
    w = random_weight(FORMATS[fmt], N, K, 5).to("cuda")
    x = torch.randn(M, K + pad, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16).cuda()
    want = ops.gemm_w(hip, x[:, :K].contiguous(), w, MATH_BF16)
    struct, stream = w.lx(), torch.cuda.Stream()
    for y_dtype, ld_y in ((torch.float32, N + 1), (torch.bfloat16, N + 4)):
        y = torch.full((M, ld_y), -3.0, dtype=y_dtype, device="cuda")
        torch.cuda.synchronize()
        assert hip.status("gemm_w", x, BF16, K + pad, ctypes.pointer(struct), MATH_BF16, None, F32, y, DTYPE[y_dtype], ld_y, M, N, K, 1.0, 0.0,
                          None, stream.cuda_stream) == 0
        torch.cuda.synchronize()
        assert torch.equal(y[:, :N], want.to(y_dtype)) and bool((y[:, N:] == -3.0).all())


# Experts: tiles of every height up to two of 128 (the experts' shares differ by about e^2), slices that end on odd load
# steps (and, in bf16, inside a K tile), a last block of columns cut short, ids outside the range.
@pytest.mark.parametrize("fmt,math", MATHS)
@pytest.mark.parametrize("T,L,I,E,top_k", [(1000, 1056, 544, 16, 1), (800, 1088, 288, 32, 2), (300, 2112, 544, 16, 4), (700, 512, 160, 40, 3)])
def test_experts_are_those_of_few_tokens(hip, fmt, math, T, L, I, E, top_k):
    gu, dn = random_stack(FORMATS[fmt], E, 2 * I, L, 3).to("cuda"), random_stack(FORMATS[fmt], E, L, I, 4).to("cuda")
    latent, _, weights = (t.cuda() for t in checks.make_routing(T, E, L, top_k, T))
    g = torch.Generator().manual_seed(T)
    ids = (torch.linspace(-1, 1, E) - torch.rand(T, E, generator=g).log().neg().log()).topk(top_k, 1).indices.int().cuda()
    ids = torch.where(torch.rand(ids.shape, generator=g).cuda() < 0.03, torch.full_like(ids, E), ids)
    assert hip.lib.dromos_plan_experts(FORMATS[fmt], T, L, I, E, top_k, 0) == 1
    got = ops.experts_grouped(hip, latent, ids, weights, gu, dn, I, E, top_k, math=math)
    step = max(1, 12 * E // top_k)  # fewer rows an expert than the block kernels are taken for
    assert hip.lib.dromos_plan_experts(FORMATS[fmt], step, L, I, E, top_k, 0) == 0
    few = [ops.experts_grouped(hip, latent[t : t + step].contiguous(), ids[t : t + step].contiguous(), weights[t : t + step].contiguous(), gu, dn,
                               I, E, top_k, math=math) for t in range(0, T, step)]
    assert torch.equal(got, torch.cat(few))


# 33 .. 64 rows on short matrices: both ends of the rule's rows, tiles and row lengths in every format, and a last tile and K
# tile cut short, on a stream with a partial-tile buffer; eagerly and from a graph.
FEW = {"bf16": [(33, 2048, 3072), (48, 3072, 4096), (57, 6400, 5120), (64, 4096, 6144)], "int8": [(33, 2048, 2048), (48, 3072, 4096), (49, 2040, 2080), (57, 6400, 5120)],
       "fp8": [(33, 2048, 2048), (48, 3072, 6144), (49, 2040, 2080), (57, 6400, 5120)], "nvfp4": [(49, 2040, 3104), (57, 3072, 4096), (64, 4096, 6144)]}


@pytest.mark.parametrize("fmt,M,N,K", [(f, *c) for f in checks.FMT_NAMES for c in FEW[f]])
def test_few_rows_on_short_matrices(hip, fmt, M, N, K):
    assert hip.lib.dromos_plan_gemm(FORMATS[fmt], MATH_BF16, M, N, K, 0, 1) >= 0
    g = torch.Generator().manual_seed(M)
    w = random_weight(FORMATS[fmt], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    want = chunks_of_32(hip, x, w, MATH_BF16, torch.full((M, N), float("nan"), device="cuda"))
    struct, stream, graph = w.lx(), ctypes.c_void_p(), ctypes.c_void_p()
    y = torch.full((M, N), float("nan"), device="cuda")
    torch.cuda.synchronize()
    assert hip.lib.lx_rt_stream_create(ctypes.byref(stream)) == 0
    call = ("gemm_w", x, BF16, K, ctypes.pointer(struct), MATH_BF16, None, F32, y, F32, N, M, N, K, 1.0, 0.0, None, stream.value)
    try:
        assert hip.status(*call) == 0 and hip.lib.lx_rt_stream_sync(stream) == 0
        assert torch.equal(y, want)
        assert hip.lib.lx_rt_capture_begin(stream) == 0 and hip.status(*call) == 0
        assert hip.lib.lx_rt_capture_end(stream, ctypes.byref(graph)) == 0
        for _ in range(3):
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            assert hip.lib.lx_rt_graph_launch(graph, stream) == 0 and hip.lib.lx_rt_stream_sync(stream) == 0
            assert torch.equal(y, want)
        assert hip.lib.lx_rt_graph_destroy(graph) == 0
    finally:
        assert hip.lib.lx_rt_stream_destroy(stream) == 0


# An infinity among a row's last values: the tiles past the row's end (K is no multiple of 128 here) must not meet it again.
# All slices in a workgroup, one, and one slice a workgroup; everything but the two rows keeps its bits.
@pytest.mark.parametrize("M,N,K", [(65, 300, 1056), (130, 257, 1088), (515, 2064, 8256), (80, 1000, 4104)])
@pytest.mark.parametrize("buffer", [False, True])
def test_infinite_weights_at_the_rows_end(hip, buffer, M, N, K):
    w = random_weight(FORMATS["bf16"], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(K)).to(torch.bfloat16).cuda()
    clean = on_a_stream(hip, buffer, x, w, MATH_BF16, torch.empty(M, N, device="cuda"))
    w.data[3, K - 1], w.data[N - 1, K - 8] = float("inf"), float("-inf")
    got = on_a_stream(hip, buffer, x, w, MATH_BF16, torch.empty(M, N, device="cuda"))
    assert torch.equal(got[:, 3], x[:, K - 1].float() * float("inf")) and torch.equal(got[:, N - 1], x[:, K - 8].float() * -float("inf"))
    got[:, [3, N - 1]] = clean[:, [3, N - 1]]
    assert torch.equal(got, clean)


def test_infinite_expert_weights_at_the_rows_end(hip):
    T, L, I, E, top_k = 1000, 1056, 544, 16, 1
    gu, dn = random_stack(FORMATS["bf16"], E, 2 * I, L, 3).to("cuda"), random_stack(FORMATS["bf16"], E, L, I, 4).to("cuda")
    latent, ids, weights = (t.cuda() for t in checks.make_routing(T, E, L, top_k, T))
    assert hip.lib.dromos_plan_experts(FORMATS["bf16"], T, L, I, E, top_k, 0) == 1
    clean = ops.experts_grouped(hip, latent, ids, weights, gu, dn, I, E, top_k)
    assert bool(clean.isfinite().all())
    to5, to7 = (ids == 5).any(1), (ids == 7).any(1)
    dn.data[5, 9, I - 1], gu.data[7, I + 11, L - 8] = float("inf"), float("-inf")  # one output row; one up row, so one intermediate value
    got = ops.experts_grouped(hip, latent, ids, weights, gu, dn, I, E, top_k)
    assert bool(got[to5, 9].isinf().all()) and bool(got[to7].isinf().all())
    got[to5, 9], got[to7] = clean[to5, 9], clean[to7]
    assert torch.equal(got, clean)


# Asked for through the variant table: row counts that the rule never sends there, in every format and math, with the
# partial-tile buffer and without.
@pytest.mark.parametrize("fmt,math", MATHS)
@pytest.mark.parametrize("M,N,K", [(1, 300, 1056), (17, 1000, 4096), (64, 257, 2080)])
@pytest.mark.parametrize("buffer", [False, True])
def test_asked_for_by_the_table(hip, buffer, fmt, math, M, N, K):
    g = torch.Generator().manual_seed(M)
    w = random_weight(FORMATS[fmt], N, K, N + K).to("cuda")
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    y = torch.full((M, N), float("nan"), device="cuda")
    assert hip.lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, 0, buffer) == -1
    want = on_a_stream(hip, buffer, x, w, math, y.clone())
    try:
        assert hip.lib.lx_tune_force(f"gemm_w_{fmt}".encode(), M, N, K, 8) == 0
        assert hip.lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, 0, buffer) >= 0
        assert torch.equal(on_a_stream(hip, buffer, x, w, math, y.clone()), want)
    finally:
        hip.lib.lx_tune_clear()
