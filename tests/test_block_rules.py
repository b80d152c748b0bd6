"""The rules that send calls to the block kernels, asked of the library without a device (256 compute units): the calls that
were measured faster there go, those that were measured slower do not."""

import ctypes
import math
import random

import pytest

from dromos_amd.abi import FORMATS, hip_library_path

UNITS = 256  # an MI355X


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(str(hip_library_path()))


# Pairs per expert, experts and sizes on both sides of the rule: few experts or short stages leave most of the device without a block.
@pytest.mark.parametrize("fmt,L,I,E,top_k,T,taken", [
    ("nvfp4", 4096, 1536, 2, 1, 32, 0), ("bf16", 1024, 512, 2, 1, 256, 0), ("fp8", 2048, 1024, 2, 1, 256, 0),
    ("int8", 2048, 1024, 8, 2, 64, 0), ("nvfp4", 1024, 2048, 4, 2, 64, 0), ("bf16", 512, 2048, 12, 2, 540, 0),
    ("fp8", 4096, 1536, 4, 2, 128, 0), ("nvfp4", 2048, 1024, 16, 4, 96, 0), ("nvfp4", 2048, 4096, 12, 2, 150, 0),
    ("bf16", 1024, 2048, 16, 2, 192, 0), ("int8", 4096, 1536, 4, 2, 128, 1), ("nvfp4", 4096, 1536, 128, 8, 255, 0), ("bf16", 4096, 1536, 128, 8, 256, 0),
    ("nvfp4", 4096, 1536, 128, 8, 256, 1), ("nvfp4", 4096, 1536, 128, 8, 2048, 1), ("bf16", 4096, 1536, 128, 8, 384, 1),
    ("fp8", 2048, 1024, 64, 8, 128, 1), ("int8", 4096, 1536, 8, 2, 128, 1), ("bf16", 2048, 1024, 16, 4, 256, 1),
    ("nvfp4", 4096, 14336, 12, 2, 1536, 1), ("fp8", 4096, 1536, 1, 1, 2048, 1)])
def test_experts(lib, fmt, L, I, E, top_k, T, taken):
    assert lib.dromos_plan_experts(FORMATS[fmt], T, L, I, E, top_k, UNITS) == taken


# lx_gemm_w: 4 * mode + shape, or -1 for the kernels for up to 64 rows.
@pytest.mark.parametrize("fmt,math,M,N,K,buffer,taken", [
    ("fp8", 0, 32, 4096, 4096, 1, False), ("fp8", 0, 64, 4096, 4096, 1, True), ("fp8", 0, 64, 4096, 4096, 0, False), ("fp8", 0, 48, 4096, 4096, 1, False),
    ("fp8", 0, 48, 3072, 3072, 1, True), ("fp8", 0, 64, 14336, 4096, 1, False), ("fp8", 0, 64, 4096, 14336, 1, False), ("fp8", 0, 64, 1024, 4096, 1, False),
    ("fp8", 0, 64, 6400, 2048, 1, False), ("int8", 0, 49, 5120, 2048, 1, False), ("fp8", 0, 64, 6400, 2560, 1, False), ("fp8", 0, 40, 3072, 2048, 1, False),
    ("fp8", 0, 64, 4608, 2560, 1, True), ("int8", 0, 64, 4096, 2048, 1, True), ("fp8", 0, 33, 2048, 2048, 1, True), ("fp8", 0, 48, 2560, 2048, 1, True), ("fp8", 0, 64, 6400, 3072, 1, True),
    ("nvfp4", 0, 65, 1500, 8192, 0, False), ("nvfp4", 0, 96, 4096, 14336, 0, False), ("nvfp4", 3, 80, 6144, 4096, 1, False), ("nvfp4", 2, 96, 256, 4096, 0, False),
    ("nvfp4", 0, 65, 1500, 8192, 1, True), ("nvfp4", 0, 97, 1500, 8192, 0, True), ("nvfp4", 0, 96, 4096, 4096, 0, True), ("nvfp4", 0, 65, 9216, 11008, 0, True),
    ("nvfp4", 0, 72, 2048, 2048, 0, True), ("fp8", 0, 65, 1500, 8192, 0, True), ("bf16", 0, 33, 5120, 5120, 1, True), ("bf16", 0, 64, 4096, 2048, 1, False), ("nvfp4", 0, 48, 4096, 4096, 1, False), ("nvfp4", 0, 49, 4096, 4096, 1, True),
    ("nvfp4", 0, 64, 5120, 5120, 1, False), ("int8", 1, 64, 4096, 4096, 1, False), ("int8", 1, 65, 4096, 4096, 0, True), ("fp8", 2, 65, 300, 512, 1, True),
    ("bf16", 0, 65, 300, 40, 0, True), ("nvfp4", 3, 4096, 14336, 4096, 1, True)])
def test_gemm(lib, fmt, math, M, N, K, buffer, taken):
    assert (lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, UNITS, buffer) >= 0) == taken


# The wide block (shape 16, whole rows or added slices) where it was measured ahead, and not where its blocks are few or a unit's only ones.
@pytest.mark.parametrize("fmt,math,M,N,K,wide", [
    ("fp8", 0, 4096, 14336, 4096, True), ("nvfp4", 0, 4096, 14336, 4096, True), ("int8", 1, 4096, 14336, 4096, True), ("fp8", 2, 4096, 14336, 4096, True),
    ("fp8", 2, 2471, 12608, 3840, True), ("fp8", 2, 1563, 13731, 4176, True), ("fp8", 2, 3708, 3601, 3712, False), ("fp8", 2, 1635, 3352, 4672, False),
    ("fp8", 2, 1024, 4096, 14336, False), ("int8", 1, 515, 4096, 11008, False), ("fp8", 0, 338, 3206, 11968, False)])
def test_wide_block(lib, fmt, math, M, N, K, wide):
    assert (lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, UNITS, 1) in (16, 20)) == wide


def test_sums_of_slices_that_do_not_fit_the_buffer_stay_in_the_workgroup(lib):
    part = lambda M: lib.dromos_plan_gemm(FORMATS["fp8"], 0, M, 1024, 14336, UNITS, 1) // 4 == 2
    assert part(128) and not lib.dromos_plan_gemm(FORMATS["fp8"], 0, 128, 1024, 14336, UNITS, 0) // 4 == 2
    assert not part(8192)


# The INT8 math's own cuts of K: not into small blocks that a unit would take two of, where one large one was as good, nor for little; one small block a
# unit is ahead.
@pytest.mark.parametrize("M,N,K,plan", [(154, 6263, 7584, {10, 11}), (191, 4148, 12320, {10, 11}), (183, 4240, 13376, {10, 11}), (172, 5984, 6048, {10, 11}), (112, 11455, 8192, {11}), (211, 8030, 13344, {11}), (639, 618, 5632, {9}), (142, 3376, 8448, {9}),
                                          (100, 2826, 13824, {10})])
def test_int8_math_slices_take_no_more_turns(lib, M, N, K, plan):
    assert lib.dromos_plan_gemm(FORMATS["int8"], 1, M, N, K, UNITS, 1) in plan


# Slices' sums stay inside the 64 MiB of the buffer that a stream has, whatever the sizes: 1 KB for 16 rows by 16 columns of each slice, of
# which there are sixteen at most.
@pytest.mark.parametrize("fmt,math_id", [("bf16", 0), ("int8", 0), ("int8", 1), ("fp8", 0), ("fp8", 2), ("nvfp4", 0)])
def test_the_sums_of_slices_fit_the_buffer(lib, fmt, math_id):
    rng = random.Random(fmt)
    cut, most = 0, 0
    for _ in range(20000):
        M, N, K = (int(2 ** rng.uniform(math.log2(low), math.log2(high))) for low, high in ((1, 70000), (1, 70000), (64, 70000)))
        slices = lib.dromos_plan_slices(FORMATS[fmt], math_id, M, N, K // 32 * 32, UNITS, 1)
        assert (slices > 0) == (lib.dromos_plan_gemm(FORMATS[fmt], math_id, M, N, K // 32 * 32, UNITS, 1) // 4 == 2)
        used = slices * -(-N // 16) * -(-M // 16) * 1024
        assert slices <= 16 and used <= 64 << 20, (M, N, K)
        assert lib.dromos_plan_slices(FORMATS[fmt], math_id, M, N, K // 32 * 32, UNITS, 0) == 0
        cut, most = cut + (slices > 1), max(most, used)
    assert cut > 1000 and most > 60 << 20


# Sizes that are no product have no plan (the slices that fit the buffer are a quotient by the rows and columns).
@pytest.mark.parametrize("M,N,K", [(128, 0, 4096), (0, 4096, 4096), (128, 4096, 0), (-5, 4096, 4096), (128, -16, 4096), (128, 4096, -64), (32, 0, 4096), (32, 4096, 0)])
def test_nothing_to_compute(lib, M, N, K):
    for fmt, math in (("bf16", 0), ("int8", 0), ("int8", 1), ("fp8", 0), ("fp8", 2), ("nvfp4", 0)):
        assert lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, UNITS, 1) == -1
        assert lib.dromos_plan_ring(FORMATS[fmt], M, N, K, UNITS, 1, None) == 0 and lib.dromos_plan_fed(FORMATS[fmt], M, N, K, UNITS, 1) == 0


@pytest.mark.parametrize("fmt,math", [("bf16", 0), ("int8", 1), ("fp8", 0), ("fp8", 2), ("nvfp4", 0)])
def test_the_variant_table_has_the_last_word(lib, fmt, math):
    # An entry is for a row count (the next power of two) of a matrix: "block" asks for the block kernel at any count, every other
    # family keeps the call from it, and an entry for up to 64 rows leaves calls of more rows alone.
    key, N, K = f"gemm_w_{fmt}".encode(), 4096, 4096
    plan = lambda M: lib.dromos_plan_gemm(FORMATS[fmt], math, M, N, K, UNITS, 1) >= 0
    variants = lib.lx_tune_variants(key)
    lib.lx_tune_variant_name.restype = ctypes.c_char_p
    names = [lib.lx_tune_variant_name(key, v).decode() for v in range(variants)]
    try:
        assert plan(130) and not plan(20)
        for M in (20, 64, 130):
            for v, name in enumerate(names):
                lib.lx_tune_clear()
                assert lib.lx_tune_set(key, M, N, K, v) == 0
                assert plan(M) == (name == "block"), (M, name)
                assert M > 64 or plan(130), "an entry for fewer rows holds here"
    finally:
        lib.lx_tune_clear()
    assert names[-1] == "block" and plan(130)
