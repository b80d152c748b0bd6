"""The rule that sends calls to the ring kernel of lx_gemm_w, and the layout of its ring, asked of the library without a device (256
compute units)."""

import ctypes

import pytest

from dromos_amd.abi import FORMATS, hip_library_path

UNITS = 256  # an MI355X


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(str(hip_library_path()))


# A wavefront's look-ahead is ordered against its own later loads only (with a slice a wavefront there is no barrier in the walk), so it
# may go nowhere but where that wavefront alone loads and reads. Every number of row tiles, two to four slices, both widths.
@pytest.mark.parametrize("M,N,K,plan", [
    (17, 4640, 2048, 8 * 32 + 2), (33, 8448, 2048, 8 * 64 + 2), (64, 6208, 2048, 8 * 32 + 2), (32, 7264, 4096, 8 * 32 + 4),
    (48, 8704, 4096, 8 * 64 + 4), (64, 9088, 4096, 8 * 32 + 4), (40, 12304, 8128, 8 * 64 + 4), (24, 7424, 8192, 8 * 32 + 4),
    (32, 4640, 3072, 8 * 32 + 3)])
def test_look_ahead_stays_in_the_wavefronts_own_part(lib, M, N, K, plan):
    lds = (ctypes.c_int * 13)()
    assert lib.dromos_plan_ring(FORMATS["nvfp4"], M, N, K, UNITS, 1, lds) == plan
    stage, waves = lds[0], [lds[1 + 3 * w : 4 + 3 * w] for w in range(4)]
    for w, (ahead, own, size) in enumerate(waves):
        assert own <= ahead and ahead + 256 <= own + size <= stage, f"wavefront {w}"
        assert w == 0 or waves[w - 1][1] + waves[w - 1][2] <= own, f"wavefront {w}"


# Calls that were measured faster by the ring kernel go there, calls that were measured slower do not: activations off the 128-byte
# lines, slices that K does not fill, whole tiles a unit (512 and 768 tiles).
@pytest.mark.parametrize("fmt,M,N,K,taken", [
    ("fp8", 32, 6144, 4096, True), ("fp8", 35, 5136, 7504, False), ("fp8", 49, 5328, 6448, False), ("fp8", 46, 5584, 7168, False), ("fp8", 27, 5952, 6400, False),
    ("fp8", 40, 8192, 4096, True), ("fp8", 48, 8192, 5120, False), ("int8", 48, 8192, 5120, True), ("fp8", 35, 8192, 5008, False), ("fp8", 64, 8192, 6144, True),
    ("fp8", 29, 7744, 7056, False), ("fp8", 43, 6480, 7136, True), ("fp8", 54, 8784, 5120, True), ("fp8", 42, 14400, 6576, False), ("fp8", 63, 11280, 6976, False),
    ("int8", 46, 14752, 7120, False), ("int8", 40, 9600, 4112, False), ("fp8", 64, 12288, 6144, False), ("int8", 40, 16192, 7168, True), ("int8", 64, 14336, 4096, True), ("fp8", 48, 14336, 4096, False), ("fp8", 37, 15104, 6592, True), ("nvfp4", 40, 14336, 2048, True), ("bf16", 38, 14336, 5120, True), ("int8", 24, 16192, 7168, False),
    ("bf16", 56, 15010, 7064, False), ("bf16", 56, 7984, 4096, True), ("bf16", 48, 8192, 4096, True), ("bf16", 48, 8192, 7680, False), ("bf16", 9, 16384, 8192, False),
    ("bf16", 9, 12512, 4096, True), ("bf16", 48, 12288, 6144, False), ("bf16", 40, 12288, 6144, True), ("bf16", 30, 9472, 2464, False), ("bf16", 29, 10544, 2432, False), ("bf16", 36, 11040, 8064, False), ("int8", 32, 8192, 7168, False),
    ("nvfp4", 32, 7264, 4096, True), ("nvfp4", 64, 12288, 3072, False), ("nvfp4", 32, 14336, 4096, False), ("nvfp4", 30, 14336, 2112, True), ("nvfp4", 64, 14336, 4096, False),
    ("nvfp4", 40, 12368, 4096, True), ("fp8", 47, 7867, 8192, False), ("nvfp4", 24, 8970, 3616, False), ("nvfp4", 16, 7264, 4096, False)])
def test_what_the_ring_takes(lib, fmt, M, N, K, taken):
    assert (lib.dromos_plan_ring(FORMATS[fmt], M, N, K, UNITS, 1, None) > 0) == taken


# The form with loader wavefronts: of the calls above none, of those that ring_cols() leaves what was measured faster.
@pytest.mark.parametrize("M,N,K,slices", [
    (64, 14336, 4096, 4), (50, 8256, 4416, 3), (33, 14336, 8192, 4), (57, 9408, 8704, 3), (40, 24000, 3072, 2), (20, 16400, 4096, 2), (12, 9600, 2112, 3), (64, 20000, 1024, 1),
    (64, 8192, 4096, 0), (64, 9088, 4096, 0), (12, 16500, 2112, 0), (16, 14336, 4096, 0), (32, 14336, 4096, 0), (44, 8656, 13184, 0), (20, 12384, 6144, 0), (8, 14336, 4160, 0),
    (64, 14336, 4112, 0), (40, 8704, 4096, 0)])
def test_what_the_form_with_loaders_takes(lib, M, N, K, slices):
    assert lib.dromos_plan_fed(FORMATS["nvfp4"], M, N, K, UNITS, 1) == slices
    assert slices == 0 or lib.dromos_plan_ring(FORMATS["nvfp4"], M, N, K, UNITS, 1, None) == 0


# Where that form was measured slower: few rows in one slice (more than 1810 tiles, as vocabularies have) or two long ones; and beyond what was
# measured.
@pytest.mark.parametrize("M,N,K,slices", [
    (32, 32000, 4096, 0), (17, 128256, 4096, 0), (24, 151936, 8192, 0), (20, 30001, 14336, 0), (25, 68208, 2048, 0), (31, 49872, 1024, 0), (17, 32000, 3072, 1), (32, 128256, 1536, 1),
    (24, 18656, 1024, 0), (32, 50304, 4160, 1), (48, 32000, 14336, 0), (34, 50848, 8192, 0), (33, 152000, 4096, 1), (49, 32000, 14336, 1), (64, 128256, 4096, 1), (64, 152016, 4096, 0), (30, 18480, 14208, 0),
    (32, 20480, 8192, 2), (23, 16574, 13952, 0), (13, 13614, 3008, 0), (14, 11888, 4032, 0), (9, 9600, 2112, 3)])
def test_what_the_form_with_loaders_leaves(lib, M, N, K, slices):
    assert lib.dromos_plan_fed(FORMATS["nvfp4"], M, N, K, UNITS, 1) == slices


# A feeder of that form passes a stage's barrier with the stage's loads here, and ends its walk with nothing on its way: behind it the ring
# is overwritten, and what it asked for ahead of the walk counts too (one without any stage, where K is one slice, asks for that only).
@pytest.mark.parametrize("weights", [0, 1])
@pytest.mark.parametrize("rows", [32, 48, 64])
def test_a_feeder_leaves_nothing_in_flight(lib, rows, weights):
    for ahead in (0, 1, 2, 7):
        for stages in (0, 1, 2, 3, 4, 5, 9, 10, 11, 40):
            for idle in (0, 1, 8):
                assert lib.dromos_feed_in_flight(rows, weights, stages, max(1, stages + idle), ahead) == 0, (stages, idle, ahead)
