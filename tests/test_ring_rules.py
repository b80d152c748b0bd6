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
    (48, 8704, 4096, 8 * 64 + 4), (64, 9088, 4096, 8 * 32 + 4), (40, 16384, 8192, 8 * 64 + 4), (24, 7424, 8192, 8 * 32 + 4),
    (32, 4640, 3072, 8 * 32 + 3)])
def test_look_ahead_stays_in_the_wavefronts_own_part(lib, M, N, K, plan):
    lds = (ctypes.c_int * 13)()
    assert lib.dromos_plan_ring(FORMATS["nvfp4"], M, N, K, UNITS, 1, lds) == plan
    stage, waves = lds[0], [lds[1 + 3 * w : 4 + 3 * w] for w in range(4)]
    for w, (ahead, own, size) in enumerate(waves):
        assert own <= ahead and ahead + 256 <= own + size <= stage, f"wavefront {w}"
        assert w == 0 or waves[w - 1][1] + waves[w - 1][2] <= own, f"wavefront {w}"
