"""The rules that send calls to the block kernels, asked of the library without a device (256 compute units): the calls that
were measured faster there go, those that were measured slower do not."""

import ctypes

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
    ("fp8", 4096, 1536, 4, 2, 128, 0), ("nvfp4", 4096, 1536, 128, 8, 255, 0), ("bf16", 4096, 1536, 128, 8, 256, 0),
    ("nvfp4", 4096, 1536, 128, 8, 256, 1), ("nvfp4", 4096, 1536, 128, 8, 2048, 1), ("bf16", 4096, 1536, 128, 8, 384, 1),
    ("fp8", 2048, 1024, 64, 8, 128, 1), ("int8", 4096, 1536, 8, 2, 128, 1), ("bf16", 2048, 1024, 16, 4, 256, 1),
    ("nvfp4", 4096, 14336, 12, 2, 1536, 1), ("fp8", 4096, 1536, 1, 1, 2048, 1)])
def test_experts(lib, fmt, L, I, E, top_k, T, taken):
    assert lib.dromos_plan_experts(FORMATS[fmt], T, L, I, E, top_k, UNITS) == taken
