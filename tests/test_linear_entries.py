"""What the entries of the matrix products refuse before anything is launched, and the answers about sizes that are kept."""

import ctypes

import pytest

from mini_gpt_inference_amd.ops import library

NULL_POINTER = -4
XIELU = 4


@pytest.mark.parametrize("shape,n", [(-1, 40), (3, 40), (4, 8), (8, 16), (26, 8), (27, 32)])
def test_xielu_without_its_coefficients_is_refused(shape, n):
    """The entry with the tile's shape given has no place for the two coefficients, which the kernels would read."""
    memory = ctypes.create_string_buffer(64)
    at = (ctypes.addressof(memory) + 15) // 16 * 16         # (never read: the entry looks at the pointers alone)
    k, o = 1600, 1600
    entry = library.kernels().mgpt_linear_mfma_shape
    assert entry(shape, 0, at, k, at, None, at, 1, o, n, o, k, XIELU, None, 0, None) == NULL_POINTER
    assert library.kernels().mgpt_linear_mfma(at, k, at, None, at, 1, o, n, o, k, XIELU, None, 0, None) == NULL_POINTER
