"""What the entries of the matrix products refuse before anything is launched, and the answers about sizes that are kept."""

import ctypes

import pytest

from mini_gpt_inference_amd.ops import kernels, library

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


def test_plans_that_another_thread_clears(monkeypatch):
    """The table of plans is bounded: a thread that fills it empties it first, perhaps while another is about to answer from it."""
    class Emptied(dict):
        def __setitem__(self, key, value):
            super().__setitem__(key, value)
            self.clear()

    sizes = [(16, 4800, 1600), (40, 4800, 1600), (8, 1600, 6400)]
    want = [kernels.linear_rows_plan(*s) for s in sizes]
    assert want[0] is not None and want[1] is None
    monkeypatch.setattr(kernels, "_ROWS_PLANS", Emptied())
    assert [kernels.linear_rows_plan(*s) for s in sizes] == want
