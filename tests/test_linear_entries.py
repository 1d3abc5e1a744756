"""What the entries of the matrix products refuse before anything is launched, and the answers about sizes that are kept."""

import ctypes

import pytest

from mini_gpt_inference_amd.ops import kernels, library
from mini_gpt_inference_amd.ops.linear import folds_before_rows_apart

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


@pytest.mark.parametrize("n,k,o,stretches", [
    (4, 896, 1792, None), (12, 896, 1792, 1), (3, 768, 2304, None), (4, 768, 2304, 1), (7, 896, 2304, None), (8, 896, 2304, 1), (2, 896, 3072, None),
    (3, 896, 3072, 1), (5, 1600, 1024, None), (6, 1600, 1024, 1), (2, 2048, 2304, None), (3, 2048, 2304, 1), (4, 6144, 768, None), (5, 6144, 768, 4),
    (7, 8192, 1024, None), (8, 8192, 1024, 4), (6, 8192, 6400, None), (7, 8192, 6400, 1), (12, 8192, 8128, None), (13, 8192, 8128, 1),
    (12, 16384, 1536, None), (13, 16384, 1536, 2), (16, 8192, 4800, 1), (17, 8192, 4800, None), (27, 7680, 4800, 1), (28, 7680, 4800, None),
    (28, 10240, 4096, 1), (29, 10240, 4096, None), (32, 2048, 2304, 1), (32, 4096, 2560, 1), (32, 5440, 2304, 4), (32, 4096, 2048, 4),
    (5, 5120, 1024, 1), (6, 5120, 1024, 4), (12, 8192, 1536, 1), (13, 8192, 1536, 2), (6, 6400, 1600, 2)])
def test_lines_of_the_products_of_few_rows(n, k, o, stretches):
    """Where the kernel for up to 32 rows is left to others, and how often it cuts the inner size, on both sides of each line."""
    plan = kernels.linear_rows_plan(n, o, k)
    assert (None if plan is None else plan[1]) == stretches


@pytest.mark.parametrize("n,k,o,folds", [
    (32, 960, 2048, True), (17, 960, 2304, False), (8, 2048, 3072, True), (9, 2048, 3072, False), (10, 1280, 3840, True), (11, 1280, 3840, False),
    (4, 3072, 2048, True), (5, 3072, 2048, False), (32, 1600, 1024, True), (24, 1408, 1280, True), (25, 1408, 1280, False), (16, 1600, 1792, True),
    (16, 1792, 1792, False), (16, 2560, 1024, True), (12, 2560, 1280, False), (5, 1600, 4800, True), (6, 1600, 4800, False), (4, 4096, 5120, True),
    (5, 4096, 5120, False), (32, 5120, 2048, True)])
def test_lines_of_the_layer_norm_in_front(n, k, o, folds):
    """Which products of a plan have their LayerNorm folded into the decode kernel instead."""
    assert kernels.linear_rows_plan(n, o, k) is not None
    assert folds_before_rows_apart(n, o, k) == folds
