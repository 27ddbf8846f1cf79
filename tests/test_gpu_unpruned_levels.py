"""The searches where their bounds leave (nearly) everything to score, and the
selection over a ring whose elements are all alike (csrc/dmo_kernels.hip,
csrc/vsdmo_numerics.h): positions bit-exact against the oracle."""
import numpy as np
import pytest

from test_gpu_search_bounds import _compare, _cube, _hex_fan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("jitter", [0.0, 1e-7, 1e-4, 0.02])
def test_hex_rings_of_equal_elements(oracle, jitter, metric):
    """every ratio within rounding of the smallest: the selection goes from one
    that replaces the last to the next"""
    xyz, cells = _cube("hex", 8, 81, jitter)
    _compare(oracle, "hex", xyz, cells, hex_metric=metric)
