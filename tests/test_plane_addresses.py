"""Plane addresses as callers hold them: any integer type, and no missing one."""
import numpy as np
import pytest

from glmmhdturb_amd._lib import plane_array


@pytest.mark.parametrize("kind", [int, np.int64, np.uint64])
def test_plane_array_takes_any_integer(kind):
    want = [0x7f0000000000 + 4096 * v for v in range(9)]
    arr, keep = plane_array([kind(p) for p in want])
    assert [arr[v] for v in range(9)] == want


def test_plane_array_refuses_a_missing_address():
    with pytest.raises(TypeError):
        plane_array([4096, None])
