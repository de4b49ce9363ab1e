"""Which kernel takes a product of a middle number of rows (csrc/hn_mid.hip), and how it
splits K: host code, asked without a GPU (the plan is then that of 256 CUs)."""
import ctypes

import pytest

from hydranet_amd import _lib


def _part_bytes(mats, m, n, k):
    f = _lib.lib().hn_mid_part_bytes
    f.restype, f.argtypes = ctypes.c_long, [ctypes.c_int] + [ctypes.c_long] * 3
    return f(mats, m, n, k)


@pytest.mark.parametrize("mats,m,n,k", [(1, 1500, 4096, 4096), (1, 1024, 6144, 4096),
                                        (1, 512, 14336, 4096), (1, 2048, 4096, 1408),
                                        (2, 700, 4096, 4096), (2, 200, 14336, 4096),
                                        (2, 160, 14336, 5120)])
def test_no_split_where_the_tiles_fill_the_chip(mats, m, n, k):
    """At no group size are K splits' partials written where there is a tile for half of
    the CUs or more."""
    assert -(-m // 64) * -(-n * mats // 256) > 128
    assert _part_bytes(mats, m, n, k) == 0
