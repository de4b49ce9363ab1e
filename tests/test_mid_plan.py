"""Which kernel takes a product of a middle number of rows (csrc/hn_mid.hip), and how it
splits K: host code, asked without a GPU (the plan is then that of 256 CUs)."""
import ctypes

import pytest

from hydranet_amd import _lib


def _part_bytes(mats, m, n, k):
    f = _lib.lib().hn_mid_part_bytes
    f.restype, f.argtypes = ctypes.c_long, [ctypes.c_int] + [ctypes.c_long] * 3
    return f(mats, m, n, k)


def _plan(mats, m, n, k, group):
    """0: not a product for these kernels; -1: K over a workgroup's waves; else K splits."""
    f = _lib.lib().hn_mid_linear_plan
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_int] + [ctypes.c_long] * 4
    r = f(mats, m, n, k, group)
    return r if r <= 0 else r & 0xffff


@pytest.mark.parametrize("mats,m,n,k", [(1, 1500, 4096, 4096), (1, 1024, 6144, 4096),
                                        (1, 512, 14336, 4096), (1, 2048, 4096, 1408),
                                        (2, 700, 4096, 4096), (2, 200, 14336, 4096),
                                        (2, 160, 14336, 5120)])
def test_no_split_where_the_tiles_fill_the_chip(mats, m, n, k):
    """At no group size are K splits' partials written where there is a tile for half of
    the CUs or more."""
    assert -(-m // 64) * -(-n * mats // 256) > 128
    assert _part_bytes(mats, m, n, k) == 0


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("mats,m,n,k,want", [
    # few stages: never split, few rows and many tiles left to the other kernels
    (1, 17, 4096, 512, 0), (1, 32, 4096, 768, 0), (2, 17, 14336, 512, 0), (1, 64, 8192, 256, 0),
    (1, 33, 4096, 512, 1), (2, 64, 4096, 768, 1), (1, 200, 4096, 512, 1), (1, 65, 256, 512, 1),
    (1, 4096, 4096, 512, 0), (2, 512, 14336, 512, 0), (1, 65, 65536, 512, 0),
    (1, 512, 14336, 512, 1),
    # up to 21 rows of a long K in few tiles, and the rows past them
    (1, 17, 1024, 8192, 0), (1, 21, 4096, 14336, 0), (1, 20, 5120, 13824, 0), (1, 17, 4096, 5632, 0),
    (1, 17, 4096, 4096, -1), (1, 21, 14336, 4096, -1),
])
def test_left_to_the_other_kernels(mats, m, n, k, group, want):
    assert _plan(mats, m, n, k, group) == want


@pytest.mark.parametrize("mats,m,n,k,group,want", [
    (1, 22, 4096, 14336, 128, -1), (1, 17, 4096, 8192, 128, -1), (1, 17, 4096, 8192, 64, -1),
    # K beyond the waves' ranges: split over workgroups only where there is work for it
    (1, 24, 4096, 8192, 32, 0), (1, 32, 1024, 14336, 64, 0), (2, 24, 1024, 8192, 32, 0),
    (1, 22, 4096, 14336, 64, 16), (1, 33, 4096, 8192, 32, 8), (1, 17, 8192, 28672, 128, 8),
])
def test_few_rows_split_with_work_enough(mats, m, n, k, group, want):
    assert _plan(mats, m, n, k, group) == want


@pytest.mark.parametrize("mats,m,n,k,group,want", [
    (1, 560, 1024, 14336, 64, 7),    # 16 stages each
    (1, 640, 4096, 11008, 64, 3),    # as many as are resident, though 86 stages go in twos
    (1, 333, 4096, 14336, 64, 4), (2, 160, 4096, 14336, 64, 4),
    (1, 1500, 4096, 14336, 64, 0), (1, 64, 8192, 28672, 64, 8), (1, 64, 4096, 14336, 32, 8),
    (1, 90, 1002, 10240, 64, 0),     # columns not a multiple of 4: no reduction
])
def test_long_k_splits(mats, m, n, k, group, want):
    assert _plan(mats, m, n, k, group) == want


@pytest.mark.parametrize("mats,m,n,k,group,want", [
    # over a workgroup's waves: up to two rounds of 256 tiles of 32 x 64 at any number of rows
    (1, 512, 1024, 4096, 128, -1), (1, 700, 1408, 4096, 128, -1), (1, 2048, 512, 4096, 128, -1),
    (1, 4096, 256, 1024, 32, -1), (1, 850, 1408, 4096, 128, 1), (1, 200, 4096, 1408, 128, -1),
    (1, 400, 4096, 1408, 128, 1),
    # up to three with the activations in L2, at group 128 from 32 stages on
    (1, 333, 4096, 4096, 128, -1), (1, 333, 4096, 4096, 64, -1), (1, 400, 4096, 4096, 128, 1),
    (1, 1500, 1024, 4096, 128, 1), (1, 333, 4096, 2048, 64, -1), (1, 333, 4096, 2048, 128, 1),
    # under two past K = 8192
    (1, 260, 1024, 14336, 128, -1), (1, 200, 4096, 14336, 128, -1), (1, 225, 4096, 14336, 128, 7),
    (1, 480, 2048, 10240, 128, -1),
    (1, 333, 4096, 14336, 128, 4),
    (2, 333, 1408, 4096, 128, -1), (2, 500, 1408, 4096, 128, 1),
])
def test_k_over_waves(mats, m, n, k, group, want):
    assert _plan(mats, m, n, k, group) == want


@pytest.mark.parametrize("e,rows,h,i,split", [
    (8, 1024, 4096, 14336, True), (128, 16000, 4096, 1408, False),
    (32, 2000, 4096, 6144, True), (32, 3000, 4096, 6144, False), (128, 16384, 512, 4608, False),
])
def test_down_slices_fit_the_prefill_workspace(e, rows, h, i, split):
    """Whether a layer's down projection runs in K slices follows from its sizes: where it
    does, the slices fit the workspace that every caller above 64 tokens passes."""
    lib = _lib.lib()
    got = lib.hn_moe_experts_decode_split_check(e, rows, rows, h, i, 128) == 0
    assert got == split
    if got:
        assert (2 << 20) + 16 * rows * h <= lib.hn_gemm_workspace_bytes()


def test_product_splits_fit_the_prefill_workspace():
    ws = _lib.lib().hn_gemm_workspace_bytes()
    for mats in (1, 2):
        for m in (65, 100, 333, 560, 1024, 1500, 2048, 4096, 8192):
            for n in (64, 256, 1000, 4096, 14336, 32000):
                for k in (1024, 1408, 4096, 8192, 14336, 28672):
                    assert (2 << 20) + _part_bytes(mats, m, n, k) <= ws, (mats, m, n, k)
