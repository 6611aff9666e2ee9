"""Which tile and how many K slices the GEMM takes (gemm.hip): a rule on sizes, types and the diagnostic switches, no launch."""
import ctypes
import os

import pytest

from voice_enabled_browser_automation_amd.ops import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.KERNEL_SO), reason="the kernel library is not built")


@pytest.fixture
def E():
    import torch  # noqa: F401  (the HIP runtime comes with it)

    from voice_enabled_browser_automation_amd.ops import _vwa_kernels as E

    yield E
    E.gemm_set_p8(2)
    E.gemm_set_split_fill(0)


SIZES = [(1011, 6144, 4096), (4096, 4096, 2048), (2048, 4096, 2048), (1011, 4096, 14336), (3000, 28672, 4096), (300, 512, 512)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_the_switch_for_the_large_tile_reaches_kept_order_products(E, M, N, K):
    """0: never, 1: from 256 rows; the slices, and with them the order of the sums, are those of the estimate's choice."""
    for kw in (dict(keep_order=True), dict(f8=1)):
        splits = E.gemm_plan(0, M, N, K, **kw)[1]
        E.gemm_set_p8(0)
        assert E.gemm_plan(0, M, N, K, **kw) == (False, splits)
        E.gemm_set_p8(1)
        assert E.gemm_plan(0, M, N, K, **kw) == (True, splits)
        E.gemm_set_p8(2)


def test_the_estimate_takes_either_tile_for_kept_order(E):
    """(what the tests of the kept order's bits rely on: the same slices, another tile)"""
    assert E.gemm_plan(0, 4096, 4096, 2048, keep_order=True) == (True, 1)
    assert E.gemm_plan(0, 2048, 4096, 2048, keep_order=True) == (False, 1)


def test_a_split_fill_keeps_the_large_tile(E):
    """The split-K fill target replaces the estimate by the rules on shape alone: large tiles that cover the CUs, or do so in
    slices of 2048 and more, stay large."""
    E.gemm_set_split_fill(75)
    assert E.gemm_plan(0, 1011, 28672, 4096) == (True, 1)      # 448 large tiles
    assert E.gemm_plan(1, 1011, 4096, 14336) == (True, 4)      # 64, in slices of 3584
    assert E.gemm_plan(1, 1011, 4096, 4096)[0] is False        # slices of 1024
    assert E.gemm_plan(0, 1011, 28672, 4096, w_tiled=False)[0] is False
    E.gemm_set_p8(0)
    assert E.gemm_plan(0, 1011, 28672, 4096)[0] is False
    E.gemm_set_p8(1)
    assert E.gemm_plan(0, 300, 512, 512)[0] is True and E.gemm_plan(0, 300, 528, 512)[0] is False


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 200])
def test_slices_of_fp8_weights_fit_the_k_groups_and_the_workspace(E, M):
    """W8A16: the slices come from an estimate; whatever the sizes they leave none empty and fit the workspace."""
    for N, K in ((16, 128), (4096, 4096), (28672, 4096), (4096, 14336), (2064, 1408), (32768, 1024)):
        for ws in (0, M * N, 3 * M * N, 1 << 25):
            large, s = E.gemm_plan(1, M, N, K, f8=2, ws_floats=ws)
            kg = K // 128
            assert not large and 1 <= s <= kg and -(-kg // -(-kg // s)) == s
            assert s == 1 or s * M * N <= ws
    if M in (17, 32):  # (one slice covers the chip; four and eight are the measured best)
        assert [E.gemm_plan(1, M, N, K, f8=2)[1] for N, K in ((28672, 4096), (6144, 4096), (4096, 14336))] == [1, 4, 8]


@pytest.mark.parametrize("kw", [dict(), dict(parts=True)])
def test_slices_of_few_rows_are_those_of_the_weight(E, kw):
    """<= 64 rows of bf16 weights: the rows of a call do not decide how its sums are cut."""
    seen = set()
    for N in (272, 1024, 2048, 4096, 6144, 9472, 12288, 28672):
        for K in (128, 1024, 1408, 4096, 6144, 14336):
            s = {E.gemm_plan(0, M, N, K, **kw)[1] for M in range(1, 65)}
            assert len(s) == 1, (N, K, s)
            seen |= s
    assert {1, 4, 8, 16} <= seen


def test_columns_of_two_launches_are_whole_rounds(E):
    """The first launch's columns: large tiles that fill the CUs a whole number of times, never all of them; products that keep an
    order, few rows and switched-off tiles have one launch."""
    seen = 0
    for M in (128, 600, 1011, 1900, 2048, 4096, 12000):
        for N in (4096, 8208, 9472, 17664, 22528, 28672, 32896):
            for K in (128, 1024, 4096):
                cut = E.gemm_cut(0, M, N, K)
                assert 0 <= cut < N and cut % 256 == 0
                if cut:
                    seen += 1
                    rows = -(-M // 256)
                    rounds, tiles = rows * -(-N // 256) // 256, rows * cut // 256
                    assert tiles <= 256 * rounds < tiles + rows  # (all of the whole rounds: no column tile more fits them)
                assert E.gemm_cut(0, M, N, K, keep_order=True) == 0 and E.gemm_cut(5, M, N, K) == 0
    assert seen > 5 and E.gemm_cut(0, 64, 32896, 4096) == 0 and E.gemm_cut(6, 2048, 32896, 4096) == 32768
    E.gemm_set_p8(0)
    assert E.gemm_cut(0, 2048, 32896, 4096) == 0


def test_a_product_past_the_offsets_has_one_launch(E):
    """A weight that 32-bit offsets do not reach is refused as a whole, wherever its columns would have been cut: the columns of the
    whole rounds alone (32768 x 32640, bf16) are within reach."""
    reach = 0x7FFFFFF0
    assert 32768 * 32640 * 2 < 32896 * 32640 * 2 < reach <= 32912 * 32640 * 2
    assert E.gemm_cut(0, 2048, 32896, 32640) == 32768
    assert E.gemm_cut(0, 2048, 32912, 32640) == 0


def test_two_wave_groups_have_stages_to_share(E):
    """Two groups of waves from 8 k-groups of a slice on, from 11 where one row block takes the weight alone, with every tile and slice
    on a CU of its own; other tiles, kept orders, row-major and fp8 weights have one group."""
    seen = set()
    for M in (65, 127, 128, 129, 300, 513, 1011, 2048, 4096):
        for N in (400, 1024, 2560, 6144, 12288, 28672):
            for K in (128, 640, 1024, 1280, 1408, 4096, 14336):
                for epi in (0, 1, 3, 5):
                    columns, slices, groups = E.gemm_choice(epi, M, N, K)
                    assert groups == 1 or columns in (128, 192)
                    assert columns != 192 or (groups == 2 and epi != 1)
                    if groups == 2:
                        seen.add((columns, slices > 1))
                        assert M >= 128 and -(-K // 128 // slices) >= (11 if M <= 128 else 8)
                        assert -(-M // 128) * -(-N // columns) * slices <= 256
                for kw in (dict(keep_order=True), dict(w_tiled=False), dict(f8=1), dict(f8=2)):
                    assert E.gemm_choice(0, M, N, K, **kw)[2] == 1
    assert seen == {(c, s) for c in (128, 192) for s in (False, True)}
    assert E.gemm_choice(0, 2048, 2048, 640)[2] == 1 and E.gemm_choice(0, 2048, 2048, 1024)[2] == 2
    assert E.gemm_choice(0, 128, 28672, 1280)[2] == 1 and E.gemm_choice(0, 129, 12288, 1280)[2] == 2


def test_a_residual_in_32_bits_keeps_its_slices(E):
    """Such a product has as many slices as on one-group tiles (which switching the groups' weights off shows), and two groups where
    these take them; other 32-bit results are planned as 16-bit ones."""
    grouped = 0
    for M in (128, 600, 1011, 2048, 4096):
        for N in (1024, 1280, 2048, 4096, 6144):
            for K in (1024, 1536, 2048, 3840, 6144):
                got, one = E.gemm_choice(1, M, N, K, y_f32=2), E.gemm_choice(1, M, N, K, w_tiled=False)
                assert E.gemm_choice(0, M, N, K, y_f32=1) == E.gemm_choice(0, M, N, K)
                whole = E.gemm_choice(1, M, N, K)
                assert got[1] > 1 or one[1] == 1, (M, N, K, got, one)
                grouped += got[2] == 2 and got != whole
    assert grouped and E.gemm_choice(1, 2048, 1024, 2048)[1] == 1 and E.gemm_choice(1, 2048, 1024, 2048, y_f32=2)[1] == 2


@pytest.mark.parametrize("epi,N,cap", [(0, 8, 256), (1, 15, 256), (2, 16, 256), (2, 31, 256), (0, 64, 0)])
def test_streaming_of_less_than_a_tile_is_an_error(E, epi, N, cap):
    """A weight of fewer rows than a tile, or a grid of none, is refused with a code ahead of the launch, which divides by the grid."""

    class Params(ctypes.Structure):  # (the first fields of SkinnyParams; the others are zero)
        _fields_ = [("X", ctypes.c_void_p), ("ldx", ctypes.c_int), ("W", ctypes.c_void_p), ("M", ctypes.c_int), ("N", ctypes.c_int),
                    ("K", ctypes.c_int), ("rest", ctypes.c_char * 448)]

    lib, p = ctypes.CDLL(build.KERNEL_SO), Params(X=1 << 20, ldx=1024, W=1 << 20, M=1, N=N, K=1024)
    assert [lib.vwa_skinny_stream(epi, ctypes.byref(p), cap, ks, None) for ks in (4, 8)] == [-2, -2]
