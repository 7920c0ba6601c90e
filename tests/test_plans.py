"""Which kernel a shape reaches, asked of the library's host-side plan queries (CPU only)."""
import pytest

from mosaic_amd import _lib

SKINNY, T128, T256, BIG, RING, MID = range(6)


def _fp8(m, n, k, workspace=True):
    return divmod(_lib.lib().mosaic_fp8_block_gemm_plan(m, n, k, int(workspace)), 256)


@pytest.mark.parametrize("m,n,k", [(200, 576, 7168), (130, 512, 16384), (255, 768, 7168), (140, 256, 16384),
                                   (143, 272, 13824), (150, 832, 8960), (130, 1152, 1280)])
def test_fp8_narrow_weights_without_workspace_run_skinny(m, n, k):
    """129..255 rows of a narrow weight: tiled with K split where the partials have room, else the skinny
    kernel (256-row tiles would be a handful of workgroups)."""
    kind, splits = _fp8(m, n, k)
    assert kind in (T128, T256) and splits >= 2
    assert _fp8(m, n, k, workspace=False) == (SKINNY, 1)


@pytest.mark.parametrize("m,n,k", [(200, 4112, 4096), (250, 2048, 1024)])
def test_fp8_wider_weights_without_workspace_stay_tiled(m, n, k):
    assert _fp8(m, n, k, workspace=False)[0] in (T128, T256)


@pytest.mark.parametrize("m,n,k", [(255, 1504, 1024), (128, 2224, 1024), (99, 2944, 1024), (189, 1296, 1152),
                                   (247, 1808, 1152)])
def test_fp8_short_k_whole_plans_stay_tiled(m, n, k):
    """8 to 11 K blocks over 16 to 31 tiles: the estimate takes the whole K in one slice, which the
    small-grid rule must not take for a grid too small to tile."""
    for workspace in (True, False):
        kind, splits = _fp8(m, n, k, workspace)
        assert kind in (T128, T256) and splits == 1


@pytest.mark.parametrize("m,n,k,kind", [
    (4733, 4352, 4480, BIG), (2867, 13920, 384, BIG), (973, 17744, 2688, BIG), (2580, 6880, 5376, BIG),
    (4096, 18432, 7168, BIG), (2119, 7440, 3840, T128), (810, 17344, 1152, T128), (786, 20688, 512, T256)])
def test_fp8_big_tiles_keep_near_ties(m, n, k, kind):
    """The 256 x 256 kernel with a tile for every CU gives way only to a plan that is clearly better."""
    assert _fp8(m, n, k) == (kind, 1)


@pytest.mark.parametrize("m,n,k,splits", [
    (6939, 592, 2560, 3), (2265, 832, 3072, 6), (2243, 3520, 3072, 2), (2428, 1200, 2048, 4), (1855, 2288, 4096, 3),
    (5220, 560, 1536, 3), (2763, 1808, 1024, 1), (193, 18432, 7168, 3), (512, 1536, 7168, 5), (768, 4096, 4096, 1)])
def test_a8_splits(m, n, k, splits):
    """K slices of the dense A8 GEMM, above the row count where the partials' rate changes and below."""
    assert _lib.lib().mosaic_mxt16_linear_a8_workspace_bytes(m, n, k) == (4 * m * n * splits if splits > 1 else 0)


@pytest.mark.parametrize("b,h,topk,whole_splits", [
    (32, 128, 640, True), (32, 128, 641, False), (32, 128, 1000, False), (32, 128, 1024, False), (32, 128, 2048, True),
    (31, 128, 1000, True), (24, 128, 1000, True), (32, 64, 1024, True), (16, 256, 1024, True), (16, 128, 1024, True)])
def test_mla_whole_splits_with_fp32_partials(b, h, topk, whole_splits):
    """Up to 1024 picks the whole-split kernel's partials are fp32: 32 rows of 128 heads past 640 picks stay
    on the block kernel, whose partials are all that the workspace then holds."""
    size = _lib.lib().mosaic_mla_decode_workspace_bytes
    splits = size(b, 16, topk) // (b * 16 * 1024)  # the block kernel's (16 heads never take whole splits)
    assert (size(b, h, topk) > b * splits * h * (1024 + 8)) == whole_splits


def test_fp8_planned_slices_are_never_empty():
    """Slices are ceil(K blocks / S) blocks each: every S that a plan names fills all of them (33 blocks in 8
    slices of 5 would leave the eighth starting past K)."""
    for m in (65, 96, 128, 129, 200, 256, 300, 777, 2048):
        for n in (16, 128, 512, 577, 1536, 4096, 7168, 18432):
            for nkb in range(1, 131):
                kind, splits = _fp8(m, n, 128 * nkb)
                if kind in (T128, T256):
                    per = -(-nkb // splits)
                    assert -(-nkb // per) == splits, (m, n, nkb, splits)
