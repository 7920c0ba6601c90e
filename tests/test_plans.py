"""Which kernel a shape reaches, asked of the library's host-side plan queries (CPU only)."""
import pytest

from mosaic_amd import _lib

SKINNY, T128, T256, BIG, RING, MID = range(6)


def _fp8(m, n, k, workspace=True):
    return divmod(_lib.lib().mosaic_fp8_block_gemm_plan(m, n, k, int(workspace)), 256)


@pytest.mark.parametrize("m,n,k", [(200, 576, 7168), (130, 512, 16384), (255, 768, 7168), (140, 256, 16384),
                                   (143, 272, 13824), (150, 832, 8960)])
def test_fp8_narrow_weights_without_workspace_run_skinny(m, n, k):
    """129..255 rows of a narrow weight: tiled with K split where the partials have room, else the skinny
    kernel (256-row tiles would be a handful of workgroups)."""
    kind, splits = _fp8(m, n, k)
    assert kind in (T128, T256) and splits >= 4
    assert _fp8(m, n, k, workspace=False) == (SKINNY, 1)


@pytest.mark.parametrize("m,n,k", [(200, 4112, 4096), (250, 2048, 1024)])
def test_fp8_wider_weights_without_workspace_stay_tiled(m, n, k):
    assert _fp8(m, n, k, workspace=False)[0] in (T128, T256)
