"""The tiles of 64 columns (gemm_mfma_ws_kernel 64 x 64 and 128 x 64): sizes that are given to them, against float64."""
import pytest
import torch

from tests import gemm_bounds_model as G
from tests import test_gemm_choice
from triton_int_amd import _lib as L

# rows off and on the tile, one column tile, a part of one, K on and off a stage, with and without splits, weights that pass the caches by
SIZES = [(64, 6848, 10240, "ws_64x64"), (33, 64, 16384, "ws_64x64"), (17, 336, 1536, "ws_64x64"), (49, 16, 2064, "ws_64x64"), (63, 400, 20480, "ws_64x64"),
         (20, 16384, 16400, "ws_64x64"), (65, 4384, 2464, "ws_128x64"), (128, 5120, 20480, "ws_128x64"), (85, 6160, 4960, "ws_128x64"), (100, 576, 20016, "ws_128x64")]


@pytest.mark.parametrize("M,N,K,name", SIZES)
def test_planned(M, N, K, name):
    lib = L.lib()
    for epi, dt, bias in ((L.EPI_SCALE_I8, 0, 1), (L.EPI_SCALE_F, 2, 3)):
        for static in (0, 1):
            pr = G.contiguous(1, M, N, K, dt)
            pl = G.plan_for(lib, pr, epi, bias, static_scratch=static)
            assert pl.name.startswith(name), pl
            G.check_launch(pr, pl, store_sample=8)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,name", SIZES)
def test_agree_with_float64(M, N, K, name):
    test_gemm_choice.test_outputs(1, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [65, 128])
def test_grouped(M):
    test_gemm_choice.test_outputs(3, M, 4096, 4096)
