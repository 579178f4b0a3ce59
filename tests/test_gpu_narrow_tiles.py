"""The tiles of 64 columns (gemm_mfma_ws_kernel 64 x 64 and 128 x 64): sizes that are given to them, against float64."""
import pytest
import torch

from tests import gemm_bounds_model as G
from tests import test_gemm_choice
from triton_int_amd import _lib as L

# rows off and on the tile, one column tile, a part of one, K on and off a stage, with and without splits; 20 x 16384 x 16400 has weights that pass the caches by
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


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(100, 16000, 15984), (100, 16000, 16016)])  # 255.7 and 256.3 MB of weights: through the caches, past them
def test_large_weights(M, N, K):
    """Both policies of the 128 x 64 tiles' weights against the tiles that such a launch is given."""
    from triton_int_amd.kernels.linear import linear_a8_w8_b32_o32
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x, w = (torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g) for s in ((M, K), (N, K)))
    bias = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda", generator=g)
    n = L.lib().ti_gemm_num_configs()
    cfg = next(i for i in range(n) if L.lib().ti_gemm_config_name(i).decode().startswith("ws_128x64x256"))
    want = linear_a8_w8_b32_o32(x, w, bias)
    assert torch.equal(linear_a8_w8_b32_o32(x, w, bias, _config=cfg), want)
    rows = [0, 63, 99]
    assert torch.equal(want[rows], (x[rows].double() @ w.double().t() + bias).to(torch.int32))
