"""int8 attention scores over an odd number of keys: which tile a launch gets, and the scores against float64."""
import pytest
import torch

from tests import gemm_bounds_model as G
from triton_int_amd import _lib as L

SIZES = [(149, 1000, 1000, 128, "mfma_256x256"), (22, 429, 429, 128, "mfma_128x128"), (5, 65, 4001, 16, "ragged_64"), (8, 300, 1001, 64, "ragged_64"), (30, 510, 510, 64, "mfma_128x128"),
         (100, 150, 150, 128, "ragged_64"), (20, 257, 2047, 128, "mfma_128x128"), (150, 90, 90, 128, "mfma_64x64"),
         # sizes that rules by padding alone sent to slower tiles
         (94, 1154, 1154, 64, "mfma_256x256"), (64, 184, 1825, 80, "mfma_256x256"), (37, 504, 504, 128, "mfma_128x128"), (47, 77, 77, 128, "mfma_64x64"), (54, 294, 294, 128, "mfma_128x128"),
         (84, 165, 165, 64, "ragged_64")]


@pytest.mark.parametrize("B,M,N,K,name", SIZES)
def test_planned(B, M, N, K, name):
    pr = G.contiguous(B, M, N, K, 0)
    pl = G.plan_for(L.lib(), pr, L.EPI_SCALE_I8, 0)
    assert pl.name.startswith(name), pl
    G.check_launch(pr, pl, store_sample=6)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K,name", SIZES)
def test_agree_with_float64(B, M, N, K, name):
    from triton_int_amd.kernels.bmm import bmm_s8t_s8n_s8t
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)  # noqa: E731
    q, k = i8(B, M, K), i8(B, N, K)
    got = bmm_s8t_s8n_s8t(q, k, 1e-3)
    alpha = torch.tensor(1e-3, device="cuda")
    for b in (0, B // 2, B - 1):
        want = ((q[b].double() @ k[b].double().t()).float() * alpha).round().clamp(-128, 127).to(torch.int8)
        assert torch.equal(got[b], want)
