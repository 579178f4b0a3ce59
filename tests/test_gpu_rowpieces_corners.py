"""int8 outputs of up to 64 rows that the row-piece kernel takes from the slabs and the 64 x 128 tiles: odd columns at any K, 16385 .. 20480
columns; against float64."""
import pytest
import torch

from tests import gemm_bounds_model as G
from triton_int_amd import _lib as L

SIZES = [(64, 17000, 4096), (49, 20479, 2048), (64, 20480, 2048), (64, 511, 1024), (17, 300, 1040), (33, 1111, 20000), (48, 5001, 12000), (63, 3, 16000), (64, 1001, 9008)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_planned(M, N, K):
    pr = G.contiguous(1, M, N, K, 0)
    pl = G.plan_for(L.lib(), pr, L.EPI_SCALE_I8, 1)
    assert pl.name.endswith("rowpieces"), pl
    G.check_launch(pr, pl, store_sample=8)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SIZES)
def test_agree_with_float64(M, N, K):
    from triton_int_amd.kernels.linear import linear_a8_w8_b8_o8
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)  # noqa: E731
    a, w, b = i8(M, K), i8(N, K), i8(N)
    al, be = torch.tensor(2.0e-4, device="cuda"), torch.tensor(0.5, device="cuda")
    acc = a.double() @ w.double().t()
    want = (b.float() * be + acc.float() * al).round().clamp(-128, 127).to(torch.int8)
    assert torch.equal(linear_a8_w8_b8_o8(a, w, b, al, be), want)
