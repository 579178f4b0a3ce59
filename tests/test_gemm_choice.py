"""The choice of tile and K splits for 65 and more rows: what it plans stays inside its operands, and launches agree with float64."""
import pytest
import torch

from tests import gemm_bounds_model as G
from triton_int_amd import _lib as L

# one row past 64, edges of the 64-, 128- and 256-row tiles, K just beyond 1024 and no multiple of a k-tile, few and many columns
SIZES = [(1, 65, 4096, 1040), (1, 100, 4096, 4096), (1, 129, 304, 16384), (1, 200, 1024, 4096), (1, 257, 512, 20480), (1, 384, 4096, 4080),
         (1, 1000, 1024, 4096), (3, 100, 1024, 2048), (4, 65, 272, 1536), (1, 513, 6848, 1520)]


@pytest.mark.parametrize("B,M,N,K", SIZES)
def test_planned_launches(B, M, N, K):
    lib = L.lib()
    for epi, dt, bias in ((L.EPI_SCALE_I8, 0, 1), (L.EPI_SCALE_F, 2, 3), (L.EPI_SCALE_F, 3, 3)):
        pr = G.contiguous(B, M, N, K, dt)
        pl = G.plan_for(lib, pr, epi, bias)
        assert pl.name.startswith("ws_") and (B == 1 or pl.splits == 1)
        G.check_launch(pr, pl, store_sample=12)
        G.check_launch(pr, G.plan_for(lib, pr, epi, bias, static_scratch=1), store_sample=4)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K", SIZES)
def test_outputs(B, M, N, K):
    from triton_int_amd.kernels.linear import linear_a8_w8_b32_o32, linear_a8_w8_b8_o8, linear_a8_w8_bfp32_ofp32, linear_group_a8_w8_b8_o8
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randint(-127, 128, (M, K), dtype=torch.int8, device=dev, generator=g)
    w = torch.randint(-127, 128, (B * N, K), dtype=torch.int8, device=dev, generator=g)
    acc = a.double() @ w.double().t()  # exact: below 2^53
    b8 = torch.randint(-127, 128, (B * N,), dtype=torch.int8, device=dev, generator=g)
    al, be = torch.tensor(2.0e-4, device=dev), torch.tensor(0.5, device=dev)
    want = (b8.float() * be + acc.float() * al).round().clamp(-128, 127).to(torch.int8)
    if B > 1:
        got = linear_group_a8_w8_b8_o8(a, w, b8, al.repeat(B), be.repeat(B), B)
        assert torch.equal(got, want)
        return
    assert torch.equal(linear_a8_w8_b8_o8(a, w, b8, al, be), want)
    assert torch.equal(linear_a8_w8_b32_o32(a, w, None).double(), acc)
    bias = torch.randn(N, device=dev, generator=g)
    for dt in (torch.float32, torch.float16):
        assert torch.equal(linear_a8_w8_bfp32_ofp32(a, w, bias, al, be, dtype=dt), (bias * be + acc.float() * al).to(dt))


# few 64 x 64 tiles against the lines of small_tiles_lead: K 16 short of a line and on it, 128-byte rows and others, 256 tiles and one more
# row of them, one GEMM and grouped, weights of 4 MB and beyond
SMALL = [(1, 129, 1440, 1232, True), (1, 1024, 1024, 1152, True), (1, 1025, 1024, 1152, False), (1, 383, 624, 2416, True), (1, 383, 624, 2432, False),
         (1, 200, 512, 1408, True), (1, 200, 512, 1536, False), (3, 143, 352, 1040, True), (2, 111, 1168, 6320, True), (2, 111, 1168, 6272, False),
         (1, 256, 3584, 1152, True), (1, 256, 3712, 1152, False)]


@pytest.mark.parametrize("B,M,N,K,small", SMALL)
def test_few_small_tiles(B, M, N, K, small):
    lib = L.lib()
    for epi, dt, bias in ((L.EPI_SCALE_I8, 0, 1), (L.EPI_SCALE_F, 2, 3), (L.EPI_SCALE_F, 4, 3)):
        pr = G.contiguous(B, M, N, K, dt)
        pl = G.plan_for(lib, pr, epi, bias)
        assert pl.name.startswith("mfma_64x64" if small else "ws_")
        G.check_launch(pr, pl, store_sample=12)


@pytest.mark.gpu
@pytest.mark.parametrize("B,M,N,K,small", SMALL)
def test_outputs_of_few_small_tiles(B, M, N, K, small):
    test_outputs(B, M, N, K)


# K = 1024: few small tiles, and the wave-specialised tiles where there are many or their weights are large
@pytest.mark.parametrize("M,N", [(65, 256), (65, 4096), (100, 3072), (128, 4096), (65, 4112), (65, 8192), (128, 8192), (100, 16384), (128, 16384)])
def test_k_1024(M, N):
    lib = L.lib()
    for epi, dt, bias in ((L.EPI_SCALE_I8, 0, 1), (L.EPI_SCALE_F, 2, 3), (L.EPI_SCALE_F, 3, 3)):
        pr = G.contiguous(1, M, N, 1024, dt)
        pl = G.plan_for(lib, pr, epi, bias)
        assert pl.name.startswith("mfma_64x64" if N <= 4096 else "ws_")
        G.check_launch(pr, pl, store_sample=12)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(65, 256), (128, 4096), (65, 4112), (100, 8192)])
def test_outputs_at_k_1024(M, N):
    test_outputs(1, M, N, 1024)


def test_sizes_beyond_the_measured_ones():
    """The times behind the choice hold up to 20480 columns and K = 28672; beyond, the estimate in units of work decides."""
    lib = L.lib()
    for M, N, K, name, splits in ((300, 20480, 4096, "ws_256x160", 1), (300, 50272, 4096, "ws_128x128", 1), (384, 50272, 1024, "ws_128x128", 1),
                                  (500, 4096, 28672, "ws_256x128", 4), (500, 4096, 28688, "ws_128x128", 2)):
        pr = G.contiguous(1, M, N, K, 2)
        pl = G.plan_for(lib, pr, L.EPI_SCALE_F, 3)
        assert pl.name.startswith(name) and pl.splits == splits, (M, N, K, pl)
        G.check_launch(pr, pl, store_sample=2)


@pytest.mark.parametrize("M,N,K", [(1036, 4096, 16384), (1234, 4096, 16384), (799, 4096, 16384), (395, 4096, 16384), (427, 4096, 16384), (666, 4096, 16384), (100, 5120, 20480)])
def test_splits_fill_one_round(M, N, K):
    """No more items than CUs; 395 and 427 rows are the ones that 256 x 128 tiles in four splits lost to 128 x 128 tiles in two."""
    lib = L.lib()
    pr = G.contiguous(1, M, N, K, 2)
    pl = G.plan_for(lib, pr, L.EPI_SCALE_F, 3)
    assert pl.splits == 1 or pl.tiles_m * pl.tiles_n * pl.splits <= 256, pl
    assert M not in (395, 427) or (pl.name.startswith("ws_128x128") and pl.splits == 2), pl
    assert M < 1000 or (pl.name.startswith("ws_256x128") and pl.splits == 1), pl
    G.check_launch(pr, pl, store_sample=4)
