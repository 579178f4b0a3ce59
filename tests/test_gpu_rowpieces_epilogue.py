"""gemm_rowpieces_kernel's store phase: every bias type and output type, with and without a residual, at the edges of the
consumer threads' share of the (row, unit) pairs.  Sums are integers and every fixed step rounds once, so all of it is exact."""
import pytest
import torch

from triton_int_amd import _lib as L

pytestmark = pytest.mark.gpu

# rows x columns: one pair; N no multiple of 4 (a unit that is cut off); 256 pairs and one more per workgroup; the largest
# share of each row class (20 units); several pairs per thread with a last pass that is nearly empty
SIZES = [(1, 4), (1, 5), (13, 5119), (16, 20480), (17, 4099), (32, 20480), (33, 10241), (48, 16384), (64, 5123), (64, 16384)]


@pytest.mark.parametrize("M,N", SIZES)
def test_store_phase(M, N):
    K = 1040
    dev = torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M * 100003 + N)
    a = torch.randint(-127, 128, (M, K), dtype=torch.int8, device=dev, generator=g)
    w = torch.randint(-127, 128, (N, K), dtype=torch.int8, device=dev, generator=g)
    acc = (a.double() @ w.double().t())
    alpha, beta = torch.tensor(3.1e-4, device=dev), torch.tensor(0.7, device=dev)
    resid = torch.randn((M, N), device=dev, generator=g)
    lib, stream = L.lib(), L.current_stream(dev)
    cfg = next(i for i in range(lib.ti_gemm_num_configs()) if lib.ti_gemm_config_name(i).decode() == f"skinny_m{(M + 15) // 16 * 16}_rowpieces")

    def launch(out, epi, bias, kind):
        rc = lib.ti_bmm_i8_config(a.data_ptr(), 0, K, 1, w.data_ptr(), 0, K, 1, out.data_ptr(), 0, N, 1, 1, M, N, K,
                                  bias.data_ptr() if bias is not None else 0, kind, alpha.data_ptr(), beta.data_ptr(), epi,
                                  L.TORCH_TO_DT[out.dtype], 0, cfg, stream)
        L.check(rc, "ti_bmm_i8_config")
        return out

    new = lambda dt: torch.empty((M, N), dtype=dt, device=dev)
    scaled = acc.float() * alpha
    b32 = torch.randint(-2000, 2000, (N,), dtype=torch.int32, device=dev, generator=g)
    assert torch.equal(launch(new(torch.int32), L.EPI_I32, b32, L.BIAS_I32).double(), acc + b32)
    assert torch.equal(launch(new(torch.int32), L.EPI_I32, None, L.BIAS_NONE).double(), acc)
    b8 = torch.randint(-127, 128, (N,), dtype=torch.int8, device=dev, generator=g)
    want8 = (b8.float() * beta + scaled).round().clamp(-128, 127).to(torch.int8)
    assert torch.equal(launch(new(torch.int8), L.EPI_SCALE_I8, b8, L.BIAS_I8), want8)
    for bt in (torch.float32, torch.float16, torch.bfloat16):
        bias = torch.randn(N, device=dev, generator=g).to(bt)
        want = bias.float() * beta + scaled
        for ot in (torch.float32, torch.float16, torch.bfloat16):
            assert torch.equal(launch(new(ot), L.EPI_SCALE_F, bias, L.TORCH_TO_BIAS[bt]), want.to(ot)), (bt, ot)
    bias = torch.randn(N, device=dev, generator=g)
    out = new(torch.float32)
    rc = lib.ti_linear_i8_residual_f32(a.data_ptr(), K, w.data_ptr(), K, bias.data_ptr(), alpha.data_ptr(), beta.data_ptr(),
                                       resid.data_ptr(), N, out.data_ptr(), N, M, N, K, stream)
    L.check(rc, "ti_linear_i8_residual_f32")
    assert torch.equal(out, bias * beta + scaled + resid)
