"""Launches stored for the Infinity Cache and launches streamed past it: the same kernels, chosen by size, the same bits.  A large
launch (streamed) is compared with the same rows in small ones (kept)."""
import pytest
import torch

from triton_int_amd.kernels.bmm import bmm_s8t_s8n_s8t
from triton_int_amd.kernels.fused import softmax_q
from triton_int_amd.kernels.linear import linear_a8_w8_b8_o8, linear_a8_w8_bfp32_ofp32
from triton_int_amd.nn.fused import DQ_Add_LayerNorm_Q, LayerNormQ

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _int8(g, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, generator=g, device=DEV)


@pytest.mark.parametrize("rows,cols", [(4097, 5120), (20500, 1028), (40960, 512)])  # 20 M elements is the line; the last is on it
def test_row_norms(rows, cols):
    g = torch.Generator(device=DEV).manual_seed(1)
    with torch.device(DEV):
        ln, dq = LayerNormQ(cols), DQ_Add_LayerNorm_Q(cols)
    for m in (ln, dq):
        m.weight, m.bias = torch.randn(cols, generator=g, device=DEV) * 20, torch.randn(cols, generator=g, device=DEV)
    dq.input_scale = 1e-5
    x = torch.randn((rows, cols), generator=g, device=DEV)
    acc = (torch.randn((rows, cols), generator=g, device=DEV) * 40000).to(torch.int32)
    y, (resid, z) = ln(x), dq(x, acc)
    for a, b in ((0, 777), (rows // 2, rows // 2 + 513), (rows - 3, rows)):
        assert torch.equal(y[a:b], ln(x[a:b]))
        r, q = dq(x[a:b], acc[a:b])
        assert torch.equal(resid[a:b], r) and torch.equal(z[a:b], q)


@pytest.mark.parametrize("rows,cols,causal", [(82000, 2048, 0), (82000, 2048, 2000), (82000, 2047, 0), (49152, 2048, 0)])  # beyond 96 Mi scores
def test_softmax(rows, cols, causal):
    g = torch.Generator(device=DEV).manual_seed(2)
    s = _int8(g, rows, cols)
    p = softmax_q(s, 0.05, causal_q_len=causal)
    for a, b in ((0, 2000), (40000, 42000) if causal else (30000, 32000), (rows - 2000 if causal == 0 else 80000, rows if causal == 0 else 82000)):
        assert torch.equal(p[a:b], softmax_q(s[a:b], 0.05, causal_q_len=causal))


@pytest.mark.parametrize("M,N,K,out", [(4096, 8192, 1024, "fp32"), (4099, 8190, 1040, "fp16"), (8200, 16384, 512, "int8"), (8195, 16384, 128, "int8")])
def test_linears(M, N, K, out):
    g = torch.Generator(device=DEV).manual_seed(3)
    x, w = _int8(g, M, K), _int8(g, N, K)
    a, b = torch.tensor(2e-4, device=DEV), torch.tensor(0.1, device=DEV)
    if out == "int8":
        bias = _int8(g, N)
        run = lambda x: linear_a8_w8_b8_o8(x, w, bias, a, b)  # noqa: E731
    else:
        bias = torch.randn(N, generator=g, device=DEV).to(torch.float32 if out == "fp32" else torch.float16)
        run = lambda x: linear_a8_w8_bfp32_ofp32(x, w, bias, a, b)  # noqa: E731
    y = run(x)
    for lo, hi in ((0, 300), (M // 2, M // 2 + 257), (M - 70, M)):
        assert torch.equal(y[lo:hi], run(x[lo:hi]))


def test_attention_scores():
    """The kernel for a short K: 132 MB of scores against single heads."""
    g = torch.Generator(device=DEV).manual_seed(4)
    q, k = _int8(g, 33, 2000, 128), _int8(g, 33, 2000, 128)
    s = bmm_s8t_s8n_s8t(q, k, 1e-3)
    for h in (0, 17, 32):
        assert torch.equal(s[h:h + 1], bmm_s8t_s8n_s8t(q[h:h + 1], k[h:h + 1], 1e-3))
