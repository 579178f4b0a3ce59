"""Launches stored for the Infinity Cache and launches streamed past it: the same kernels, chosen by size, the same bits.  A large
launch (streamed) is compared with the same rows in small ones (kept)."""
import ctypes

import pytest
import torch

from triton_int_amd import _lib as L
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


@pytest.mark.parametrize("rows,cols,causal", [(82000, 2048, 0), (82000, 2048, 2000), (82000, 2047, 0),
                                              (32768, 2048, 0), (32769, 2048, 0), (49176, 2047, 0), (49177, 2047, 0)])  # beyond 64 and 96 Mi scores; each line from both sides
def test_softmax(rows, cols, causal):
    g = torch.Generator(device=DEV).manual_seed(2)
    s = _int8(g, rows, cols)
    p = softmax_q(s, 0.05, causal_q_len=causal)
    for a, b in ((0, 2000), (40000, 42000) if causal else (30000, 32000), (rows - 2000 if causal == 0 else 80000, rows if causal == 0 else 82000)):
        assert torch.equal(p[a:b], softmax_q(s[a:b], 0.05, causal_q_len=causal))


@pytest.mark.parametrize("M,N,K,out", [(4096, 8192, 1024, "fp32"), (4099, 8190, 1040, "fp16"), (8200, 16384, 512, "int8"), (8195, 16384, 128, "int8")])
def test_linears(M, N, K, out):
    """int8: 135 MB and more of operands and outputs, streamed, against rows of it, kept.  4- and 2-byte outputs stream at any size: whole launches
    against rows of them on other tiles."""
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


def _name():
    return L.lib().ti_gemm_config_name(L.lib().ti_gemm_last_config()).decode()


def test_attention_scores():
    """The kernel for a short K: 132 MB of scores (streamed) against eight heads of them (32 MB, kept)."""
    g = torch.Generator(device=DEV).manual_seed(4)
    q, k = _int8(g, 33, 2000, 128), _int8(g, 33, 2000, 128)
    s = bmm_s8t_s8n_s8t(q, k, 1e-3)
    assert _name().startswith("shortk_")
    for h in (0, 13, 25):
        part = bmm_s8t_s8n_s8t(q[h:h + 8], k[h:h + 8], 1e-3)
        assert _name().startswith("shortk_") and torch.equal(s[h:h + 8], part)


def _scores(q, k, config):
    """q [B,M,K], k [B,N,K] -> int8 [B,M,N], through the C entry"""
    (B, M, K), N = q.shape, k.shape[1]
    out = torch.full((B, M, N), 99, dtype=torch.int8, device=DEV)
    alpha = torch.tensor(0.4 / (74 * K ** 0.5), device=DEV)
    rc = L.lib().ti_bmm_i8_config(q.data_ptr(), M * K, K, 1, k.data_ptr(), k.stride(0), k.stride(1), k.stride(2), out.data_ptr(), M * N, N, 1, B, M, N, K, 0, L.BIAS_NONE,
                                  alpha.data_ptr(), 0, L.EPI_SCALE_I8, L.DT_I8, L.ROUND_RNE_CLAMP, config, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, L.lib().ti_last_error()
    return out


@pytest.mark.parametrize("name", ["stream_256x256", "stream_128x128", "ws_256x128", "ws_256x160", "ws_128x128", "shortk_256x256", "kn ws_256x128", "kn ws_128x128"])
def test_next_launch_reads(name):
    """Every kernel of both policies: 108 MB, streamed, and kept because the caller says that its next launch reads it; ragged rows and columns."""
    n = L.lib().ti_gemm_num_configs()
    cfg = next(i for i in range(n) if L.lib().ti_gemm_config_name(i).decode().startswith(name.split()[-1]))
    g = torch.Generator(device=DEV).manual_seed(5)
    B, M, N, K = 6, 2051, 8208, 128
    if name.startswith("kn"):
        k = _int8(g, B, K, N).transpose(1, 2)
    else:
        k = _int8(g, B, N, K)
    q = _int8(g, B, M, K)
    streamed, kept = _scores(q, k, cfg), _scores(q, k, cfg | 0x10000)
    assert torch.equal(streamed, kept)
    assert torch.equal(streamed[2:3, 1000:], _scores(q[2:3, 1000:].contiguous(), k[2:3], cfg))  # kept: 9 MB
    chosen = _scores(q, k, 0xff | 0x10000)
    assert torch.equal(chosen, streamed)
