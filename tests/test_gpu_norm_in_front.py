"""A LayerNorm in front of a few rows' GEMM in one launch: the bits of the separate launches."""
import pytest
import torch

from tests.util import DEV
from triton_int_amd import _lib as L

pytestmark = pytest.mark.gpu
COMBO = -3


def rand8(g, *s):
    return torch.randint(-127, 128, s, dtype=torch.int8, device=DEV, generator=g)


def gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


# rows; heads; K: the shortest, no multiple of 256, the last of four vectors a thread, the first of five, the longest.  Units per workgroup 1 .. 15
@pytest.mark.parametrize("M,seqs,heads,K", [(1, 1, 1, 1024), (2, 1, 8, 1040), (3, 3, 40, 4096), (4, 2, 33, 4112), (1, 1, 40, 5120), (4, 4, 13, 5120), (2, 2, 53, 2000)])
@pytest.mark.parametrize("with_beta", [True, False])
def test_qkv(M, seqs, heads, K, with_beta):
    g, lib, st = gen(M * K), L.lib(), L.current_stream(torch.device(DEV))
    N, T, S = heads * 128, 37, M // seqs
    x = torch.randn(M, K + 4, device=DEV, generator=g)[:, :K]
    gamma, beta = torch.randn(K, device=DEV, generator=g) * 20, torch.randn(K, device=DEV, generator=g)
    w, bias = rand8(g, 3 * N, K), rand8(g, 3 * N)
    al, be = torch.rand(3, device=DEV, generator=g) * 1e-3, torch.rand(3, device=DEV, generator=g)
    kv = lambda: (torch.zeros(seqs * heads, T, 128, dtype=torch.int8, device=DEV), torch.zeros(seqs * heads, 128, T, dtype=torch.int8, device=DEV))
    (k1, v1), (k2, v2) = kv(), kv()
    h8, want, got = (torch.empty(M, n, dtype=torch.int8, device=DEV) for n in (K, 3 * N, 3 * N))
    bp = beta.data_ptr() if with_beta else 0
    tail = lambda k, v: (seqs, M, N, K, k.data_ptr() + (T - S) * 128, T * 128, 128, v.data_ptr() + (T - S), T, 128, st)
    L.check(lib.ti_layernorm_q(x.data_ptr(), K + 4, gamma.data_ptr(), bp, 1e-5, h8.data_ptr(), K, M, K, 0, 0, 0, 0, st), "ln")
    L.check(lib.ti_qkv_decode_i8_seqs(h8.data_ptr(), K, w.data_ptr(), K, bias.data_ptr(), al.data_ptr(), be.data_ptr(), want.data_ptr(), 3 * N, *tail(k1, v1)), "qkv")
    L.check(lib.ti_layernorm_qkv_decode_i8_seqs(x.data_ptr(), K + 4, gamma.data_ptr(), bp, 1e-5, w.data_ptr(), K, bias.data_ptr(), al.data_ptr(), be.data_ptr(),
                                                got.data_ptr(), 3 * N, *tail(k2, v2)), "ln + qkv")
    assert torch.equal(got, want) and torch.equal(k1, k2) and torch.equal(v1, v2)


@pytest.mark.parametrize("M,N,K", [(1, 4, 1024), (2, 4099, 1040), (3, 20480, 4096), (4, 16384, 4112), (1, 20480, 5120), (4, 20480, 5120), (2, 8192, 2000)])
def test_fc1(M, N, K):
    g, lib, st = gen(M * N + K), L.lib(), L.current_stream(torch.device(DEV))
    acc = (torch.randn(M, K, device=DEV, generator=g) * 4e4).to(torch.int32)
    x = torch.randn(M, K + 8, device=DEV, generator=g)[:, :K]
    gamma, beta = torch.randn(K, device=DEV, generator=g) * 20, torch.randn(K, device=DEV, generator=g)
    w, bias = rand8(g, N, K), torch.randn(N, device=DEV, generator=g)
    a, b = torch.tensor(2e-5, device=DEV), torch.tensor(30.0, device=DEV)
    h8 = torch.empty(M, K, dtype=torch.int8, device=DEV)
    r1, r2 = (torch.full((M, K), float("nan"), device=DEV) for _ in range(2))
    got, want = (torch.empty(M, N, dtype=torch.int8, device=DEV) for _ in range(2))
    L.check(lib.ti_dq_add_layernorm_q(acc.data_ptr(), K, 1e-5, 0, x.data_ptr(), K + 8, gamma.data_ptr(), beta.data_ptr(), 1e-5, r1.data_ptr(), K, h8.data_ptr(), K, 0, K,
                                      M, K, 0, 0, 0, st), "dq")
    L.check(lib.ti_bmm_i8_config(h8.data_ptr(), 0, K, 1, w.data_ptr(), 0, K, 1, want.data_ptr(), 0, N, 1, 1, M, N, K, bias.data_ptr(), L.TORCH_TO_BIAS[torch.float32],
                                 a.data_ptr(), b.data_ptr(), L.EPI_GELU_I8, L.TORCH_TO_DT[torch.int8], 0, -1, st), "fc1")
    L.check(lib.ti_dq_add_layernorm_linear_gelu_i8(acc.data_ptr(), K, 1e-5, x.data_ptr(), K + 8, gamma.data_ptr(), beta.data_ptr(), 1e-5, r2.data_ptr(), K,
                                                   w.data_ptr(), K, bias.data_ptr(), a.data_ptr(), b.data_ptr(), got.data_ptr(), N, M, N, K, st), "both")
    assert torch.equal(r1, r2) and torch.equal(got, want)


def test_declined():
    g, lib, st = gen(0), L.lib(), L.current_stream(torch.device(DEV))
    M, N, K = 8, 512, 8192
    acc, x, r = torch.zeros(M, K, dtype=torch.int32, device=DEV), torch.zeros(M, K, device=DEV), torch.full((M, K), 7.0, device=DEV)
    gamma, w, s = torch.ones(K, device=DEV), rand8(g, N, K), torch.ones((), device=DEV)
    out = torch.full((M, N), 3, dtype=torch.int8, device=DEV)
    for m, k, xp in ((5, 4096, x.data_ptr()), (1, 5136, x.data_ptr()), (1, 1008, x.data_ptr()), (1, 4096, x.data_ptr() + 4), (1, 4090, x.data_ptr())):
        assert lib.ti_dq_add_layernorm_linear_gelu_i8(acc.data_ptr(), K, 1.0, xp, K, gamma.data_ptr(), 0, 1e-5, r.data_ptr(), K, w.data_ptr(), K, 0, s.data_ptr(),
                                                      s.data_ptr(), out.data_ptr(), N, m, N, k, st) == COMBO
    for a, xp, ro in ((acc, x, x), (acc, x, acc), (acc, x, x[1:]), (acc[1:], x, acc)):  # in place: other workgroups still read what one writes
        assert lib.ti_dq_add_layernorm_linear_gelu_i8(a.data_ptr(), K, 1.0, xp.data_ptr(), K, gamma.data_ptr(), 0, 1e-5, ro.data_ptr(), K, w.data_ptr(), K, 0,
                                                      s.data_ptr(), s.data_ptr(), out.data_ptr(), N, 2, N, 4096, st) == COMBO
    assert (out == 3).all() and (r == 7.0).all() and (x == 0).all() and (acc == 0).all()
