"""q/k/v projections of up to 64 rows with the cache append in the same launch, against the grouped launch and torch indexing."""
import pytest
import torch

from triton_int_amd import _lib as L
from triton_int_amd.kernels import linear

pytestmark = pytest.mark.gpu


# one row, odd lengths, several sequences, 16-row edges, the largest; K off a stage; (64, 1): a decode step of 64 sequences
@pytest.mark.parametrize("B,S,heads,D,K,T,room", [(1, 3, 2, 128, 1024, 9, 16), (1, 17, 3, 128, 1040, 40, 48), (2, 17, 4, 64, 2064, 33, 33), (3, 21, 2, 128, 1024, 21, 21),
                                                  (1, 48, 8, 128, 1024, 99, 128), (1, 49, 12, 16, 1024, 60, 77), (1, 64, 40, 128, 5120, 70, 96), (4, 16, 32, 128, 4096, 16, 16),
                                                  (64, 1, 2, 128, 1024, 7, 8)])
@pytest.mark.parametrize("cached", [True, False])
def test_append_in_the_launch(B, S, heads, D, K, T, room, cached):
    g = torch.Generator(device="cuda").manual_seed(B * 10 + T)
    i8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)  # noqa: E731
    H, M = heads * D, B * S
    a, w3, b3 = i8(M, K), i8(3 * H, K), i8(3 * H)
    al = torch.full((3,), 40.0 / (73.0 * 73.0 * K ** 0.5), device="cuda")
    be = torch.full((3,), 0.1, device="cuda")
    k, vt = i8(B * heads, room, D), i8(B * heads, D, room)
    want = linear.linear_group_a8_w8_b8_o8(a, w3, b3, al, be, 3)
    want_k, want_vt = k.clone(), vt.clone()
    if cached:
        want_k[:, T - S:T] = want[:, H:2 * H].reshape(B, S, heads, D).transpose(1, 2).reshape(B * heads, S, D)
    want_vt[:, :, T - S:T] = want[:, 2 * H:].reshape(B, S, heads, D).permute(0, 2, 3, 1).reshape(B * heads, D, S)
    out = torch.empty_like(want)
    lib, st = L.lib(), torch.cuda.current_stream().cuda_stream
    args = lambda kd, vd, m: (a.data_ptr(), K, w3.data_ptr(), K, b3.data_ptr(), al.data_ptr(), be.data_ptr(), out.data_ptr(), 3 * H, B, m, H, K,  # noqa: E731
                              kd, k.stride(0), k.stride(1), vd, vt.stride(1), D, st)
    kd, vd = k.data_ptr() + (T - S) * D if cached else None, vt.data_ptr() + T - S
    L.check(lib.ti_qkv_append_i8_seqs(*args(kd, vd, M)), "ti_qkv_append_i8_seqs")
    assert torch.equal(out, want) and torch.equal(k, want_k) and torch.equal(vt, want_vt)
    # a cache inside an operand: declined, nothing done
    assert lib.ti_qkv_append_i8_seqs(*args(kd, w3.data_ptr() + 64, M)) == -3  # TI_E_COMBO
    assert torch.equal(vt, want_vt)
