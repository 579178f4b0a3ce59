"""The attention of few query rows at the key counts where a launch gets another number of chunks per wave, against the chain of three
kernels: the same bits."""
import pytest
import torch

from triton_int_amd.kernels.bmm import bmm_s8t_s8n_s8t
from triton_int_amd.kernels.fused import attention_i8, softmax_q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [17, 256, 257, 512, 513, 768, 769, 1025, 1280, 1281, 1536, 1537, 2049, 3072, 3073, 4096])
@pytest.mark.parametrize("heads,S,q_len", [(8, 2, 2), (3, 17, 17), (40, 16, 0), (70, 15, 5)])
@pytest.mark.parametrize("aligned", [True, False])
def test_lengths(T, heads, S, q_len, aligned):
    g = torch.Generator(device="cuda").manual_seed(T + S)
    i8 = lambda *s: (torch.randn(s, generator=g, device="cuda") * 30).round_().clamp_(-127, 127).to(torch.int8)  # noqa: E731
    q, k, vt = i8(heads, S, 128), i8(heads, T, 128), i8(heads, 128, (T + 15) // 16 * 16 + (0 if aligned else 3))[:, :, :T]
    got = attention_i8(q, k, vt, 2.5e-3, 0.1, 0.05, causal_q_len=q_len)
    probs = softmax_q(bmm_s8t_s8n_s8t(q, k, 2.5e-3), 0.1, causal_q_len=q_len)
    assert torch.equal(got, bmm_s8t_s8n_s8t(probs, vt.contiguous(), 0.05))
