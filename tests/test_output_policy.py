"""Which int8 outputs of the persistent GEMM kernels stay in the Infinity Cache: by the bytes of operands and outputs, or because the caller's
next launch reads them."""
import pytest

from triton_int_amd import _lib as L

NEXT_READS = 0x100ff  # 0xff | TI_CONFIG_NEXT_READS


@pytest.mark.parametrize("batch,shared_a,M,N,K,alone,read_next", [
    (1, 1, 1500, 2048, 2048, 1, 1),        # 10 MB
    (1, 1, 2048, 4096, 4096, 0, 1),        # 34 MB: weights and activations would be pushed out for outputs that nobody may read
    (1, 1, 232, 4096, 4096, 0, 1),         # weights are most of the launch
    (1, 1, 1023, 4096, 4096, 0, 1),        # outputs of a quarter of the weights: the line
    (1, 1, 1024, 4096, 4096, 1, 1),
    (1, 1, 2048, 16384, 4096, 0, 1),
    (3, 1, 2048, 5120, 5120, 0, 1),        # 10 + 79 + 31 MB
    (3, 0, 1024, 4096, 4096, 1, 1),        # 13 + 50 + 13 MB
    (6, 0, 1300, 2048, 4096, 0, 1),        # 32 + 50 + 16 MB; shared activations 5 + 50 + 16
    (6, 1, 1300, 2048, 4096, 1, 1),
    (20, 0, 2048, 2048, 256, 0, 1),
    (1, 1, 15625, 16384, 1024, 0, 1),      # 256.0 MB of outputs: the line
    (1, 1, 15626, 16384, 1024, 0, 0),
    (1, 1, 8, 1 << 30, 1 << 20, 0, 0),     # products beyond 64 bits of integers
])
def test_by_bytes(batch, shared_a, M, N, K, alone, read_next):
    keeps = L.lib().ti_gemm_keeps_outputs
    assert keeps(batch, shared_a, M, N, K, -1) == alone
    assert keeps(batch, shared_a, M, N, K, 9) == alone
    assert keeps(batch, shared_a, M, N, K, NEXT_READS) == read_next
    assert keeps(batch, shared_a, M, N, K, 9 | 0x10000) == read_next
