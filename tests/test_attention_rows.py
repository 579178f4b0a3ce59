"""Which attention kernel a launch runs on, and that the choice changes no bit."""
import pytest
import torch


def test_up_to_16_query_rows_run_on_the_one_pass_kernel_at_any_batch():
    """A 128-row block with 16 live rows walks the keys three times on a quarter of the waves: 27 sequences of 40 heads that
    decode one token each are more than 1024 groups and still belong on the one-pass kernel."""
    from triton_int_amd import _lib as L

    rows = lambda heads, S, T: L.lib().ti_attention_i8_rows(heads, S, T, 128, 128, T)
    for heads in (1, 1024, 1025, 1080, 5120, 65535):
        for S in (1, 2, 15, 16):
            assert rows(heads, S, 1) == rows(heads, S, 2048) == rows(heads, S, 4096) == 16, (heads, S)
            assert rows(heads, S, 4097) == 128  # the scores of a row no longer fit the registers
    assert rows(64, 256, 1064) == 16 and rows(65, 256, 1064) == 128 and rows(1280, 17, 2048) == 128


def test_more_query_rows_run_on_the_kernel_that_measures_faster():
    """Several rounds of 16-row groups against few keys, or against caches that every round reads again, cost more than one
    round of 128-row blocks."""
    from triton_int_amd import _lib as L

    rows = lambda heads, S, T: L.lib().ti_attention_i8_rows(heads, S, T, 128, 128, T)
    for heads, S, T in ((160, 64, 64), (80, 128, 128), (512, 32, 128), (512, 17, 1024), (256, 64, 2048), (160, 48, 64), (340, 48, 2048), (40, 384, 384)):
        assert rows(heads, S, T) == 128, (heads, S, T)
    for heads, S, T in ((32, 64, 1064), (64, 128, 333), (8, 17, 64), (32, 512, 2048), (40, 128, 512), (128, 17, 2048), (40, 333, 2048), (1, 129, 4096)):
        assert rows(heads, S, T) == 16, (heads, S, T)


def test_rows_of_vt_at_any_byte_cost_the_groups_more():
    """us, groups / blocks, V^T rows of 16-byte pieces and others: 32 heads x 387 x 387 13.9 / 20.3 and 29.5 / 21.8."""
    from triton_int_amd import _lib as L

    rows = lambda heads, S, T, pitch: L.lib().ti_attention_i8_rows(heads, S, T, 128, 128, pitch)
    for heads, S, T in ((32, 387, 387), (40, 377, 763), (64, 129, 129)):
        assert rows(heads, S, T, (T + 15) // 16 * 16) == 16 and rows(heads, S, T, T) == 128, (heads, S, T)
    for heads, S, T in ((40, 207, 207), (48, 229, 229), (80, 115, 243), (8, 19, 1103)):
        assert rows(heads, S, T, T) == 16, (heads, S, T)


@pytest.mark.gpu
@pytest.mark.parametrize("S", [1, 16, 17])
@pytest.mark.parametrize("heads,T", [(1024, 33), (1025, 33), (1030, 80), (2600, 17)])
def test_more_heads_than_four_rounds_of_the_chip(heads, S, T):
    """All heads in one launch against the same heads in launches of 500, bit for bit."""
    from triton_int_amd.kernels.fused import attention_i8

    g = torch.Generator(device="cuda").manual_seed(heads + S)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)
    q, k, vt = i8(heads, S, 128), i8(heads, T, 128), i8(heads, 128, T)
    causal = S if S <= T else 0
    call = lambda p: attention_i8(q[p], k[p], vt[p], 1e-3, 0.1, 0.05, causal_q_len=causal)
    got = call(slice(None))
    assert torch.equal(got, torch.cat([call(slice(i, i + 500)) for i in range(0, heads, 500)])) and got.any()


@pytest.mark.gpu
@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("seqs,heads", [(1, 3), (1, 33), (13, 5), (43, 3)])  # 8, 4, 2 and 1 workgroups per head
def test_one_query_row_equals_the_three_kernels(seqs, heads, aligned):
    """All lengths at which a wave, a group of loads or a piece of V^T ends, against scores -> softmax -> P.V, bit for bit."""
    from triton_int_amd.kernels import bmm
    from triton_int_amd.kernels.fused import attention_i8, softmax_q

    H = seqs * heads
    g = torch.Generator(device="cuda").manual_seed(H)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)
    for T in (1, 15, 16, 17, 63, 64, 65, 511, 1008, 1023, 1024, 1025, 2033, 2048, 2049, 4095, 4096):
        room = (T + 31) // 16 * 16 + (0 if aligned else 3)
        q, k, vt = i8(H, 1, 128), i8(H, T, 128), i8(H, 128, room)[:, :, :T]
        for qk_alpha, scale, pv_alpha in ((1e-3, 0.05, 0.05), (-2e-3, 0.5, 0.02), (6e-4, 0.5, 0.05)):
            p = softmax_q(bmm.bmm_s8t_s8n_s8t(q, k, qk_alpha), scale)
            want = bmm.bmm_s8t_s8n_s8t(p, vt.contiguous(), pv_alpha)
            for causal in (0, 1):
                got = attention_i8(q, k, vt, qk_alpha, scale, pv_alpha, causal_q_len=causal)
                assert torch.equal(got, want), (T, qk_alpha, causal)
        assert want.any()  # few saturated scores: probabilities above 1/254 however long the row
        # one score for every key: a wave's sum of 256 largest exponentials
        got = attention_i8(torch.zeros_like(q), k, vt, 1e-3, 0.05, 0.5)
        p = softmax_q(torch.zeros((H, 1, T), dtype=torch.int8, device="cuda"), 0.05)
        assert torch.equal(got, bmm.bmm_s8t_s8n_s8t(p, vt.contiguous(), 0.5)), T
