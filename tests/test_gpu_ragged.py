"""Kernels on sizes that are no multiple of anything: attention over any number of keys, several sequences in
one launch."""
import numpy as np
import pytest
import torch

from tests.test_gpu_rowops import _attention_chain_checked
from tests.util import gpu, rng

pytestmark = pytest.mark.gpu


# the last number: the pitch of V^T's rows (0: exactly T, so that rows start at any byte)
@pytest.mark.parametrize("BH,S,T,q_len,pitch", [
    (2, 1, 1, 1, 0), (3, 1, 15, 0, 16), (2, 16, 17, 16, 0), (2, 5, 63, 5, 64), (40, 1, 1531, 1, 2048), (3, 3, 1025, 3, 0),
    (300, 1, 77, 1, 80), (2, 16, 2047, 0, 0), (2, 2, 2049, 2, 4096), (1, 1, 4093, 0, 0),     # few query rows
    (3, 17, 65, 17, 0), (2, 47, 1000, 47, 0), (2, 130, 1007, 0, 1024), (2, 48, 333, 24, 336), (1, 129, 4096, 129, 4096),  # groups of 16
    (49, 333, 333, 333, 336), (49, 333, 333, 333, 0), (70, 240, 257, 0, 0), (130, 128, 129, 128, 0), (2, 17, 4097, 17, 0)])  # blocks of 128
def test_attention_i8_over_any_number_of_keys(BH, S, T, q_len, pitch):
    """Equal to the three-launch chain, bit for bit, whatever the length and the alignment of V^T's rows."""
    from triton_int_amd.kernels import fused

    g = rng(BH * 1000 + S * 7 + T)
    q, k = (g.integers(-127, 128, size=(BH, n, 128), dtype=np.int8) for n in (S, T))
    vt = g.integers(-127, 128, size=(BH, 128, T), dtype=np.int8)
    room = torch.full((BH, 128, max(pitch, T)), 99, dtype=torch.int8, device="cuda")  # what lies past T must not matter
    gvt = room[:, :, :T]
    gvt.copy_(gpu(vt))
    for qk_alpha, score_scale, pv_alpha in ((1e-3, 0.05, 1.0 / 127.0), (4e-3, 0.2, 0.03)):
        want = _attention_chain_checked(q, k, vt, qk_alpha, score_scale, pv_alpha, q_len)
        got = fused.attention_i8(gpu(q), gpu(k), gvt, qk_alpha, score_scale, pv_alpha, causal_q_len=q_len)
        assert torch.equal(got, want), f"{int((got != want).sum())} values differ"


@pytest.mark.parametrize("B,heads,S,T", [(3, 2, 1, 53), (2, 3, 150, 150), (16, 4, 1, 1007)])
def test_attention_i8_of_several_sequences_in_one_launch(B, heads, S, T):
    """4-D operands with a stride per sequence and per head: each sequence as if launched by itself."""
    from triton_int_amd.kernels import fused

    g = torch.Generator(device="cuda").manual_seed(B * 100 + T)
    i8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    q = i8(B, S, 3, heads, 128)[:, :, 0].transpose(1, 2)   # views of a [B, S, 3H] projection
    k, vt = i8(B, heads, T + 3, 128)[:, :, :T], i8(B, heads, 128, T + 16)[:, :, :, :T]
    out = torch.zeros((B, S, heads, 128), dtype=torch.int8, device="cuda")
    fused.attention_i8(q, k, vt, 2e-3, 0.1, 0.02, causal_q_len=S, out=out.transpose(1, 2))
    for b in range(B):
        want = fused.attention_i8(q[b], k[b], vt[b], 2e-3, 0.1, 0.02, causal_q_len=S)
        assert torch.equal(out[b].transpose(0, 1), want)


@pytest.mark.parametrize("B,S,heads,D,K,T,room", [(16, 1, 2, 128, 1024, 53, 64), (3, 5, 5, 16, 1040, 37, 37), (1, 16, 3, 128, 2064, 100, 128)])
def test_qkv_decode_of_several_sequences_into_views_of_longer_caches(B, S, heads, D, K, T, room):
    """Projections equal to the grouped launch's; caches equal to torch indexing, the rest of them untouched.
    The append kernel alone on the same projections: the same caches."""
    from triton_int_amd.kernels import fused, linear

    g = torch.Generator(device="cuda").manual_seed(B * 10 + T)
    i8 = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    H = heads * D
    a, w3, b3 = i8(B * S, K), i8(3 * H, K), i8(3 * H)
    al = torch.full((3,), 40.0 / (73.0 * 73.0 * K ** 0.5), device="cuda")
    be = torch.full((3,), 0.1, device="cuda")
    k0, vt0 = i8(B * heads, room, D), i8(B * heads, D, room)
    want = linear.linear_group_a8_w8_b8_o8(a, w3, b3, al, be, 3)
    want_k, want_vt = k0.clone(), vt0.clone()
    want_k[:, T - S:T] = want[:, H:2 * H].reshape(B, S, heads, D).transpose(1, 2).reshape(B * heads, S, D)
    want_vt[:, :, T - S:T] = want[:, 2 * H:].reshape(B, S, heads, D).permute(0, 2, 3, 1).reshape(B * heads, D, S)
    k, vt = k0.clone(), vt0.clone()
    got = linear.linear_qkv_decode_a8_w8_b8_o8(a, w3, b3, al, be, k[:, :T], vt[:, :, :T], seqs=B)
    assert torch.equal(got, want) and torch.equal(k, want_k) and torch.equal(vt, want_vt)
    k, vt = k0.clone(), vt0.clone()
    fused.kv_append_i8(want[:, H:2 * H], want[:, 2 * H:], k[:, :T], vt[:, :, :T], seqs=B)
    assert torch.equal(k, want_k) and torch.equal(vt, want_vt)
    vt = vt0.clone()
    fused.kv_append_i8(None, want[:, 2 * H:], None, vt[:, :, :T], seqs=B)
    assert torch.equal(vt, want_vt)


@pytest.mark.parametrize("M,N,K", [(1, 512, 16), (16, 20480, 1024), (17, 516, 1040), (33, 1001, 272), (48, 4100, 4096), (64, 16384, 528),
                                   (48, 20478, 256), (16, 26000, 48), (50, 2052, 8192)])
def test_row_piece_kernel_edges(M, N, K):
    """One unit of 4 weight rows per workgroup up to 20 and more than one round, K below and off a stage, N off a
    unit: integer sums and fixed-order epilogues, so every output type is exact (against torch in float64)."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import linear

    lib = L.lib()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    i8 = lambda *shape: torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    a, w, b8 = i8(M, K), i8(N, K), i8(N)
    b32 = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda", generator=g)
    bf, res = torch.randn(N, device="cuda", generator=g), torch.randn((M, N), device="cuda", generator=g)
    acc = (a.double() @ w.double().t()).to(torch.int32)
    alpha, one = torch.tensor(30.0 / (K ** 0.5 * 5400.0), device="cuda"), torch.tensor(1.0, device="cuda")
    f = alpha * acc.float()
    want = bf + f
    # forced: a short K may run on another kernel, and has to give the same there
    names = [lib.ti_gemm_config_name(i).decode() for i in range(lib.ti_gemm_num_configs())]
    for cfg in (names.index(f"skinny_m{(M + 15) // 16 * 16}_rowpieces"), -1):
        assert torch.equal(linear.linear_a8_w8_b32_o32(a, w, b32, _config=cfg), acc + b32)
        assert cfg in (-1, lib.ti_gemm_last_config())
        assert torch.equal(linear.linear_a8_w8_b8_o8(a, w, b8, alpha, one, _config=cfg), (b8.float() + f).round().clamp(-128, 127).to(torch.int8))
        assert torch.equal(linear.linear_a8_w8_bfp32_ofp32(a, w, bf, alpha, one, _config=cfg), want)
        assert torch.equal(linear.linear_a8_w8_bfp32_ofp32(a, w, bf, alpha, one, dtype=torch.float16, _config=cfg), want.half())
    assert torch.equal(linear.linear_a8_w8_bfp32_ofp32_residual(a, w, bf, alpha, one, res), want + res)


@pytest.mark.parametrize("M,N,K", [(1, 512, 16), (3, 1024, 272), (4, 5120, 20480), (5, 2052, 2064), (13, 1001, 784), (16, 4096, 16384), (16, 9000, 1040),
                                   (32, 1024, 1296), (20, 4096, 16384), (40, 12288, 512), (48, 3000, 10240), (64, 2048, 768), (57, 8192, 1008)])
def test_row_piece_kernel_every_stage_length(M, N, K):
    """The chosen and every forced stage length (256, 512, 1024 bytes of K) whose stages fit, K below, at and off a
    stage: exact int32 sums; with the residual's epilogue against the plain one's."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import linear

    lib = L.lib()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, w = (torch.randint(-128, 128, s, dtype=torch.int8, device="cuda", generator=g) for s in ((M, K), (N, K)))
    b32 = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda", generator=g)
    want = (a.double() @ w.double().t()).to(torch.int32) + b32
    names = [lib.ti_gemm_config_name(i).decode() for i in range(lib.ti_gemm_num_configs())]
    cfg = names.index(f"skinny_m{(M + 15) // 16 * 16}_rowpieces")
    for c in (cfg, -1):
        assert torch.equal(linear.linear_a8_w8_b32_o32(a, w, b32, _config=c), want)
    mt, per = (M + 15) // 16 * 16, -(-((N + 3) // 4) // 256)
    for kc in (256, 512, 1024):
        if kc == 256 or (per <= 12 and 3 * (mt + 16 * -(-per // 4)) * kc <= 160 * 1024 and (kc == 512 or mt <= 32)):
            assert torch.equal(linear.linear_a8_w8_b32_o32(a, w, b32, _config=cfg | (kc // 256) << 8), want), kc


@pytest.mark.parametrize("B,M,N,K,pad", [(1, 65, 80, 16, 48), (3, 130, 128, 144, 0), (1, 256, 1024, 4112, 16), (70, 129, 208, 304, 0), (2, 257, 144, 128, 32),
                                         (1, 100, 512, 8192, 0), (40, 700, 128, 1040, 0), (2, 1, 16, 2064, 0)])
def test_kn_operand_on_the_wave_specialised_kernels(B, M, N, K, pad):
    """[K,N] operands with whole 16-byte pieces, both tile sizes and the chosen configuration: K below, at and off a
    k-tile, N and M off a tile, rows at a pitch, split K: exact against torch in float64."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels._gemm import bmm

    lib = L.lib()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randint(-128, 128, (B, M, K + pad), dtype=torch.int8, device="cuda", generator=g)[:, :, :K]
    b = torch.randint(-128, 128, (B, K, N + pad), dtype=torch.int8, device="cuda", generator=g)[:, :, :N]
    alpha = torch.tensor(40.0 / (K ** 0.5 * 5400.0), device="cuda")
    acc = torch.stack([x.double() @ y.double() for x, y in zip(a, b)]).to(torch.int32)
    f = acc.float() * alpha
    names = [lib.ti_gemm_config_name(i).decode() for i in range(lib.ti_gemm_num_configs())]
    for cfg in [-1] + [i for i, nm in enumerate(names) if nm.startswith(("ws_256x128", "ws_128x128"))]:
        for dt, ep, want in ((torch.int8, L.EPI_SCALE_I8, f.round().clamp(-128, 127).to(torch.int8)), (torch.float32, L.EPI_SCALE_F, f),
                             (torch.float16, L.EPI_SCALE_F, f.half())):
            got = bmm(a, b, b_is_kn=True, epilogue=ep, out_dtype=dt, alpha=alpha, config=cfg)
            assert torch.equal(got, want), (cfg, dt)


@pytest.mark.parametrize("M,N,K", [(64, 4096, 16384), (33, 528, 10256), (100, 512, 5120), (300, 1024, 20480)])
def test_split_k_adds_the_residual_in_its_last_item(M, N, K):
    """Linear + residual with K split over workgroups: the bits of the linear followed by an fp32 add."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import linear

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, w = (torch.randint(-128, 128, s, dtype=torch.int8, device="cuda", generator=g) for s in ((M, K), (N, K)))
    bf, res = torch.randn(N, device="cuda", generator=g), torch.randn((M, N), device="cuda", generator=g)
    alpha, one = torch.tensor(30.0 / (K ** 0.5 * 5400.0), device="cuda"), torch.tensor(1.0, device="cuda")
    acc = (a.double() @ w.double().t()).to(torch.int32)
    for _ in range(3):  # the counters are back at zero after every launch
        assert torch.equal(linear.linear_a8_w8_bfp32_ofp32_residual(a, w, bf, alpha, one, res), bf + alpha * acc.float() + res)
        assert L.lib().ti_gemm_last_splits() > 1


@pytest.mark.parametrize("B,M,N,K", [(1, 1, 1, 1), (2, 65, 63, 15), (3, 130, 129, 17), (40, 128, 128, 333), (2, 64, 16, 64), (1, 300, 1000, 1001),
                                     (70, 129, 200, 31), (1, 17, 8, 130), (5, 1, 128, 777)])
def test_ragged_kernel_any_alignment_and_layout(B, M, N, K):
    """Rows that start anywhere (views of a padded buffer at an odd offset), any K, b as [B,N,K] and as [B,K,N],
    both tile sizes: exact against torch in float64; what surrounds the operands must not matter."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import bmm

    lib = L.lib()
    g = torch.Generator(device="cuda").manual_seed(B + M + N + K)

    def view(rows, cols):  # [B, rows, cols] at an odd offset of rows of cols + 3
        buf = torch.randint(-128, 128, (B, rows, cols + 3), dtype=torch.int8, device="cuda", generator=g)
        return buf[:, :, 1:cols + 1]

    a, b_nk, b_kn = view(M, K), view(N, K), view(K, N)
    alpha = torch.tensor(30.0 / (K ** 0.5 * 5400.0), device="cuda")
    names = [lib.ti_gemm_config_name(i).decode() for i in range(lib.ti_gemm_num_configs())]
    for b, kn in ((b_nk, False), (b_kn, True)):
        acc = (a.double() @ (b if kn else b.transpose(1, 2).contiguous()).double()).to(torch.int32)
        for cfg in [-1] + [i for i, nm in enumerate(names) if nm.startswith("ragged")]:
            got = (bmm.bmm_s8t_s8t_s32t if kn else bmm.bmm_s8t_s8n_s32t)(a, b, _config=cfg)
            assert torch.equal(got, acc), (kn, cfg)
            if not (M == N == K == 1):
                assert lib.ti_gemm_config_name(lib.ti_gemm_last_config()).decode().startswith("ragged")
            got8 = (bmm.bmm_s8t_s8t_s8t if kn else bmm.bmm_s8t_s8n_s8t)(a, b, alpha, _config=cfg)
            assert torch.equal(got8, (alpha * acc.float()).round().clamp(-128, 127).to(torch.int8)), (kn, cfg)
    # fp32 output, and an int8 output whose rows start anywhere
    assert torch.equal(bmm.bmm_s8t_s8n_f32t(a, b_nk, alpha), alpha * (a.double() @ b_nk.double().transpose(1, 2).contiguous()).float())
    out = torch.full((B, M, N + 5), 77, dtype=torch.int8, device="cuda")
    bmm.bmm_s8t_s8t_s8t(a, b_kn, alpha, out=out[:, :, 3:N + 3])
    assert torch.equal(out[:, :, 3:N + 3], bmm.bmm_s8t_s8t_s8t(a, b_kn, alpha)) and bool((out[:, :, :3] == 77).all() and (out[:, :, N + 3:] == 77).all())


@pytest.mark.parametrize("M,N,K", [(1, 1, 1025), (17, 63, 1024), (62, 304, 9542), (65, 130, 4097), (129, 128, 2111)])
def test_ragged_kernel_with_k_split(M, N, K):
    """Exact for every split, chosen and forced, both tile sizes and operand layouts, every output class; repeated, since
    the tickets have to be back at zero after each launch."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import bmm, linear

    lib = L.lib()
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, w, wt = (torch.randint(-128, 128, (1, r, c + 3), dtype=torch.int8, device="cuda", generator=g)[:, :, 1:c + 1] for r, c in ((M, K), (N, K), (K, N)))
    acc = (a.double() @ w.double().transpose(1, 2).contiguous()).to(torch.int32)
    acc_kn = (a.double() @ wt.double()).to(torch.int32)
    alpha, one = torch.tensor(30.0 / (K ** 0.5 * 5400.0), device="cuda"), torch.tensor(1.0, device="cuda")
    names = [lib.ti_gemm_config_name(i).decode() for i in range(lib.ti_gemm_num_configs())]
    chosen = {}
    for cfg in [-1] + [i | (s << 8) for i, nm in enumerate(names) if nm.startswith("ragged") for s in (1, 2, 3, 5, 16)]:
        for _ in range(2):
            assert torch.equal(bmm.bmm_s8t_s8n_s32t(a, w, _config=cfg), acc), cfg
            chosen.setdefault(cfg, lib.ti_gemm_last_splits())
            assert torch.equal(bmm.bmm_s8t_s8t_s32t(a, wt, _config=cfg), acc_kn), cfg
            assert torch.equal(bmm.bmm_s8t_s8n_s8t(a, w, alpha, _config=cfg), (alpha * acc.float()).round().clamp(-128, 127).to(torch.int8)), cfg
    assert chosen[-1] > 1
    bf = torch.randn(N, device="cuda", generator=g)
    half = linear.linear_a8_w8_bfp32_ofp32(a[0], w[0], bf.half(), alpha, one)
    assert half.dtype == torch.float16 and torch.equal(half, (bf.half().float() + alpha * acc[0].float()).half())
    res = torch.randn(M, N, device="cuda", generator=g)
    assert torch.equal(linear.linear_a8_w8_bfp32_ofp32_residual(a[0], w[0], bf, alpha, one, res), bf + alpha * acc[0].float() + res)


@pytest.mark.parametrize("rows,cols,q_len", [(3, 1, 0), (4, 7, 0), (6, 15, 3), (5, 17, 5), (8, 333, 8), (6, 1001, 0), (3, 1024 + 9, 3), (2, 2047, 2), (2, 8191, 0)])
@pytest.mark.parametrize("scale", [0.0, 0.1])
def test_softmax_q_rows_at_any_byte(rows, cols, q_len, scale):
    """Rows of an odd pitch at an odd offset, in and out: within the oracle's stated step, equal to the contiguous call,
    and nothing written beside the rows."""
    import oracle as O
    from tests.util import cpu, mismatch_report
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import fused

    g = rng(rows * 10 + cols)
    x = g.integers(-128, 128, size=(rows, cols), dtype=np.int8)
    wide = torch.full((rows, cols + 6), 99, dtype=torch.int8, device="cuda")
    wide[:, 3:cols + 3] = gpu(x)
    out = torch.full((rows, cols + 4), 77, dtype=torch.int8, device="cuda")
    rc = L.lib().ti_softmax_q(wide.data_ptr() + 3, cols + 6, scale, out.data_ptr() + 1, cols + 4, rows, cols, q_len, L.current_stream(out.device))
    assert rc == 0
    got = out[:, 1:cols + 1]
    assert bool((out[:, 0] == 77).all() and (out[:, cols + 1:] == 77).all())
    mx, rate = mismatch_report(cpu(got), O.softmax_q(x, scale, causal_q_len=q_len))
    assert mx <= 1 and rate <= max(2e-3, 1.5 / got.numel())
    assert torch.equal(got, fused.softmax_q(gpu(x), scale, causal_q_len=q_len))


@pytest.mark.parametrize("shape", [(1,), (7,), (8, 1024), (3, 1001), (2000, 640), (1, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_quantize_per_tensor_is_the_torch_steps_bit_for_bit(shape, dtype):
    """Against torch's own steps on the GPU, unaligned views and a tensor of zeros included."""
    from triton_int_amd.kernels import fused

    g = torch.Generator(device="cuda").manual_seed(sum(shape))
    base = (torch.randn((int(np.prod(shape)) + 1,), device="cuda", generator=g) * 3).to(dtype)
    ws = torch.tensor(0.0123, device="cuda")
    for x in (base[:-1].view(shape), base[1:].view(shape), base[1:].view(shape) * 1e-3, torch.zeros(shape, dtype=dtype, device="cuda")):
        kept = x.clone()
        q, s, alpha = fused.quantize_per_tensor_absmax(x, ws)
        want_s = x.abs().max() / 127
        assert q.dtype == torch.int8 and q.shape == x.shape and torch.equal(x, kept)
        assert torch.equal(s, want_s) and torch.equal(alpha, want_s.float() * ws)
        assert torch.equal(q, (x / want_s).round_().to(torch.int8))


@pytest.mark.parametrize("M,N,K,batch,kernel", [
    (1, 4096, 64, 1, "slab"), (16, 20480, 256, 1, "slab"), (16, 1024, 272, 1, "rowpieces"), (17, 4096, 128, 1, "slab"), (32, 512, 144, 1, "rowpieces"),
    (33, 12288, 64, 1, "slab"), (33, 11264, 64, 1, "rowpieces"), (64, 20480, 80, 1, "rowpieces"),                # one round
    (1, 26000, 1008, 1, "slab"), (12, 13824, 256, 3, "slab"), (20, 20480, 512, 3, "slab"), (20, 12288, 528, 3, "rowpieces"),
    (64, 11008, 64, 4, "slab"), (64, 16384, 272, 3, "rowpieces"), (8, 4096, 1024, 1, "rowpieces")])               # more, and K of 1024
def test_short_k_against_few_rows_at_the_edges_of_the_rule(M, N, K, batch, kernel):
    """Which kernel a short K runs on, and the same sums from both, residual included."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import linear
    from triton_int_amd.kernels._gemm import linear_group

    lib = L.lib()
    names = [lib.ti_gemm_config_name(i).decode() for i in range(lib.ti_gemm_num_configs())]
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, w = (torch.randint(-128, 128, s, dtype=torch.int8, device="cuda", generator=g) for s in ((M, K), (batch * N, K)))
    want = (a.double() @ w.double().t()).to(torch.int32)
    other = names.index(f"skinny_m{(M + 15) // 16 * 16}_rowpieces" if kernel == "slab" else f"skinny_m{16 if M <= 16 else 32 if M <= 32 else 64}_slab16")
    for cfg in (-1, other):
        if batch == 1:
            got = linear.linear_a8_w8_b32_o32(a, w, torch.zeros(N, dtype=torch.int32, device="cuda"), _config=cfg)
        else:
            got = linear_group(a, w, batch, epilogue=L.EPI_I32, out_dtype=torch.int32, config=cfg)
        assert torch.equal(got, want), cfg
        assert (kernel in names[lib.ti_gemm_last_config()]) == (cfg == -1)
    if batch == 1:
        one, res = torch.tensor(1.0, device="cuda"), torch.randn((M, N), device="cuda", generator=g)
        got = linear.linear_a8_w8_bfp32_ofp32_residual(a, w, torch.zeros(N, device="cuda"), one, one, res)
        assert torch.equal(got, want.float() + res)
