"""KV caches in every memory layout that a program may keep them in."""
import pytest
import torch

D = 128


def _i8(g, *shape):
    return torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)


def _layer(hidden, seed=0):
    """A decoder layer whose activations use the range of int8 at every stage."""
    from triton_int_amd.nn.opt import W8A8OPTDecoderLayer

    torch.manual_seed(seed)
    with torch.device("cuda"):
        layer = W8A8OPTDecoderLayer(hidden, hidden // D, 256)
    acc = 20.0 * 73.0 * hidden ** 0.5
    value = lambda v: torch.tensor(v, dtype=torch.float32, device="cuda")
    for norm in (layer.ln1, layer.ln2):
        norm.weight = torch.full((hidden,), 20.0, device="cuda")
    for lin in (layer.q_proj, layer.k_proj, layer.v_proj):
        lin.a, lin.b = value(30.0 / acc), value(0.1)
    layer.ln2.input_scale = 0.3 / acc
    layer.fc1.a, layer.fc1.b, layer.fc2.a = value(1.0 / acc), value(30.0), value(0.3 / (20.0 * 73.0 * 16.0))
    layer.qk_alpha, layer.score_scale, layer.pv_alpha = 2.5e-3, 0.1, 0.05
    return layer


def _in_layout(values, layout):
    """`values` [heads, rows, cols] as a view of another memory layout."""
    if layout is None:
        return values.clone()
    BH, R, C = values.shape
    if layout == "rows_first":  # memory [rows, heads, cols]
        t = torch.zeros((R, BH, C), dtype=torch.int8, device="cuda").transpose(0, 1)
    elif layout == "cols_first":  # memory [cols, heads, rows]: no unit stride along a row
        t = torch.zeros((C, BH, R), dtype=torch.int8, device="cuda").permute(1, 2, 0)
    elif layout == "pitch":  # rows two bytes apart
        t = torch.zeros((BH, R, C + 2), dtype=torch.int8, device="cuda")[:, :, :C]
    else:  # contiguous, but from byte `layout` on
        t = torch.zeros(BH * R * C + layout, dtype=torch.int8, device="cuda")[layout:].view(BH, R, C)
    return t.copy_(values)


def _check_layer(hidden, S, T, k_layout, vt_layout):
    """The layer's output and both caches: those of contiguous caches, bit for bit."""
    layer = _layer(hidden)
    g = torch.Generator(device="cuda").manual_seed(S * 1000 + T)
    x = torch.randn((1, S, hidden), device="cuda", generator=g)
    k0, vt0 = _i8(g, hidden // D, T, D), _i8(g, hidden // D, D, T)
    k, vt = k0.clone(), vt0.clone()
    want = layer(x, kv_cache=(k, vt))
    k2, vt2 = _in_layout(k0, k_layout), _in_layout(vt0, vt_layout)
    got = layer(x, kv_cache=(k2, vt2))
    assert torch.equal(got, want) and torch.equal(k2, k) and torch.equal(vt2, vt)
    assert not torch.equal(k, k0) and not torch.equal(vt, vt0)


def test_kv_append_takes_heads_side_by_side_and_refuses_rows_that_overlap():
    """The check of the strides alone: addresses are never used, since a call that passes it ends at the missing GPU."""
    from triton_int_amd import _lib as L

    lib, S, heads, refused = L.lib(), 5, 3, -4  # TI_E_STRIDE
    H = heads * D

    def status(k_head_stride, k_row_stride, n=heads):
        return lib.ti_kv_append_i8_seqs(4096, H, 4096, H, 4096, k_head_stride, k_row_stride, 4096, 64, 1, S, n, D, None)

    for head, row in ((D, H - 1), (D - 1, H), (D + 1, H), ((S - 1) * D + D - 1, D), (0, H), (S * D, D - 1)):
        assert status(head, row) == refused, (head, row)
    if not torch.cuda.is_available():
        for head, row in ((D, H), (D, 4 * H), (64 * D, D), (S * D, D), (D + 16, H + 64)):
            assert status(head, row) != refused, (head, row)
        assert status(0, D, 1) != refused


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(1, 53), (17, 40), (20, 80), (70, 133)])
@pytest.mark.parametrize("seqs", [1, 2])
def test_kv_append_into_a_cache_of_whole_positions(seqs, S, T):
    """K stored [T, seqs*heads, D]: the new rows where torch indexing puts them, the rest untouched."""
    from triton_int_amd.kernels import fused

    heads = 3
    g = torch.Generator(device="cuda").manual_seed(S + T)
    qkv = _i8(g, seqs * S, 3 * heads * D)
    k0, vt0 = _i8(g, seqs * heads, T, D), _i8(g, seqs * heads, D, T)
    k, vt = _in_layout(k0, "rows_first"), vt0.clone()
    fused.kv_append_i8(qkv[:, heads * D:2 * heads * D], qkv[:, 2 * heads * D:], k, vt, seqs=seqs)
    by_head = lambda t: t.reshape(seqs, S, heads, D).transpose(1, 2).reshape(seqs * heads, S, D)
    k0[:, T - S:] = by_head(qkv[:, heads * D:2 * heads * D])
    vt0[:, :, T - S:] = by_head(qkv[:, 2 * heads * D:]).transpose(1, 2)
    assert torch.equal(k, k0) and torch.equal(vt, vt0)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [256, 1024])
@pytest.mark.parametrize("S,T", [(1, 53), (20, 53), (20, 80), (200, 400)])
def test_layer_on_a_k_cache_of_whole_positions(hidden, S, T):
    _check_layer(hidden, S, T, "rows_first", None)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [256, 1024])
@pytest.mark.parametrize("k_layout,S,T", [(1, 20, 53), (1, 20, 64), (4, 1, 53), (4, 1, 64), (8, 130, 160), ("pitch", 20, 53), ("cols_first", 1, 53),
                                          ("cols_first", 20, 64)])
def test_layer_on_a_k_cache_that_the_attention_kernel_does_not_take(hidden, k_layout, S, T):
    """Rows of K that do not start at multiples of 16 bytes: the three-launch chain, same bits."""
    _check_layer(hidden, S, T, k_layout, None)


@pytest.mark.gpu
@pytest.mark.parametrize("vt_layout", [None, 1, "pitch"])
@pytest.mark.parametrize("S,T", [(1, 53), (1, 64), (20, 53), (130, 144)])
def test_layer_on_a_vt_cache_at_any_byte(vt_layout, S, T):
    _check_layer(1024, S, T, None, vt_layout)


@pytest.mark.gpu
@pytest.mark.parametrize("k_layout", [1, 2, 4, "pitch", "rows_first"])
@pytest.mark.parametrize("S,T", [(1, 53), (1, 64), (5, 53)])
def test_decode_step_on_a_k_cache_that_the_projections_launch_does_not_write(k_layout, S, T):
    """Rows of K that do not start at multiples of 4 bytes: projections and append as two launches, same bits."""
    _check_layer(1024, S, T, k_layout, None)


@pytest.mark.gpu
@pytest.mark.parametrize("k_layout", [None, "cols_first"])
@pytest.mark.parametrize("hidden,T", [(256, 53), (1024, 53), (1024, 64)])
def test_decode_step_on_v_as_it_leaves_the_projection(k_layout, hidden, T):
    """V kept as [T, heads * 128] and passed as its transposed view: V^T rows without unit stride."""
    layer, heads = _layer(hidden), hidden // D
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((1, 1, hidden), device="cuda", generator=g)
    k0, v = _i8(g, heads, T, D), _i8(g, T, hidden)
    k, vt = k0.clone(), v.t().contiguous().view(heads, D, T)
    want = layer(x, kv_cache=(k, vt))
    k2, vt2 = _in_layout(k0, k_layout), v.t().view(heads, D, T)
    assert vt2.stride(2) == hidden
    got = layer(x, kv_cache=(k2, vt2))
    assert torch.equal(got, want) and torch.equal(k2, k) and torch.equal(vt2, vt)


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(1, 16), (1, 5), (2, 2)])
def test_more_sequences_than_one_launch_takes(S, T):
    """65600 sequences of one head: the bits of the same sequences in parts."""
    layer, B = _layer(128), 65600
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((B, S, 128), device="cuda", generator=g)
    k0, vt0 = _i8(g, B, T, D), _i8(g, B, D, T)
    parts = [slice(b, min(b + 30000, B)) for b in range(0, B, 30000)]
    k, vt, k2, vt2 = k0.clone(), vt0.clone(), k0, vt0
    want = torch.cat([layer(x[p], kv_cache=(k[p], vt[p])) for p in parts])
    assert torch.equal(layer(x, kv_cache=(k2, vt2)), want) and torch.equal(k2, k) and torch.equal(vt2, vt)
    assert torch.equal(layer(x), torch.cat([layer(x[p]) for p in parts]))
