"""The extension module's decoder layer against the step-by-step path: the same bits over the forms both take, and everything
that only Python can honour is left to it."""
import threading

import pytest
import torch

from tests.util import DEV
from triton_int_amd import _lib as L
from triton_int_amd.nn import fused, linear, opt
from triton_int_amd.nn.linear import W8A8B8O8Linear, W8A8BFP32OFP32Linear

pytestmark = pytest.mark.gpu
HIDDEN, HEADS, FFN = 1024, 8, 2048


@pytest.fixture(scope="module")
def layer():
    with torch.device(DEV):
        m = opt.W8A8OPTDecoderLayer(HIDDEN, HEADS, FFN)
    m.randomize(3)
    m.qk_alpha, m.score_scale, m.pv_alpha = 2e-4, 0.1, 0.05
    m(torch.zeros(1, 1, HIDDEN, device=DEV))  # the pack is there
    return m


def cache(B, T, room, seed, k_rows_first=False, odd=False):
    g = torch.Generator(device=DEV).manual_seed(seed)
    new = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device=DEV, generator=g)
    k = new(T, B * HEADS, 128).transpose(0, 1) if k_rows_first else new(B * HEADS, room, 128)[:, :T]
    vt = new(B * HEADS, 128, room + 3 if odd else room)[:, :, :T]
    return k, vt


def native(layer, x, kv):
    return L.layer_host.decoder_layer(layer, x, kv, opt._TYPES, opt._GLOBAL_HOOKS)


def both(layer, x, kv=None):
    clone = lambda c: None if c is None else tuple(torch.empty_strided(t.shape, t.stride(), dtype=t.dtype, device=t.device).copy_(t) for t in c)
    kv1, kv2 = clone(kv), clone(kv)
    got, want = native(layer, x, kv1), layer._forward_steps(x, kv2, None, None)
    assert got is not None and got.shape == want.shape and got.is_contiguous() and not got.requires_grad
    assert torch.equal(got, want)
    if kv is not None:
        assert torch.equal(kv1[0], kv2[0]) and torch.equal(kv1[1], kv2[1])
    assert torch.equal(layer(x, kv_cache=clone(kv)), want)


@pytest.mark.parametrize("B,S", [(1, 1), (1, 15), (2, 17), (3, 43), (1, 130), (4, 16)])
def test_prompt(layer, B, S):
    x = torch.randn(B, S, HIDDEN, device=DEV, generator=torch.Generator(device=DEV).manual_seed(S))
    both(layer, x)
    both(layer, torch.cat([x, x], -1)[..., :HIDDEN])  # rows of a wider tensor


@pytest.mark.parametrize("B,S,T,room,first,odd", [(1, 1, 64, 64, False, False), (2, 1, 65, 128, False, True), (16, 1, 31, 64, False, False), (3, 5, 40, 40, True, False),
                                                  (1, 17, 100, 256, False, False), (2, 64, 64, 80, False, True), (17, 1, 33, 48, False, False)])
def test_cache(layer, B, S, T, room, first, odd):
    x = torch.randn(B, S, HIDDEN, device=DEV, generator=torch.Generator(device=DEV).manual_seed(T))
    both(layer, x, cache(B, T, room, B, first, odd))
    layer.causal = False
    try:
        both(layer, x, cache(B, T, room, B, first, odd))
    finally:
        layer.causal = True


def test_what_only_python_can_honour(layer):
    x = torch.randn(1, 3, HIDDEN, device=DEV)
    want = layer(x)
    assert native(layer, x, None) is not None
    seen = []
    handle = layer.fc1.register_forward_hook(lambda m, i, o: seen.append(tuple(o.shape)))
    assert native(layer, x, None) is None and torch.equal(layer(x), want) and seen == [(1, 3, FFN)]
    handle.remove()
    handle = torch.nn.modules.module.register_module_forward_pre_hook(lambda m, i: seen.append(type(m)))
    assert native(layer, x, None) is None
    handle.remove()
    layer.fc2.forward_add = lambda a, r: seen.append("add") or W8A8BFP32OFP32Linear.forward_add(layer.fc2, a, r)
    assert native(layer, x, None) is None and torch.equal(layer(x), want) and seen[-1] == "add"
    del layer.fc2.forward_add

    class Other(W8A8B8O8Linear):
        pass
    layer.q_proj.__class__ = Other
    assert native(layer, x, None) is None
    layer.q_proj.__class__ = W8A8B8O8Linear
    # another weight tensor: the pack is stale until the Python path has rebuilt it
    old = layer.k_proj.weight
    layer.k_proj.weight = torch.zeros_like(old)
    assert native(layer, x, None) is None
    changed = layer(x)
    assert native(layer, x, None) is not None and torch.equal(native(layer, x, None), changed)
    layer.k_proj.weight = old
    assert torch.equal(layer(x), want)
    # a mutated buffer is seen as it is now
    bias = layer.fc2.bias.clone()
    layer.fc2.bias += 1.0
    assert torch.equal(native(layer, x, None), layer._forward_steps(x, None, None, None))
    layer.fc2.bias.copy_(bias)
    for bad in (x.half(), x.cpu(), x[0], x[:, :0], x.transpose(0, 1).expand(3, 2, HIDDEN).transpose(0, 1)[..., ::2]):
        assert native(layer, bad, None) is None
    k, vt = cache(1, 8, 16, 0)
    for kv in ((k[:, :, :64], vt), (k[1:], vt[1:]), (k, vt.half()), [k, vt], (k, None)):
        assert native(layer, x, kv) is None
    assert native(layer, torch.randn(1, 9, HIDDEN, device=DEV), (k, vt)) is None  # more new positions than the cache holds


@pytest.mark.parametrize("where,name", [
    (fused.LayerNormQ, "forward"), (fused.DQ_Add_LayerNorm_Q, "forward"), (linear.W8A8B32O32LinearWithoutScaling, "_launch"), (linear._Int8Linear, "forward"),
    (fused.W8A8BFP32OFP32_GeLu_Q, "_launch"), (W8A8BFP32OFP32Linear, "forward_add"), (torch.nn.Module, "__call__"), (torch.nn.Module, "_call_impl"),
    (opt.W8A8OPTDecoderLayer, "_append"), (opt.W8A8OPTDecoderLayer, "_qkv_pack"), (opt.W8A8OPTDecoderLayer, "_forward_steps"),
    (opt, "attention_i8"), (opt, "linear_group_a8_w8_b8_o8"), (fused, "dq_add_layernorm_q_cpp"), (linear, "linear_a8_w8_b32_o32")])
def test_replaced_for_every_instance(layer, monkeypatch, where, name):
    """A method replaced on a class, or a launcher in the module that calls it, runs inside the layer."""
    x = torch.randn(1, 17, HIDDEN, device=DEV)
    want, seen, original = layer(x), [], getattr(where, name)

    def replacement(*args, **kwargs):
        seen.append(name)
        return original(*args, **kwargs)
    with monkeypatch.context() as m:
        m.setattr(where, name, replacement)
        assert native(layer, x, None) is None
        assert torch.equal(layer(x), want) and seen
    assert torch.equal(native(layer, x, None), want)


def test_on_another_stream_and_captured(layer):
    x = torch.randn(2, 3, HIDDEN, device=DEV)
    want = layer._forward_steps(x, None, None, None)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = layer(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            static = layer(x)
    torch.cuda.current_stream().wait_stream(s)
    assert torch.equal(got, want)
    for _ in range(3):
        static.zero_()
        graph.replay()
        assert torch.equal(static, want)
        torch.cuda.synchronize()


def test_buffers_replaced_by_another_thread(layer):
    x = torch.randn(2, 3, HIDDEN, device=DEV)
    want = layer(x)
    first, stop = layer.fc2.weight, threading.Event()

    def replace():
        stream = torch.cuda.Stream()
        while not stop.is_set():
            with torch.cuda.stream(stream):
                fresh = first.clone()
                stream.synchronize()
            layer.fc2.weight = fresh

    stream0 = torch.cuda.current_stream()
    worker = threading.Thread(target=replace)
    worker.start()
    try:
        for _ in range(50):
            got = layer(x)
            stream0.synchronize()
            assert torch.equal(got, want)
    finally:
        stop.set()
        worker.join()
        layer.fc2.weight = first
