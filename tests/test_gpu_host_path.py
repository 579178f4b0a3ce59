"""The launchers' host path in the extension module (csrc/host.cpp): what it takes gives what the Python path gives, and
what is not the ordinary case is left to the Python path."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rms", [1, 7, np.bool_(True), 0, np.bool_(False), None])
def test_a_flag_that_is_no_bool_counts_as_its_truth_value(rms):
    """use_rms_norm=1 is RMSNorm, as use_rms_norm=True is, in every launcher that has the argument."""
    from triton_int_amd.kernels import fused

    g = torch.Generator(device="cuda").manual_seed(3)
    x, skip = (torch.randn(5, 96, device="cuda", generator=g) + 1.0 for _ in range(2))
    w = 10.0 * torch.rand(96, device="cuda", generator=g)
    calls = {
        "q": lambda f: (fused.layer_norm_fwd_fused_single_pass_q(x, w, None, 1e-5, f),),
        "fp": lambda f: (fused.layer_norm_fwd_fused_single_pass(x, w, None, 1e-5, f),),
        "skip": lambda f: (fused.skip_layer_norm_fwd_fused_single_pass(x, skip, w, None, 1e-5, f),),
        "skip2": lambda f: fused.skip_layer_norm_fwd_fused_single_pass2(x, skip, w, None, 1e-5, f),
    }
    for name, call in calls.items():
        got, want, other = call(rms), call(bool(rms)), call(not rms)
        assert all(torch.equal(a, b) for a, b in zip(got, want)), name
        assert not torch.equal(want[0], other[0]), f"{name}: the two norms agree, so the test shows nothing"


def test_out_of_memory_is_torchs_exception():
    """An output that does not fit raises torch.OutOfMemoryError, as torch.empty does, from every launcher that allocates."""
    from triton_int_amd.kernels import bmm, fused, linear

    a, w = (torch.ones(s, dtype=torch.int8, device="cuda") for s in ((1 << 15, 16), (1 << 14, 16)))
    x, s = torch.ones((1 << 15, 1 << 12), device="cuda"), torch.tensor(1.0, device="cuda")
    b32, g = torch.zeros(1 << 14, dtype=torch.int32, device="cuda"), torch.ones(1 << 12, device="cuda")
    calls = {
        "linear": lambda: linear.linear_a8_w8_b32_o32(a, w, b32),
        "bmm": lambda: bmm.bmm_s8t_s8n_s32t(a[None], w[None]),
        "layernorm_q": lambda: fused.layer_norm_fwd_fused_single_pass_q(x, g, None, 1e-5, True),
        "layernorm": lambda: fused.layer_norm_fwd_fused_single_pass(x, g, None, 1e-5, True),
        "gelu_q": lambda: fused.gelu_q(x, s),
        "per_token": lambda: fused.quantize_per_token_absmax(x),
        "per_tensor": lambda: fused.quantize_per_tensor_absmax(x),
    }
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (32 << 20)) / total)
    taken = []
    try:
        # what other tests left free inside torch's segments, down to half of the smallest output (128 MB)
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                taken.append(torch.empty(64 << 20, dtype=torch.uint8, device="cuda"))
        for name, call in calls.items():
            with pytest.raises(torch.OutOfMemoryError):
                call()
                pytest.fail(f"{name}: its output was allocated")
    finally:
        taken.clear()
        torch.cuda.set_per_process_memory_fraction(1.0)
    for name, call in calls.items():
        call()
    torch.cuda.synchronize()


def test_launches_from_several_threads():
    """Eight threads, a stream each, split-K and other kernels: every result is the one of a single thread."""
    import threading

    from triton_int_amd.kernels import fused, linear

    g = torch.Generator(device="cuda").manual_seed(5)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)
    w, b32, gamma = i8(512, 10240), torch.zeros(512, dtype=torch.int32, device="cuda"), torch.ones(10240, device="cuda")
    xs = [torch.randn((100, 10240), device="cuda", generator=g) for _ in range(8)]

    def once(x):
        q, scale = fused.quantize_per_token_absmax(x)
        return linear.linear_a8_w8_b32_o32(q, w, b32), linear.linear_a8_w8_b32_o32(q[:5], w, b32), scale, \
            fused.layer_norm_fwd_fused_single_pass_q(x, gamma, None, 1e-5, True)

    want = [once(x) for x in xs]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(20):
                    got = once(xs[i])
                    stream.synchronize()
                    if not all(torch.equal(a, b) for a, b in zip(got, want[i])):
                        wrong.append(i)
        except Exception as e:
            wrong.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


class _Declines:
    """In the extension module's place: every call goes the Python path."""

    def __getattr__(self, name):
        return lambda *args: None


class _Records:
    """Passes calls on to the extension module and notes which of them it took."""

    def __init__(self, host):
        self.host, self.taken = host, []

    def __getattr__(self, name):
        def call(*args):
            y = getattr(self.host, name)(*args)
            self.taken.append((name, y is not None))
            return y
        return call


def _flat(y):
    return [t for part in y for t in _flat(part)] if isinstance(y, (tuple, list)) else [y]


def _operands():
    g = torch.Generator(device="cuda").manual_seed(11)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda", generator=g)
    f32 = lambda *s: torch.randn(s, device="cuda", generator=g)
    s = lambda v: torch.tensor(v, dtype=torch.float32, device="cuda")
    return g, i8, f32, s


def _ordinary_calls():
    """(name of the function in the module, call) for every function and the options that change its route."""
    from triton_int_amd.kernels import bmm, fused, linear

    g, i8, f32, s = _operands()
    al, be = s(1e-3), s(0.5)
    a, a3, w, b8, bf = i8(37, 96), i8(2, 19, 96), i8(48, 96), i8(48), f32(48)
    b32 = torch.randint(-1000, 1000, (48,), dtype=torch.int32, device="cuda", generator=g)
    calls = []
    add = lambda name, f: calls.append((name, f))
    for x in (a, a3, a[:1], a[::2], i8(40, 200)[:, 7:103], a[:0]):  # rows, leading dimensions, one row, pitches, no row
        add("linear", lambda x=x: linear.linear_a8_w8_b32_o32(x, w, b32))
        add("linear", lambda x=x: linear.linear_a8_w8_b8_o8(x, w, b8, al, be))
        add("linear", lambda x=x: linear.linear_a8_w8_bfp32_ofp32(x, w, bf, al, be, dtype=torch.float16))
    add("linear", lambda: linear.linear_a8_w8_bfp32_ofp32(a, w, bf.bfloat16(), al, be))
    add("linear", lambda: linear.linear_a8_w8_b32_o32(a, w, b32, torch.empty((37, 48), dtype=torch.int32, device="cuda")))
    w_kn = i8(96, 48)
    add("linear", lambda: linear.linear_a8_w8_b32_o32(a, w_kn.t(), b32))
    al3, be3 = torch.stack([al, al * 2, al]), torch.stack([be, be, be * 2])
    add("linear", lambda: linear.linear_group_a8_w8_b8_o8(a, w, b8, al3, be3, 3))
    res = f32(37, 48)
    add("linear_residual", lambda: linear.linear_a8_w8_bfp32_ofp32_residual(a, w, bf, al, be, res))
    p, q, v = i8(3, 20, 33), i8(3, 17, 33), i8(3, 33, 17)
    add("bmm", lambda: bmm.bmm_s8t_s8n_s32t(p, q))
    add("bmm", lambda: bmm.bmm_s8t_s8t_s32t(p, v))
    add("bmm", lambda: bmm.bmm_s8t_s8n_s8t(p, q, al))
    add("bmm", lambda: bmm.bmm_s8t_s8t_s8t(p, v, al))
    add("bmm", lambda: bmm.bmm_s8t_s8n_f32t(p.transpose(1, 2).contiguous().transpose(1, 2), q, al))
    add("bmm", lambda: bmm.bmm_s8t_s8n_s8t(p, q, al, torch.zeros((20, 3, 17), dtype=torch.int8, device="cuda").transpose(0, 1)))
    x, gm, bt = f32(2, 9, 160), f32(160), f32(160)
    for rms in (False, True):
        for beta in (bt, None):
            add("layernorm_q", lambda rms=rms, beta=beta: fused.layer_norm_fwd_fused_single_pass_q(x, gm, beta, 1e-5, rms))
            for dt in (torch.float32, torch.float16, torch.bfloat16):
                c = lambda t, dt=dt: None if t is None else t.to(dt)
                add("layernorm_fp", lambda rms=rms, beta=beta, c=c: fused.layer_norm_fwd_fused_single_pass(c(x), c(gm), c(beta), 1e-6, rms))
                add("layernorm_fp", lambda rms=rms, beta=beta, c=c: fused.skip_layer_norm_fwd_fused_single_pass2(c(x), c(x * 2), c(gm), c(beta), 1e-6, rms))
    acc = torch.randint(-9999, 9999, (2, 9, 160), dtype=torch.int32, device="cuda", generator=g)
    add("dq_add_layernorm_q", lambda: fused.dq_add_layernorm_q(acc, 1e-4, x, gm, bt, 1e-5))
    acc_wide = torch.randint(-9999, 9999, (2, 9, 192), dtype=torch.int32, device="cuda", generator=g)
    w160, w160x160 = i8(48, 160), i8(160, 160)
    add("gelu_q", lambda: fused.gelu_q(x, s(30.0)))
    add("gelu_q", lambda: fused.gelu_q(x, 30.0))
    add("linear", lambda: linear.linear_a8_w8_b8_o8(a, w, b8, al, 1))
    scores = i8(3, 20, 33)
    add("softmax_q", lambda: fused.softmax_q(scores, 0.1))
    add("softmax_q", lambda: fused.softmax_q(scores, 0.1, 20))
    for t in (x, x.half(), x[:, :, :1], torch.zeros_like(x)):
        add("quantize_per_token", lambda t=t: fused.quantize_per_token_absmax(t.contiguous()))
        add("quantize_per_tensor", lambda t=t: fused.quantize_per_tensor_absmax(t.contiguous(), s(0.25)))
    add("quantize_per_tensor", lambda: fused.quantize_per_tensor_absmax(x))
    # rows that are slices of wider ones, with any leading dimensions that make one row after the other
    for cut in (lambda t: t[..., 3:163], lambda t: t[0, :, 16:176], lambda t: t[:, 4:5, :160], lambda t: t[1:, :1, 8:168], lambda t: t[:1, :0, :160]):
        y, z = cut(f32(2, 9, 200)), cut(f32(2, 9, 184))
        add("layernorm_q", lambda y=y: fused.layer_norm_fwd_fused_single_pass_q(y, gm, bt, 1e-5))
        for dt in (torch.float32, torch.float16):
            wide = [cut(t.to(dt)) for t in (f32(2, 9, 200), f32(2, 9, 176))]
            add("layernorm_fp", lambda t=wide, dt=dt: fused.skip_layer_norm_fwd_fused_single_pass2(t[0], t[1], gm.to(dt), bt.to(dt), 1e-6))
        add("dq_add_layernorm_q", lambda z=z, b=cut(acc_wide): fused.dq_add_layernorm_q(b, 1e-4, z, gm, bt, 1e-5))
        add("softmax_q", lambda b=cut(i8(2, 9, 209)): fused.softmax_q(b, 0.1))
        add("quantize_per_token", lambda y=y: fused.quantize_per_token_absmax(y))
        cut8 = lambda n, c=cut: c(i8(2, 9, n))
        add("linear", lambda b=cut8(208): linear.linear_a8_w8_b32_o32(b, w160, b32))
        add("linear_residual", lambda b=cut8(208), r=cut(f32(2, 9, 240)): linear.linear_a8_w8_bfp32_ofp32_residual(b, w160x160, gm, al, be, r))
    for lead in ((4,), (2, 3)):
        Q, K, V = i8(*lead, 5, 128), i8(*lead, 21, 128), i8(*lead, 128, 21)
        add("attention", lambda Q=Q, K=K, V=V: fused.attention_i8(Q, K, V, 1e-3, 0.1, 0.05, 5))
        add("attention", lambda Q=Q, K=K, V=V: fused.attention_i8(Q, K, V, 1e-3, 0.1, 0.05, 0, torch.empty_like(Q)))

    def caches(B, T):
        return torch.zeros((B * 2, T, 128), dtype=torch.int8, device="cuda"), torch.zeros((B * 2, 128, T), dtype=torch.int8, device="cuda")

    h, w3, b3 = i8(6, 1024), i8(768, 1024), i8(768)
    qkv = i8(30, 768)

    def decode(seqs):
        k, vt = caches(seqs, 13)
        return linear.linear_qkv_decode_a8_w8_b8_o8(h, w3, b3, al3, be3, k, vt, seqs=seqs), k, vt

    def append(seqs, with_k):
        k, vt = caches(seqs, 41)
        fused.kv_append_i8(qkv[:, 256:512], qkv[:, 512:], k if with_k else None, vt, seqs=seqs)
        return k, vt

    for seqs in (1, 3):
        add("qkv_decode", lambda seqs=seqs: decode(seqs))
        add("kv_append", lambda seqs=seqs: append(seqs, True))
        add("kv_append", lambda seqs=seqs: append(seqs, False))
    return calls


def test_every_function_gives_what_the_python_path_gives(monkeypatch):
    """The module takes each of these calls, and its result has the bits, type, shape and layout of the Python path's."""
    from triton_int_amd import _lib as L

    calls, seen = _ordinary_calls(), set()
    for i, (name, call) in enumerate(calls):
        records = _Records(L.host)
        with monkeypatch.context() as m:
            m.setattr(L, "host", records)
            got = _flat(call())
        assert (name, True) in records.taken, f"call {i} ({name}) was declined"
        seen.add(name)
        with monkeypatch.context() as m:
            m.setattr(L, "host", _Declines())
            want = _flat(call())
        assert len(got) == len(want)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b), f"call {i} ({name})"
    methods = {n for n in dir(L.host) if not n.startswith("__")}
    assert seen == methods, methods - seen


def test_python_float_scales_are_uploaded_before_the_module_is_asked(monkeypatch):
    """Scales as python floats: the module takes the call instead of declining it, with the bits of device-tensor scales; a
    scale tensor of the dequantising norm, which the module does not take, is not offered to it."""
    from triton_int_amd import _lib as L
    from triton_int_amd.kernels import bmm, fused, linear

    g, i8, f32, s = _operands()
    a, w, b8, bf, res = i8(37, 96), i8(48, 96), i8(48), f32(48), f32(37, 48)
    p, q, x, gm = i8(3, 20, 33), i8(3, 17, 33), f32(9, 160), f32(160)
    acc = torch.randint(-9999, 9999, (9, 160), dtype=torch.int32, device="cuda", generator=g)
    calls = [lambda v: linear.linear_a8_w8_b8_o8(a, w, b8, v(1e-3), v(0.5)),
             lambda v: linear.linear_a8_w8_bfp32_ofp32(a, w, bf, v(1e-3), v(0.5)),
             lambda v: linear.linear_a8_w8_bfp32_ofp32_residual(a, w, bf, v(1e-3), v(0.5), res),
             lambda v: bmm.bmm_s8t_s8n_s8t(p, q, v(1e-3)),
             lambda v: fused.dq_add_layernorm_q(acc, v(0.5), x, gm, None, 1e-5)]
    for call in calls:
        records = _Records(L.host)
        want = _flat(call(s))
        with monkeypatch.context() as m:
            m.setattr(L, "host", records)
            got = _flat(call(float))
        assert [t for _, t in records.taken] == [True]
        assert all(torch.equal(u, v) for u, v in zip(got, want))
    records = _Records(L.host)
    with monkeypatch.context() as m:
        m.setattr(L, "host", records)
        fused.dq_add_layernorm_q(acc, s(0.5), x, gm, None, 1e-5)
    assert not records.taken


def test_what_is_not_the_ordinary_case_is_declined():
    """The module returns None, and nothing has been written, for every argument that the Python path converts or refuses."""
    from triton_int_amd import _lib as L

    g, i8, f32, s = _operands()
    h, al, be = L.host, s(1e-3), s(0.5)
    a, w, b8 = i8(8, 96), i8(48, 96), i8(48)

    class Sub(torch.Tensor):
        pass

    def linear(a=a, w=w, b=b8, alpha=al, beta=be, out=None, epi=L.EPI_SCALE_I8, dt=L.TORCH_TO_DT[torch.int8], groups=0):
        return h.linear(a, w, b, alpha, beta, out, epi, dt, L.ROUND_RNE_CLAMP, -1, groups)

    assert linear() is not None
    out = torch.full((8, 48), 77, dtype=torch.int8, device="cuda")
    declined = {
        "a on the CPU": linear(a=a.cpu()), "w on the CPU": linear(w=w.cpu()), "bias on the CPU": linear(b=b8.cpu()),
        "a subclass": linear(a=a.as_subclass(Sub)), "no tensor": linear(a=[1, 2]), "a of another type": linear(a=a.float()),
        "a float as scale": linear(alpha=1e-3), "a scale of another type": linear(alpha=al.double()), "one dimension": linear(a=a[0]),
        "K that does not match": linear(w=i8(48, 80)), "a bias of another size": linear(b=i8(47)), "a strided bias": linear(b=i8(96)[::2]),
        "a bias of no known type": linear(b=b8.double()), "rows that need a copy": linear(a=i8(2, 96, 8).transpose(1, 2)),
        "columns apart": linear(a=i8(8, 192)[:, ::2]), "out of another type": linear(out=out.int()), "out of another size": linear(out=out[:4]),
        "a strided out": linear(out=torch.zeros((8, 96), dtype=torch.int8, device="cuda")[:, ::2]), "out on the CPU": linear(out=out.cpu()),
        "an epilogue that does not fit": linear(out=out, epi=L.EPI_SCALE_F), "groups that do not divide": linear(groups=5),
        "scales without a group each": linear(groups=3, out=out), "an output type that does not exist": linear(dt=99),
        "bmm with a flag that is no bool": h.bmm(a[None], w[None], 0, al, None, L.EPI_SCALE_I8, L.TORCH_TO_DT[torch.int8], 0, -1),
        "bmm with batches that differ": h.bmm(i8(2, 8, 96), w[None], False, al, None, L.EPI_SCALE_I8, L.TORCH_TO_DT[torch.int8], 0, -1),
        "layernorm_q of fp16": h.layernorm_q(f32(4, 32).half(), f32(32), None, 1e-5, False, 0),
        "layernorm_q of a view": h.layernorm_q(f32(4, 64)[:, ::2], f32(32), None, 1e-5, False, 0),
        "layernorm_q without a weight": h.layernorm_q(f32(4, 32), None, None, 1e-5, False, 0),
        "layernorm_q with a text": h.layernorm_q(f32(4, 32), f32(32), None, "1e-5", False, 0),
        "layernorm_fp of two types": h.layernorm_fp(f32(4, 32), None, f32(32).half(), None, 1e-5, False, True, False),
        "softmax_q with a tensor as scale": h.softmax_q(i8(4, 32), s(0.1), 0), "softmax_q beyond its range": h.softmax_q(i8(4, 32), 65.0, 0),
        "gelu_q of a view": h.gelu_q(f32(4, 64)[:, ::2], al, 0), "per token of bf16": h.quantize_per_token(f32(4, 32).bfloat16()),
        "per tensor of nothing": h.quantize_per_tensor(f32(0, 32), None),
        "attention of 64 columns": h.attention(i8(2, 3, 64), i8(2, 9, 64), i8(2, 64, 9), 1e-3, 0.1, 0.05, 0, None),
        "attention on rows at odd bytes": h.attention(i8(2, 3, 129)[:, :, 1:], i8(2, 9, 128), i8(2, 128, 9), 1e-3, 0.1, 0.05, 0, None),
        "kv_append into rows that overlap": h.kv_append(i8(3, 128), i8(3, 128), i8(1, 1, 128).expand(1, 5, 128), i8(1, 128, 5), 1),
    }
    assert [k for k, y in declined.items() if y is not None] == []
    torch.cuda.synchronize()
    assert (out == 77).all()
    for name in ("linear", "bmm", "softmax_q"):
        with pytest.raises(TypeError):
            getattr(h, name)(a)


def test_an_integer_beyond_any_double_is_refused():
    """As float() refuses it, from every launcher that takes a number, with nothing launched on the value it would leave."""
    from triton_int_amd.kernels import fused

    g, i8, f32, s = _operands()
    x, gm, big = f32(9, 160), f32(160), 10 ** 400
    acc = torch.randint(-9999, 9999, (9, 160), dtype=torch.int32, device="cuda", generator=g)
    q, k, vt = i8(2, 3, 128), i8(2, 9, 128), i8(2, 128, 9)
    for call in (lambda: fused.layer_norm_fwd_fused_single_pass_q(x, gm, None, big), lambda: fused.layer_norm_fwd_fused_single_pass(x, gm, None, big),
                 lambda: fused.dq_add_layernorm_q(acc, big, x, gm, None, 1e-5), lambda: fused.dq_add_layernorm_q(acc, 0.5, x, gm, None, big),
                 lambda: fused.softmax_q(i8(4, 32), big), lambda: fused.attention_i8(q, k, vt, big, 0.1, 0.05),
                 lambda: fused.attention_i8(q, k, vt, 1e-3, 0.1, big)):
        with pytest.raises(OverflowError):
            call()
