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
    try:
        for name, call in calls.items():
            with pytest.raises(torch.OutOfMemoryError):
                call()
                pytest.fail(f"{name}: its output was allocated")
    finally:
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
