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
