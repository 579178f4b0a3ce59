"""What a launch does whose K split finds no memory: it chooses among the unsplit launches, instead of running the split's tile with
whole K (three quarters of the chip idle).  On the CPU, against the library as it is built: native/fake_hip.h stands in for HIP."""
import re
import subprocess

import pytest

from tests import gemm_bounds_model as G
from tests.native import build_native
from triton_int_amd import _lib as L

# the split choice needs more than 32 MiB of partial sums at the first four, 32 MiB at the last
SIZES = [(666, 4096, 16384), (768, 4096, 16384), (300, 10240, 20480), (128, 20480, 20480), (384, 4096, 16384)]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = build_native("split_memory.cpp", tmp_path_factory.mktemp("native"))

    def run(mode, room, *sizes):
        r = subprocess.run([out, mode, str(room), *(",".join(map(str, s)) for s in sizes)], capture_output=True, text=True, check=True, timeout=60)
        rows = [line.split() for line in r.stdout.splitlines()]
        return [(int(rc), name, int(splits), int(n), int(held)) for rc, name, splits, n, held in rows]
    return run


def workgroups(name, M, N):
    bm, bn = map(int, re.match(r"ws_(\d+)x(\d+)x", name).groups())
    return -(-M // bm) * -(-N // bn)


def test_static_scratch_plans_an_unsplit_choice():
    lib = L.lib()
    for M, N, K in SIZES[:4]:
        pr = G.contiguous(1, M, N, K, 2)
        split = G.plan_for(lib, pr, L.EPI_SCALE_F, 3)
        assert split.splits > 1 and split.partial_bytes > 32 << 20
        pl = G.plan_for(lib, pr, L.EPI_SCALE_F, 3, static_scratch=1)
        assert pl.splits == 1 and pl.name.startswith("ws_128x128") and pl.tiles_m * pl.tiles_n >= 160 > split.tiles_m * split.tiles_n
        G.check_launch(pr, pl, store_sample=2)


def test_capture_without_a_workspace(program):
    for (rc, name, splits, launches, held), (M, N, K) in zip(program("capturing", 1 << 40, *SIZES), SIZES):
        assert (rc, splits, launches, held) == (0, 1, 1, 0)
        assert workgroups(name, M, N) >= 160, name


def test_workspace_is_given(program):
    for rc, name, splits, launches, held in program("none", 1 << 40, *SIZES):
        assert rc == 0 and splits > 1 and launches in (1, 2) and held > 0  # the clearing kernel of a new workspace


def test_no_memory_for_a_workspace(program):
    """The launches run all the same, and a smaller workspace that is there is kept and used."""
    for (rc, name, splits, launches, held), (M, N, K) in zip(program("none", 0, *SIZES), SIZES):
        assert (rc, splits, launches, held) == (0, 1, 1, 0)
        assert workgroups(name, M, N) >= 160, name
    small = (100, 1024, 4096)
    room = program("none", 1 << 40, small)[0][4]
    first, second, third = program("none", room, small, SIZES[0], small)
    assert first[0] == 0 and first[2] > 1 and first[4] == room
    assert second[0] == 0 and second[2] == 1 and second[4] == room
    assert third == (0, first[1], first[2], 1, room)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(100, 1024, 4096), (300, 1024, 8192), (666, 512, 16384)])
def test_captured_without_a_workspace(M, N, K):
    """On a stream that never split K: the unsplit choice's outputs, with and without a residual, at every replay."""
    import torch

    from triton_int_amd.kernels.linear import linear_a8_w8_b32_o32, linear_a8_w8_bfp32_ofp32_residual
    lib, dev = L.lib(), torch.device("cuda", 0)
    g = torch.Generator(device=dev).manual_seed(M)
    a, w = (torch.randint(-127, 128, s, dtype=torch.int8, device=dev, generator=g) for s in ((M, K), (N, K)))
    bias, resid = torch.randn(N, device=dev, generator=g), torch.randn(M, N, device=dev, generator=g)
    al, be = torch.tensor(2.0e-4, device=dev), torch.tensor(0.5, device=dev)
    want, want_r = linear_a8_w8_b32_o32(a, w, None), linear_a8_w8_bfp32_ofp32_residual(a, w, bias, al, be, resid)
    assert lib.ti_gemm_last_splits() > 1
    assert torch.equal(want.double(), a.double() @ w.double().t())
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    L.release_workspaces(all_streams=True)
    with torch.cuda.stream(stream), torch.cuda.graph(graph, stream=stream):
        got = linear_a8_w8_b32_o32(a, w, None)
        assert lib.ti_gemm_last_splits() == 1
        got_r = linear_a8_w8_bfp32_ofp32_residual(a, w, bias, al, be, resid)
        assert lib.ti_gemm_last_splits() == 1
    for _ in range(3):
        got.zero_(), got_r.zero_()
        torch.cuda.synchronize()
        graph.replay()
        assert torch.equal(got, want) and torch.equal(got_r, want_r)
        torch.cuda.synchronize()
