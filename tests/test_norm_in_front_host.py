"""The entry points with a LayerNorm in front of a GEMM decline what only two launches compute as their header says, on the CPU."""
import subprocess

import pytest

from tests import gemm_bounds_model as G
from tests.native import build_native

OK, COMBO = 0, -3


@pytest.fixture(scope="module")
def said(tmp_path_factory):
    program = build_native("norm_in_front.cpp", tmp_path_factory.mktemp("native"))
    out = subprocess.run([program], capture_output=True, text=True, check=True, timeout=60).stdout
    return {name: (int(rc), int(launches)) for name, rc, launches in (line.split() for line in out.splitlines())}


def test_outputs_that_share_memory(said):
    apart = {"fc1", "fc1_no_bias", "fc1_out_after_acc", "fc1_out_before_x", "qkv", "qkv_out_after_x", "qkv_k_ends_before_x"}
    shared = [n for n in said if ("_in_" in n or "_is_" in n)]
    assert len(shared) >= 14
    for name in apart:
        assert said[name] == (OK, 1), name
    for name in shared:
        assert said[name] == (COMBO, 0), name


def test_pitches_of_whole_pieces(said):
    """The separate norm sums rows at other pitches in another order, a single row among them."""
    for name, got in said.items():
        if "_row" in name:
            assert got == ((COMBO, 0) if "_odd_" in name else (OK, 1)), name


def test_no_columns(said):
    """The residual is an output whatever the number of columns: without any, the separate launches write it."""
    assert said["fc1_no_columns"] == (COMBO, 0)
    assert said["fc1_empty"] == said["fc1_empty_no_columns"] == (OK, 0)


@pytest.mark.parametrize("K", [1024, 1040, 1264, 1280, 2000, 4080, 4096, 4112, 5104, 5120])
def test_lds_of_every_share_of_the_weights(K):
    """Every kernel with a norm in front, at every number of rows and of units per workgroup, one GEMM and three grouped."""
    seen = set()
    for batch in (1, 3):
        wgs = 256 // batch
        for per in range(1, 21):
            for N in (per * wgs * 4, per * wgs * 4 - 5):
                for M in range(1, 5):
                    seen.add(G.check_norm_in_front(batch, M, N, K))
    assert seen == {(1, 1024), (2, 1024), (3, 512), (4, 256), (5, 256)}
