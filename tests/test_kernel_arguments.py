"""The argument blocks of the built GEMM kernels: what one variant needs does not lengthen every launch's."""
import os
import re
import subprocess
import tempfile

import pytest
import yaml

from tests import isa_lint
from triton_int_amd import _lib

READELF = os.path.join(os.path.dirname(isa_lint.OBJDUMP), "llvm-readelf")


@pytest.mark.skipif(not (os.path.exists(isa_lint.OBJDUMP) and os.path.exists(READELF)), reason="ROCm LLVM tools not installed")
def test_only_the_kernels_with_a_norm_in_front_take_its_arguments():
    sizes = {}
    with tempfile.TemporaryDirectory() as tmp:
        for obj in isa_lint.extract_code_objects(_lib.LIB_PATH, tmp):
            notes = subprocess.run([READELF, "--notes", obj], check=True, capture_output=True, text=True).stdout
            for text in re.findall(r"^\s*---\n(.*?)^\.\.\.", notes, re.S | re.M):
                for kernel in yaml.safe_load(text).get("amdhsa.kernels", []):
                    if "gemm_" in kernel[".name"] and kernel[".args"]:
                        sizes[kernel[".name"]] = kernel[".args"][0][".size"]
    # two kinds of norm, five shares of the weights, two lengths of K
    norm = {n: s for n, s in sizes.items() if re.search(r"gemm_rowpieces_kernelILi16ELi[1-5]ELi\d+ELi[12]ELi[45]EE", n)}
    plain = {s for n, s in sizes.items() if n not in norm}
    assert len(norm) == 20 and len(sizes) > 100
    assert plain == {280} and set(norm.values()) == {360}
