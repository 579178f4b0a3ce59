"""The extension module's source (csrc/host.cpp): what cannot be seen from a call's result."""
import os
import re
import struct

import pytest

SOURCE = os.path.join(os.path.dirname(__file__), "..", "triton_int_amd", "csrc", "host.cpp")


def test_every_launch_and_allocation_runs_without_the_interpreters_lock():
    """A launch may wait for the device (a full queue, a workspace that grows): ctypes releases the lock around a call, and so
    does every function here.  Python objects are read before."""
    src = re.sub(r"//.*", "", open(SOURCE).read())
    bodies = re.split(r"\nPyObject\* (?=\w+\(PyObject\*, PyObject\* const\* v)", src)[1:]
    assert len(bodies) == len(re.findall(r"TI_METHOD\(\w+\)", src)) - 1  # the macro's own definition
    for body in bodies:
        name = body.split("(")[0]
        parts = body.split("const NoGil unlocked;")
        assert len(parts) == 2, name
        depth, end = 1, 0
        while depth:  # the block that holds the lock's release
            depth += {"{": 1, "}": -1}.get(parts[1][end], 0)
            end += 1
        unlocked, rest = parts[1][:end], parts[0] + parts[1][end:]
        assert re.search(r"\bti_\w+\(", unlocked), name
        assert not re.search(r"\bti_\w+\(|c\.empty\(", rest), f"{name}: launches or allocates under the lock"
        assert not re.search(r"\bPy\w+|THP\w+|\bv\[|\b(integer|number|flag|scale|vector|tensor)\(", unlocked), f"{name}: reads a Python object without the lock"


@pytest.mark.parametrize("name", ["_host.so", "_layer_host.so"])
def test_no_thread_local_storage(name):
    """A module with thread-local storage of its own, loaded after torch and HIP, puts every thread-local access of those on the
    slow path (glibc before 2.39)."""
    path = os.path.join(os.path.dirname(SOURCE), "..", name)
    with open(path, "rb") as f:
        elf = f.read()
    table, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    types = [struct.unpack_from("<I", elf, table + i * size)[0] for i in range(count)]
    assert 1 in types and 7 not in types  # PT_LOAD, PT_TLS


def test_the_layer_reads_held_tensors_without_the_interpreters_lock():
    """Another thread may replace what a Python tensor object holds while the layer launches: every tensor that is read without the
    lock is the copy that the call holds."""
    src = re.sub(r"//.*", "", open(os.path.join(os.path.dirname(SOURCE), "host_layer.cpp")).read())
    assert re.search(r"const Tensor& tensor\([^)]*\) \{[^}]*all\.push_back\(::tensor\(o, dev, type\)\);\s*return all\.back\(\);", src)
    before, after = src.split("const NoGil unlocked;")
    unlocked = after[:after.index("need(rc == TI_OK)")]
    assert not re.search(r"\bPy\w+|THP\w+|\bv\[", unlocked)
    used = set(re.findall(r"\bm?ptr\((\w+)\)", unlocked)) | set(re.findall(r"(\w+)\.sizes\(\)", unlocked))
    own = set(re.findall(r"Tensor (\w+)(?: = c\.empty|;)", src))
    assert src.count("held.tensor(PyTuple_GET_ITEM(v[2], ") == 2  # the caches
    for name in used - own:
        assert f"const Tensor& {name} = held.tensor(" in before, name
    # references into the vector stay valid: it never grows past its inline storage
    room = int(re.search(r"SmallVector<Tensor, (\d+)> all;", src).group(1))
    linears, norms = 6, 2
    caches = 2
    assert 1 + 4 + linears * 4 + norms * 2 + caches <= room and f"need(all.size() < {room})" in src
