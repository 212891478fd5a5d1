"""The C entry points of the kernel libraries, the bindings that call them, and what the compiler made of the kernels."""
import ctypes
import glob
import hashlib
import os
import re
import struct

import pytest

from yalis_amd.ops import hip
from yalis_amd.ops.build import CSRC, KERNEL_LIBS, build_dir

# The number that libraries and bindings compare when a library is loaded, and the entry points that it stands for.  Where one of
# these changes, the number goes up (yk_abi_version in runtime.hip, _ABI in ops/hip.py): a library built before would read its
# arguments from the wrong places.
ENTRY_POINTS = (31, "f92e1e712e204564")


def prototypes():
    """name -> (result type, parameter types) of every extern "C" function that is not file-local."""
    found = {}
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        with open(path) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        for result, name, args in re.findall(r'extern "C" ([\w ]+?[\w*] ?\*?)\s*(yk_\w+)\(([^)]*)\)\s*{', text):
            types = []
            for arg in filter(None, (a.strip() for a in args.split(","))):
                if arg != "void":
                    types.append(re.sub(r"\s+", " ", re.sub(r"\w+$", "", arg)).strip())
            found[name] = (result.strip(), tuple(types))
    return found


def kind(c_type):
    if "*" in c_type or c_type == "hipStream_t":
        return ctypes.c_void_p
    return {"int": ctypes.c_int, "float": ctypes.c_float, "size_t": ctypes.c_size_t, "long long": ctypes.c_longlong, "double": ctypes.c_double,
            "int64_t": ctypes.c_int64, "uint64_t": ctypes.c_uint64, "unsigned": ctypes.c_uint, "unsigned long long": ctypes.c_uint64}[c_type]


def test_bindings_match_the_entry_points():
    c = prototypes()
    tables = {**hip._SIGNATURES, **{name: sig for table in hip._LATER_SIGNATURES.values() for name, sig in table.items()}}
    assert len(tables) > 50
    for name, (args, result) in tables.items():
        assert name in c, name
        assert [kind(t) for t in c[name][1]] == list(args), name
        assert kind(c[name][0]) == result, name


def test_the_number_goes_up_with_the_entry_points():
    with open(os.path.join(CSRC, "runtime.hip")) as f:
        number = int(re.search(r"yk_abi_version\(\) { return (\d+); }", f.read()).group(1))
    digest = hashlib.sha256(repr(sorted(prototypes().items())).encode()).hexdigest()[:16]
    assert number == hip._ABI
    assert (number, digest) == ENTRY_POINTS, "entry points changed: raise the number in both places, then note it and the digest here"


# Kernels that keep a few words of a lane in scratch memory, bytes: each measured no slower than with fewer values in flight.
IN_SCRATCH = {"gemm_block_kernelILi256ELi256ELi2ELi2ELi1ELi2ELb1E": 12, "attn_mfma_kernelILi128ELi1ELb0ELi0ELb1E": 8, "sum_norm_vec_kernelIfLb0ELi1ELi2E": 52,
              "streams_norm_vec_kernelILi16ELi4E": 44}


def test_kernels_keep_to_their_registers():
    """A kernel whose values do not fit its registers keeps them in memory, without an error: what the built libraries say of each (the
    metadata of the code objects in them) is nothing, or what is noted above."""
    msgpack = pytest.importorskip("msgpack")
    kernels = {}
    for name in KERNEL_LIBS:
        path = os.path.join(build_dir(), f"libyalis_{name}.so")
        if not os.path.exists(path):
            pytest.skip("no built library")
        with open(path, "rb") as f:
            data = f.read()
        for found in re.finditer(b"\x7fELF\x02\x01\x01\x40", data):  # code objects for the GPU
            at = data.find(b"AMDGPU\0\0", found.start())
            size = struct.unpack("<I", data[at - 8: at - 4])[0]
            for kernel in msgpack.unpackb(data[at + 8: at + 8 + size])["amdhsa.kernels"]:
                kernels[kernel[".name"]] = kernel[".private_segment_fixed_size"]
    assert len(kernels) > 200
    wrong = {k: v for k, v in kernels.items() if v > max((size for name, size in IN_SCRATCH.items() if name in k), default=0)}
    assert not wrong
