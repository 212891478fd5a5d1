"""The C entry points of the kernel libraries and the bindings that call them."""
import ctypes
import glob
import hashlib
import os
import re

from yalis_amd.ops import hip
from yalis_amd.ops.build import CSRC

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
