"""The ctypes binding against the header: without a declared list of arguments a call passes pointers as 32-bit integers."""
import ctypes
import os
import re

import pytest

from randumb_amd import _lib

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "randumb_hip.h")
PLAIN = {"int64_t": ctypes.c_int64, "int32_t": ctypes.c_int32, "uint32_t": ctypes.c_uint32, "int": ctypes.c_int, "float": ctypes.c_float}


def _declared():
    text = re.sub(r"/\*.*?\*/", " ", open(HEADER).read(), flags=re.S)
    return {name: (ret.strip(), [a.strip() for a in args.split(",")] if args.strip() != "void" else [])
            for ret, name, args in re.findall(r"^((?:const )?\w+ \*?)\s*(rdb_\w+)\(([^)]*)\);", text, flags=re.M)}


def test_the_header_declares_what_is_exported():
    assert sorted(_declared()) == sorted(_lib.EXPORTS)


@pytest.mark.parametrize("name", _lib.EXPORTS)
def test_arguments_and_result_as_declared(name):
    ret, args = _declared()[name]
    f = getattr(_lib.load(), name)
    assert f.restype is (ctypes.c_char_p if "*" in ret else PLAIN[ret])
    assert f.argtypes is not None and len(f.argtypes) == len(args), (f.argtypes, args)
    for bound, arg in zip(f.argtypes, args):
        if "*" in arg:
            assert bound is ctypes.c_void_p or issubclass(bound, ctypes._Pointer), (arg, bound)
        else:
            assert bound is PLAIN[arg.split()[0]], (arg, bound)
