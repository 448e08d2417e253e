"""What rtx_sync says of the flags that kernels raise (csrc/device_errors.h), compiled for the CPU."""
import ctypes
import os
import subprocess

import pytest

from conftest import PKG

SOURCE = r"""
#include "device_errors.h"
extern "C" int code(uint32_t flags) { return rtx::device_error(flags).code; }
extern "C" const char* text(uint32_t flags) { return rtx::device_error(flags).text; }
extern "C" uint32_t flag(int i) {
    const uint32_t f[] = {rtx::kErrStackOverflow, rtx::kErrSortTimeout, rtx::kErrBadAs, rtx::kErrCollapseTimeout};
    return f[i];
}
"""


@pytest.fixture(scope="module")
def errors(tmp_path_factory):
    d = tmp_path_factory.mktemp("errors")
    src, lib = d / "errors.cpp", d / "errors.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-I", os.path.join(PKG, "csrc"), str(src),
                    "-o", str(lib)], check=True)
    e = ctypes.CDLL(str(lib))
    e.text.restype = ctypes.c_char_p
    return e


def test_each_flag_names_its_own_cause(errors):
    overflow, sort, bad, collapse = (errors.flag(i) for i in range(4))
    assert [overflow, sort, bad, collapse] == [1, 2, 4, 8]
    assert errors.code(0) == 0
    assert errors.code(overflow) == -1001 and b"stack overflow" in errors.text(overflow)
    assert errors.code(sort) == -4 and b"sort" in errors.text(sort)
    assert errors.code(bad) == -1002 and b"invalid acceleration structure" in errors.text(bad)
    # a wait that ran out is no fault of the geometry
    assert errors.code(collapse) == -4 and b"collapse queue" in errors.text(collapse)
    assert errors.code(overflow | sort | bad | collapse) == -1001 and errors.code(bad | collapse) == -4
