"""The traversal's rules that are plain functions of sizes (csrc/trace_rules.h), compiled for the CPU."""
import ctypes
import os
import subprocess

import pytest

from conftest import PKG

SOURCE = r"""
#include "trace_rules.h"
extern "C" {
int pops_entry(uint32_t sp, uint32_t entries) { return rtx::pops_entry(sp, entries); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, lib = d / "rules.cpp", d / "rules.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-I", os.path.join(PKG, "csrc"), str(src),
                    "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("entries", [1, 2, 12, 76, 4096])
def test_a_lane_pops_only_what_its_stack_holds(rules, entries):
    """Two pushes past the end are counted and dropped (a BLAS entry pushes up to two groups): the entries above the end
    are never taken, those below it always."""
    for sp in list(range(min(entries, 80) + 1)) + [entries, entries + 1, entries + 2]:
        assert bool(rules.pops_entry(sp, entries)) == (1 <= sp <= entries), sp
