"""The traversal's rules that are plain functions of sizes (csrc/trace_rules.h), compiled for the CPU, and the LDS that
the built kernels take by themselves."""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG

SOURCE = r"""
#include "trace_rules.h"
extern "C" {
int pops_entry(uint32_t sp, uint32_t entries) { return rtx::pops_entry(sp, entries); }
// out: grid, lds, first_waves, lean, queues, resident blocks per CU, rays per chunk
void plan(uint32_t block, uint32_t per_cu, uint32_t cus, uint32_t simd, uint32_t lane_bytes, uint32_t start,
          uint32_t chunk, uint32_t n, uint32_t paths, uint32_t* out) {
    const rtx::TraceShape s = {block, per_cu, cus * per_cu, simd, lane_bytes, start};
    const rtx::TracePlan p = rtx::plan_trace(s, chunk, n, paths != 0);
    const uint32_t fixed = p.lean ? 0u : rtx::kOctTableBytes;
    const uint32_t v[] = {p.grid, p.lds, p.first_waves, p.lean, p.queues, rtx::resident_blocks(s, p.lds + fixed),
                          rtx::rays_per_chunk(chunk, n, p.grid * (block / 64), p.first_waves, paths != 0)};
    for (int i = 0; i < 7; ++i) out[i] = v[i];
}
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


def _plan(rules, block, per_cu, cus=256, depth=12, ray=True, start=None, chunk=1, n=0, paths=False):
    waves = block // 64 * per_cu // 4
    out = (ctypes.c_uint32 * 7)()
    rules.plan(block, per_cu, cus, 5 if waves >= 5 else 4 if waves == 4 else 3, 8 * depth + (24 if ray else 0),
               per_cu if start is None else start, chunk, n, int(paths), out)
    return dict(zip(("grid", "lds", "first_waves", "lean", "queues", "resident", "chunk"), out))


def _units(b):  # LDS of a CU is given out in 128 units of 1,280 B
    return -(-b // 1280)


def test_the_tables_and_tasks_take_no_block_from_a_cu(rules):
    """Over every configuration that the library accepts: as many blocks of a launch fit a CU's LDS as would with the
    stack and the world rays alone, and the default launch keeps its table and tasks."""
    for block in (64, 128, 192, 256):
        for per_cu in range(1, 33):
            for depth in range(1, 4097):
                if (8 * depth + 24) * block > 64 * 1024:
                    break
                for ray in (False, True):
                    p = _plan(rules, block, per_cu, depth=depth, ray=ray)
                    waves = block // 64 * per_cu // 4
                    alone = 128 // _units((8 * depth + 24 * ray) * block)
                    want = min(per_cu, 4 * (5 if waves >= 5 else 4 if waves == 4 else 3) // (block // 64), alone)
                    assert p["resident"] == want, (block, per_cu, depth, ray, p)
                    extra = 0 if p["lean"] else 8 * block
                    assert p["lds"] == (8 * depth + 24 * ray) * block + extra
    assert not _plan(rules, 256, 4)["lean"] and not _plan(rules, 64, 16)["lean"]
    assert _plan(rules, 64, 20)["lean"] and _plan(rules, 64, 16, depth=16)["lean"]


@pytest.mark.parametrize("chunk", [1, 64, 128, 4096])
@pytest.mark.parametrize("shape", [(64, 1), (64, 13), (64, 20), (64, 32), (128, 10), (192, 3), (256, 4), (256, 5), (256, 32)])
def test_first_chunks_belong_to_waves_that_start_at_once(rules, shape, chunk):
    """Waves own a first chunk only among the blocks that start at once, by what the chip holds and beside what runs
    already; the first chunks and the queues' chunks cover the rays, and the queues are used exactly where rays are left
    for them."""
    block, per_cu = shape
    cus, wb = 4, block // 64
    for ray in (False, True):
        full = _plan(rules, block, per_cu, cus, ray=ray)
        for n in [1, 2, 63, 64, 65, 777, 64 * cus * per_cu * wb - 1, 64 * cus * per_cu * wb, 64 * cus * per_cu * wb + 1,
                  512 * cus * per_cu * wb, 2 ** 28, 2 ** 32 - 1]:
            for paths in (False, True):
                p = _plan(rules, block, per_cu, cus, ray=ray, chunk=chunk, n=n, paths=paths)
                assert p["first_waves"] <= full["resident"] * cus * wb, (n, p)
                assert 1 <= p["grid"] <= cus * per_cu and p["first_waves"] <= p["grid"] * wb
                assert p["chunk"] >= 1 and bool(p["queues"]) == (p["chunk"] * p["first_waves"] < n)
                for start in (0, 1, per_cu // 2):
                    b = _plan(rules, block, per_cu, cus, ray=ray, chunk=chunk, n=n, paths=paths, start=start)
                    assert b["first_waves"] == min(min(start, full["resident"]) * cus, b["grid"]) * wb
                    assert bool(b["queues"]) == (b["chunk"] * b["first_waves"] < n) and b["lds"] == p["lds"]
        d = _plan(rules, block, per_cu, cus, ray=ray, chunk=chunk, n=0)  # a count that only the device knows
        assert d["queues"] and d["grid"] == cus * per_cu


READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLER = "/opt/rocm/llvm/bin/clang-offload-bundler"
OBJECT = os.path.join(PKG, "_build", "trace.o")


@pytest.mark.skipif(not (os.path.exists(OBJECT) and os.path.exists(READELF) and shutil.which("objcopy")),
                    reason="needs the object file of the build and the ROCm binary tools")
def test_static_lds_of_the_traversal_kernels(tmp_path):
    """What the launch rules count is what the kernels take: the octant table, and nothing in the lean form (five waves
    per SIMD, and the LEAN = true instances of four)."""
    fat, code = str(tmp_path / "fat"), str(tmp_path / "code")
    subprocess.run(["objcopy", "-O", "binary", "--only-section=.hip_fatbin", OBJECT, fat], check=True)
    subprocess.run([BUNDLER, "--unbundle", "--type=o", f"--input={fat}", f"--output={code}",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
    notes = subprocess.run([READELF, "--notes", code], check=True, capture_output=True, text=True).stdout
    seen = {"lean": 0, "full": 0}
    for part in notes.split(".group_segment_fixed_size:")[1:]:
        lds, name = int(part.split()[0]), re.search(r"\.name:\s+(\S+)", part).group(1)
        m = re.search(r"trace_kernel(_w[45])?ILi\dE((?:Lb[01]E)+)", name)
        if not m:
            continue
        lean = m.group(1) == "_w5" or (m.group(1) == "_w4" and m.group(2).endswith("Lb1E"))
        assert lds == (0 if lean else 2048), name
        seen["lean" if lean else "full"] += 1
    assert seen["lean"] > 10 and seen["full"] > 10, seen


@pytest.mark.parametrize("entries", [1, 2, 12, 76, 4096])
def test_a_lane_pops_only_what_its_stack_holds(rules, entries):
    """Two pushes past the end are counted and dropped (a BLAS entry pushes up to two groups): the entries above the end
    are never taken, those below it always."""
    for sp in list(range(min(entries, 80) + 1)) + [entries, entries + 1, entries + 2]:
        assert bool(rules.pops_entry(sp, entries)) == (1 <= sp <= entries), sp
