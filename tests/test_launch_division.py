"""How launches divide their work (vk_cinematic_amd/csrc/spg_launch.h), on the
CPU: the header is compiled with the host compiler and driven over the edges
of its ranges, above all counts near 2^32, which no GPU test can hold."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "vk_cinematic_amd", "csrc")


def _run(tmp_path, body):
    """Compiles `body` (statements of main; return 0 = passed) and runs it."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text('#include "spg_launch.h"\n#include <stdio.h>\nusing namespace spg;\n'
                   'int main()\n{\n' + body + '\n    return 0;\n}\n')
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-D__host__=", "-D__device__=",
                    "-I", CSRC, "-o", str(exe), str(src)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    return r.stdout


@pytest.mark.parametrize("rays", [0, 1, 63, 64, 65, 255, 257, 16383, 16385, 2560 * 128 + 1,
                                  2**32 - 129, 2**32 - 128, 2**32 - 127, 2**32 - 64,
                                  2**32 - 1])
@pytest.mark.parametrize("waves", [1, 8, 2560, 8192])
def test_chunks_cover_the_rays_once(tmp_path, rays, waves):
    """The chunks are non-empty, follow one another and end at the last ray;
    none is larger than the limit (in 64 bits, so that a wrapped end shows)."""
    _run(tmp_path, f"""
    const uint64_t n = {rays}ull;
    const uint32_t want = walk_waves((uint32_t)n), grid = {waves}u;
    const WorkChunks w((uint32_t)n, want < grid ? want : grid, 128u);
    uint64_t at = 0;
    for (uint32_t j = 0; j < w.chunks; ++j)
    {{
        const uint64_t lo = w.begin(j), hi = w.end(j);
        if (lo != at || hi <= lo || hi > n || hi - lo > 128)
        {{
            printf("chunk %u of %u: [%llu, %llu) after %llu\\n", j, w.chunks,
                   (unsigned long long)lo, (unsigned long long)hi, (unsigned long long)at);
            return 1;
        }}
        at = hi;
    }}
    if (at != n) {{ printf("ends at %llu\\n", (unsigned long long)at); return 1; }}""")


@pytest.mark.parametrize("most", [2048, 65535])   # tone map; accumulation
@pytest.mark.parametrize("items", [1, 255, 256, 257, 2048 * 256 + 3, 2**32 - 65535 * 256,
                                   2**32 - 2048 * 256 + 1, 2**32 - 256, 2**32 - 1])
def test_strided_loops_end_and_cover_the_items_once(tmp_path, items, most):
    """The grid has a block for every 256 items up to the limit, and threads
    at both ends of it (and where the count's remainder falls) step through
    their own residue once and stop."""
    _run(tmp_path, f"""
    const uint64_t n = {items}ull;
    const uint32_t grid = stride_blocks((uint32_t)n, 256, {most}u);
    const uint64_t want = (n + 255) / 256 < {most}ull ? (n + 255) / 256 : {most}ull;
    if (grid != want) {{ printf("grid %u\\n", grid); return 1; }}
    const uint64_t step = grid * 256ull;
    const uint64_t at[] = {{0, 1, step / 2, n % step, (n + step - 1) % step, step - 1}};
    for (uint64_t first : at)
    {{
        uint64_t expect = first;
        for (uint32_t i = (uint32_t)first; i < (uint32_t)n;
             i = stride_next(i, (uint32_t)step, (uint32_t)n), expect += step)
            if (i != expect)
            {{
                printf("thread %llu: item %u after %llu\\n", (unsigned long long)first, i,
                       (unsigned long long)(expect - step));
                return 1;
            }}
        if (expect < n) {{ printf("thread %llu ends early\\n", (unsigned long long)first); return 1; }}
    }}""")


def test_tuned_refill_thresholds_differ_from_the_default(tmp_path):
    """Every threshold the batch tuner times is another launch than the
    default (0 stands for it): valid, distinct and not the default's value."""
    _run(tmp_path, """
    for (uint32_t a : kRefillSweep)
    {
        int same = a == kSceneRefill ? 1 : 0;
        for (uint32_t b : kRefillSweep) same += a == b ? 1 : 0;
        if (a < 1 || a > 64 || same != 1) { printf("threshold %u\\n", a); return 1; }
    }""")


def test_spill_area_begins_where_the_shortest_lds_stack_ends(tmp_path):
    """Entry i of a walk's stack spills at row i - kMinShortStack at the
    lowest: no row below the first one used, none used below the first."""
    _run(tmp_path, """
    const int shortest = kSceneShortStack < kMeshShortStack ? kSceneShortStack : kMeshShortStack;
    if (kMinShortStack != shortest)
    {
        printf("area from entry %d, stacks spill from %d\\n", kMinShortStack, shortest);
        return 1;
    }""")


@pytest.mark.parametrize("words", [6, 7])   # a scene query's ray and its result
def test_record_offsets_do_not_wrap(tmp_path, words):
    """The last record below 2^32 words, the first above it and the last ray."""
    _run(tmp_path, f"""
    const uint64_t at[] = {{0, 1, 613566756, 613566757, 715827882, 715827883, 4294967295}};
    for (uint64_t i : at)
        if (record_at((uint32_t)i, {words}u) != i * {words}ull) return 1;""")
