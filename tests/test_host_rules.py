"""Sizes and bookkeeping of the backend's host side (csrc/fbhip_host.h), compiled
with a plain C++ compiler: what a kernel writes fits what is allocated for it."""

from __future__ import annotations

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "ferrisboost_amd", "csrc")


def run_cpp(tmp_path, body: str) -> None:
    """Compiles and runs a main() of `body`, where CHECK(x) fails the test."""
    src = tmp_path / "t.cpp"
    src.write_text('#include "fbhip_host.h"\n#include <cstdio>\n#include <cstdlib>\n'
                   "#include <initializer_list>\n#include <random>\n#include <vector>\n"
                   "using namespace fbh;\n"
                   "#define CHECK(x) do { if (!(x)) { std::printf(\"%d: %s\\n\", __LINE__, #x); "
                   "std::exit(1); } } while (0)\n"
                   f"int main() {{\n{body}\nreturn 0;\n}}\n")
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-fsanitize=undefined", "-I", CSRC,
                    str(src), "-o", str(exe)], check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True)
    assert got.returncode == 0, got.stdout + got.stderr


def test_reduction_scratch_holds_every_pass(tmp_path):
    """quantile_partials_kernel writes QUANTILE_BLOCKS pairs at any row count, the
    bounds and quantisation passes a pair a block and the pair these reduce to."""
    run_cpp(tmp_path, """
    for (uint64_t n : {1ull, 255ull, 256ull, 257ull, 5000ull, 65024ull, 65025ull, 65536ull,
                       2097152ull, 4294967295ull}) {
        const uint32_t b = reduction_blocks(n);
        CHECK(b >= 1 && b <= 8192);
        CHECK(reduction_words(b) >= 2ull * b + 2);
        CHECK(reduction_words(b) >= 2ull * QUANTILE_BLOCKS);
    }""")


def test_a_failed_regrow_leaves_no_pointer(tmp_path):
    """A kept table whose larger replacement cannot be allocated: the next request,
    also one that the old size would have served, allocates again."""
    run_cpp(tmp_path, """
    std::vector<int *> freed;
    int blocks[3];
    int *p = &blocks[0];
    uint64_t bytes = 64, taken = 0;
    const auto release = [&](int *q) { freed.push_back(q); };
    bool failed = false;
    try {
        regrow(p, bytes, 128, release, [&](uint64_t) -> int * { throw 1; });
    } catch (int) {
        failed = true;
    }
    CHECK(failed && p == nullptr && bytes == 0);
    CHECK(freed.size() == 1 && freed[0] == &blocks[0]);
    const auto take = [&](uint64_t b) { taken = b; return &blocks[1]; };
    regrow(p, bytes, 64, release, take);
    CHECK(p == &blocks[1] && bytes == 64 && taken == 64);
    taken = 0;
    regrow(p, bytes, 32, release, take);
    CHECK(p == &blocks[1] && bytes == 64 && taken == 0);
    CHECK(freed.size() == 2 && freed[1] == nullptr);""")


def test_sketch_bound_covers_every_layout(tmp_path):
    """What the sketch's buffers are said to need covers the layout of any batch
    counts: all features full, mixed with missing values, or empty."""
    run_cpp(tmp_path, """
    std::mt19937_64 r(7);
    for (int it = 0; it < 4000; it++) {
        const uint32_t n = 1 + r() % (it % 4 ? 700 : 5000);
        const uint64_t limit = 16ull << r() % 11;
        const uint64_t most = 1 + r() % (it % 3 ? 40 : 3000);
        const uint32_t kind = it % 5;
        std::vector<uint64_t> m(n);
        for (auto &v : m)
            v = kind == 0 ? most : kind == 1 ? r() % (most + 1) : kind == 2 ? r() % 2
                : kind == 3 ? (r() % 2 ? most : 1) : (r() % 5 ? most : 0);
        for (auto &v : m) v = std::min(v, most);
        const SketchPlan p = sketch_plan(m, limit);
        const SketchSlots b = sketch_slots_most(most, n, limit);
        CHECK(p.slots.a <= b.a && p.slots.b <= b.b && p.slots.t <= b.t);
        CHECK(p.slots.all_a <= b.all_a && p.slots.all_t <= b.all_t);
        CHECK(p.groups.front().j0 == 0 && p.groups.back().j1 == n);
        for (size_t g = 0; g + 1 < p.groups.size(); g++) {
            CHECK(p.groups[g].j1 == p.groups[g + 1].j0);
            CHECK(p.abase[p.groups[g].j1] - p.abase[p.groups[g].j0] <= p.slots.a);
        }
    }""")


def test_sketch_bytes_count_the_groups_buffers():
    """400k x 2000 at 256 bins: 11 GB of summaries in groups of features, not the 33
    that all features' would take at once; and no less than the values alone."""
    from ferrisboost_amd import _native as N

    got = N.hip().fbh_sketch_device_bytes(400_000, 2000, 256, None)
    assert 11e9 < got < 16e9
    # few features share one group: every batch's entries, merged and final ones
    m = -(-1_000_000 // 4096)
    got = N.hip().fbh_sketch_device_bytes(1_000_000, 10, 256, None)
    least = 4 * 1_000_000 * 10 + 10 * 16 * 4096 * (m + 2 * ((m + 1) // 2) + 1)
    assert least < got < 2 * least


def test_the_integration_recipe_builds_every_source():
    """INTEGRATION.md's build step names the sources of the library, with the flags that
    its results depend on."""
    import re

    from ferrisboost_amd import build

    with open(os.path.join(os.path.dirname(os.path.dirname(CSRC)), "INTEGRATION.md")) as f:
        recipe = re.search(r"// build.rs.*?```", f.read(), flags=re.S).group(0)
    assert sorted(re.findall(r"\{src\}/(\w+\.hip)", recipe)) == sorted(build.BACKEND_SRCS)
    flags = [f for f in build.HIP_FLAGS if not f.startswith("-W")]
    assert all(f'"{f}"' in recipe for f in flags)
