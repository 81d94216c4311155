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
