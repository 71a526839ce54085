"""repeat_add (hessboost_amd/csrc/host/repeat_add.h) against the chain of
additions it stands for, bit for bit: the terms 1/n of a label mean, terms
that lie halfway between two spacings of some binade, powers of two."""
import os
import shutil
import subprocess
import textwrap

import pytest

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "hessboost_amd", "csrc", "host")

PROGRAM = textwrap.dedent(r"""
    #include <cstdio>
    #include <cstring>
    #include <initializer_list>
    #include "repeat_add.h"
    int main() {
        long bad = 0, seen = 0;
        auto check = [&](double c, uint64_t most, uint64_t every) {
            double s = 0.0;
            for (uint64_t k = 0; k <= most; k++) {
                if (k % every == 0 || k == most || k < 70) {
                    const double got = hbr::repeat_add(c, k);
                    seen++;
                    bad += std::memcmp(&got, &s, 8) != 0;
                }
                s += c;
            }
        };
        for (uint64_t n : {1ull, 2ull, 3ull, 7ull, 10ull, 100ull, 4000ull, 99999ull, 1000003ull, 10500000ull, 16777217ull})
            check(1.0 / (double)n, n < 3000000 ? n : 3000000, n < 2000 ? 1 : 997);
        for (int b = 1; b < 53; b++) {
            check(1.0 + std::ldexp(1.0, -b), 100000, 61);
            check(1.0 + std::ldexp(1.0, -b) + std::ldexp(1.0, -52), 100000, 61);
            check(std::ldexp(3.0, -b), 100000, 61);
        }
        std::printf("%ld %ld\n", seen, bad);
        return 0;
    }
""")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_repeated_addition_equals_the_chain(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", HEADER, "-o", str(exe), str(src)], check=True)
    seen, bad = map(int, subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split())
    assert seen > 100_000 and bad == 0
