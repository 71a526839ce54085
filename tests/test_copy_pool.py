"""CopyPool (hessboost_amd/csrc/host/copy_pool.h): copies of sizes around its
pieces, one after another, from several threads, and with no helpers."""
import os
import shutil
import subprocess
import textwrap

import pytest

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "hessboost_amd", "csrc", "host")

PROGRAM = textwrap.dedent(r"""
    #include <cstdio>
    #include <initializer_list>
    #include <vector>
    #include "copy_pool.h"
    int main() {
        const uint64_t piece = 256 << 10, most = 9 * piece + 77;
        std::vector<unsigned char> src(most + 1);
        for (uint64_t i = 0; i < src.size(); i++) src[i] = (unsigned char)(i * 2654435761u >> 13);
        long bad = 0, seen = 0;
        for (unsigned helpers : {0u, 1u, 7u}) {
            hbr::CopyPool pool(helpers);
            std::mutex one_at_a_time;
            auto work = [&](unsigned seed) {
                std::vector<unsigned char> dst(most + 1);
                for (int round = 0; round < 40; round++)
                    for (uint64_t n : {uint64_t(0), uint64_t(1), piece - 1, piece, piece + 1, 2 * piece, most - seed}) {
                        std::memset(dst.data(), 0x5a ^ src[n], n + 1);
                        std::lock_guard<std::mutex> lock(one_at_a_time);
                        pool.copy(dst.data(), src.data() + seed % 2, n);
                        bad += std::memcmp(dst.data(), src.data() + seed % 2, n) != 0;
                        bad += dst[n] != (unsigned char)(0x5a ^ src[n]);
                        seen++;
                    }
            };
            std::vector<std::thread> callers;
            for (unsigned t = 0; t < 3; t++) callers.emplace_back(work, t);
            for (auto &t : callers) t.join();
        }
        std::printf("%ld %ld\n", seen, bad);
        return 0;
    }
""")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_byte_is_copied_and_none_beside_it(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I", HEADER, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=100).stdout
    seen, bad = map(int, out.split())
    assert seen == 3 * 3 * 40 * 7 and bad == 0
