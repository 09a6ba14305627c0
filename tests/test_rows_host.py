"""Which row a group of lanes takes, at the sizes where 32-bit products wrap."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bootcmatchg_amd", "csrc")


def run_cpp(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text('#include "rows.h"\n#include <algorithm>\n#include <cstdio>\n#include <initializer_list>\nusing namespace bcmg;\n'
                   "int main() {\n%s\nreturn 0;\n}\n" % body)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o",
                    exe], check=True)
    return subprocess.run([exe], check=True, capture_output=True, text=True).stdout


def test_rows_of_lane_groups(tmp_path):
    """Every G up to the block's lanes, the last rows of 2^31 lanes and beyond:
    the row is (block * 256 + thread) / G in 64 bits."""
    out = run_cpp(tmp_path, """
    for (int G = 1; G <= ROW_BS; G *= 2)
        for (unsigned long long lanes : {1ull << 10, (1ull << 31) - 1, 1ull << 31,
                                         (1ull << 31) + 300, (1ull << 32) - 256})
            for (unsigned t : {0u, 1u, 63u, 64u, 255u}) {
                const unsigned block = (unsigned)(lanes / ROW_BS);
                const unsigned long long want = ((unsigned long long)block * ROW_BS + t) / G;
                if (want > 0x7fffffffull) continue;
                const int got = group_row(block, t, G);
                if (got < 0 || (unsigned long long)got != want)
                    std::printf("G %d lanes %llu t %u: %d\\n", G, lanes, t, got);
            }
    """)
    assert out == ""
