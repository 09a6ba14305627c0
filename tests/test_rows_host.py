"""Which row a group of lanes takes, at the sizes where 32-bit products wrap."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bootcmatchg_amd", "csrc")


def run_cpp(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text('#include "rows.h"\n#include "slab_plan.h"\n#include <algorithm>\n#include <cstdio>\n#include <initializer_list>\nusing namespace bcmg;\n'
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


def test_grids_of_lane_groups(tmp_path):
    """A launch stays below 2^32 lanes and its steps reach every row once: a
    wavefront a row at 2^26 rows and more, a lane a row at 2^31 - 1."""
    out = run_cpp(tmp_path, """
    for (int G = 1; G <= 64; G *= 2)
        for (int n : {1, 3, 4, 255, 256, 257, 1 << 25, (1 << 25) + 1, 1 << 26, (1 << 26) + 5,
                      (1 << 30) + 7, 0x7fffffff}) {
            const unsigned long long blocks = group_blocks(n, G);
            const long long step = row_step((unsigned)blocks, G);
            if (blocks == 0 || blocks * ROW_BS >= 1ull << 32) std::printf("grid %d %d\\n", G, n);
            if (step < n && blocks != 1u << 23) std::printf("short %d %d\\n", G, n);
            if (step - n >= ROW_BS / G) std::printf("empty blocks %d %d\\n", G, n);
        }
    """)
    assert out == ""


def test_blocks_inside_the_operator(tmp_path):
    """A block is inside where every row's neighbours are: against 64 bits, with
    offsets and rows up to 2^31."""
    out = run_cpp(tmp_path, """
    for (long long n : {512ll, 4097ll, (1ll << 30) + 9, (3ll << 29) + 11, 0x7fffffffll})
        for (long long lo : {-n + 1, -5ll, 0ll, 3ll})
            for (long long hi : {-2ll, 0ll, 7ll, n / 2, n - 1})
                for (long long r0 : {0ll, 256ll, n / 512 * 256, n / 256 * 256 - 256}) {
                    if (hi < lo || r0 < 0 || r0 >= n) continue;
                    const bool want = r0 + lo >= 0 && r0 + 256 + hi <= n && r0 + 256 <= n;
                    if (inner_rows((int)n, (int)lo, (int)hi).holds((int)r0, 256) != want)
                        std::printf("n %lld lo %lld hi %lld r0 %lld\\n", n, lo, hi, r0);
                }
    """)
    assert out == ""


def test_slabs_fit_their_workgroup(tmp_path):
    """The rows of a slab with its halo, for bands up to 2^31 and many sweeps:
    what is taken has the cells that four a lane hold, the rest is refused."""
    out = run_cpp(tmp_path, """
    for (int band : {0, 1, 8, 63, 64, 2048, 1 << 20, 1 << 28, (1 << 29) + 1, 1 << 30, 0x7ffffffe})
        for (int sweeps : {2, 3, 4, 16, 1000, 100000})
            for (int gpr : {1, 2, 3, 16})
                for (int n : {1, 4096, 1 << 20, 0x7fffffff}) {
                    const IlSlab p = il_slab_fit(n, band, gpr, sweeps);
                    const double least = (16.0 + 2.0 * band * sweeps) * gpr;
                    const double cells = (p.L + 2.0 * band * sweeps) * gpr;
                    const bool fits = p.rpt >= 1 && p.rpt <= 4 && cells <= p.rpt * SLAB_BS &&
                                      cells > (p.rpt - 1) * SLAB_BS && p.us > 0;
                    if (least <= 4 * SLAB_BS ? !fits : p.rpt != 0)
                        std::printf("band %d sweeps %d gpr %d n %d: L %d rpt %d\\n", band, sweeps,
                                    gpr, n, p.L, p.rpt);
                }
    """)
    assert out == ""
