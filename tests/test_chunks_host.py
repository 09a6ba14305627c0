"""The space of the pool's chunks, driven on host addresses: blocks never overlap,
freed neighbours join, what is held stays near what is out, and a chunk goes
back once nothing of it is out."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "bootcmatchg_amd", "csrc")

HEAD = r"""
#include "chunks.h"
#include <cstdio>
#include <cstdint>
#include <random>
using namespace bcmg;
static char *const SPACE = reinterpret_cast<char *>((uintptr_t)1 << 40);
static size_t at = 0;
/* the pool's way to a block; chunks follow each other without a gap */
static char *take(Chunks &c, size_t n)
{
    char *p = c.take(n);
    if (p) return p;
    const size_t s = c.next_size(n);
    c.add(SPACE + at, s);
    at += s;
    return c.take(n);
}
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
"""


def run_cpp(tmp_path, body):
    src = tmp_path / "t.cpp"
    src.write_text(HEAD + "int main() {\n%s\nreturn 0;\n}\n" % body)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, str(src), "-o",
                    exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "", r.stdout


def test_blocks_do_not_overlap_and_come_back(tmp_path):
    """Random sizes and orders: each block inside one chunk, apart from the
    others, on 256 bytes; all given back, every chunk is whole."""
    run_cpp(tmp_path, r"""
    std::mt19937_64 rng(5);
    for (int round = 0; round < 20; round++) {
        Chunks c;
        std::map<char *, size_t> out;
        for (int step = 0; step < 4000; step++) {
            if (out.empty() || rng() % 5 < 3) {
                const size_t n = std::min<size_t>(Chunks::SUB_MAX,
                                                  ((size_t)256 << (rng() % 16)) + 256 * (rng() % 8));
                char *p = take(c, n);
                CHECK(p && ((uintptr_t)p & 255) == 0);
                auto nx = out.lower_bound(p);
                CHECK(nx == out.end() || p + n <= nx->first);
                if (nx != out.begin()) { auto pv = std::prev(nx); CHECK(pv->first + pv->second <= p); }
                out[p] = n;
            } else {
                auto it = std::next(out.begin(), rng() % out.size());
                c.give(it->first, it->second);
                out.erase(it);
            }
            size_t used = 0;
            for (auto &b : out) used += b.second;
            CHECK(c.total() == c.free() + used);
        }
        while (!out.empty()) {
            auto it = std::next(out.begin(), rng() % out.size());
            c.give(it->first, it->second);
            out.erase(it);
        }
        CHECK(c.free() == c.total());
        c.take_whole();
        CHECK(c.empty() && c.total() == 0 && c.free() == 0);
    }
    """)


def test_freed_neighbours_serve_a_longer_block(tmp_path):
    """Blocks of one size, all freed, hold a block of their sum without another
    chunk; blocks of two chunks that touch are not joined."""
    run_cpp(tmp_path, r"""
    Chunks c;
    std::vector<char *> b;
    for (int k = 0; k < 8; k++) b.push_back(take(c, (size_t)1 << 20));
    CHECK(c.total() == Chunks::CHUNK_MIN);
    for (int k : {1, 6, 3, 0, 7, 2, 5}) CHECK(!c.give(b[k], (size_t)1 << 20));
    char *p = c.take((size_t)4 << 20);
    CHECK(p == b[0]);
    CHECK(!c.give(p, (size_t)4 << 20));
    CHECK(c.give(b[4], (size_t)1 << 20));
    c.add(SPACE + at, Chunks::CHUNK_MIN);   /* right behind the first */
    CHECK(c.take(Chunks::CHUNK_MIN + 256) == nullptr);
    CHECK(c.take_whole().size() == 2);
    """)


def test_what_is_held_stays_near_what_is_out(tmp_path):
    """A set-up's pattern: per level, temporaries of several sizes around the
    level's own arrays, levels shrinking by four; twice in a row, as a second
    operator's. Chunk bytes stay below twice the most that was out plus
    CHUNK_MIN."""
    run_cpp(tmp_path, r"""
    std::mt19937_64 rng(7);
    auto cls = [](size_t n) {
        if (n <= 4096) return (n + 255) & ~(size_t)255;
        const size_t step = (size_t)1 << (61 - __builtin_clzll(n));
        return (n + step - 1) & ~(step - 1);
    };
    Chunks c;
    size_t out = 0, peak = 0;
    auto get = [&](size_t n) { n = cls(n); char *p = take(c, n); out += n; peak = std::max(peak, out);
                               return std::make_pair(p, n); };
    auto back = [&](std::pair<char *, size_t> b) { c.give(b.first, b.second); out -= b.second; };
    for (size_t rows : {226981u, 262144u}) {
        std::vector<std::pair<char *, size_t>> keep;
        for (size_t n = rows; n > 40; n /= 4) {
            for (int s = 0; s < 2; s++) {
                std::vector<std::pair<char *, size_t>> tmp;
                for (int k = 0; k < 14; k++) tmp.push_back(get(n * (4 + rng() % 13) + 4));
                keep.push_back(get(n * 8));
                keep.push_back(get(n * 14 * 4));
                while (!tmp.empty()) {
                    const size_t k = rng() % tmp.size();
                    back(tmp[k]);
                    tmp.erase(tmp.begin() + k);
                }
            }
        }
        CHECK(c.total() <= 2 * peak + Chunks::CHUNK_MIN);
        if (rows == 226981u) for (auto &b : keep) back(b);
    }
    """)


def test_one_block_keeps_its_chunk_only(tmp_path):
    """A large operator's blocks freed beside a small live one: what stays is the
    chunk of the live block, and it serves blocks of any size."""
    run_cpp(tmp_path, r"""
    Chunks c;
    std::vector<char *> big;
    for (int k = 0; k < 6; k++) big.push_back(take(c, (size_t)5 << 20));
    char *live = take(c, 4096);
    for (int k = 0; k < 20; k++) big.push_back(take(c, (size_t)5 << 20));
    for (char *p : big) c.give(p, (size_t)5 << 20);
    const size_t before = c.total();
    CHECK(before >= (size_t)130 << 20);
    c.take_whole();
    CHECK(c.total() <= Chunks::CHUNK_MAX && c.total() - c.free() == 4096);
    CHECK(c.take((size_t)5 << 20) != nullptr);
    (void)live;
    """)
