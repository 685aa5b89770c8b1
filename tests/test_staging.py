"""The host staging of a plan (staging.hpp), compiled for the CPU with an
allocator that can refuse."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "staging.hpp"
static bool refuse;
static int held;
struct Fake {
    static void *get(size_t bytes) {
        if (refuse) return nullptr;
        held++;
        return malloc(bytes);
    }
    static void put(void *q) {
        held--;
        free(q);
    }
};
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main() {
    const size_t n = 1003;
    for (int r = 0; r < 2; r++) {
        refuse = r;
        mtk::Staging<Fake> s;
        s.alloc(n);
        CHECK(s.p && s.pinned == !refuse && held == !refuse);
        CHECK((size_t)s.p % sizeof(double) == 0);
        for (size_t i = 0; i < n; i++) s.p[i] = (float)i;
        for (size_t i = 0; i < n; i++) CHECK(s.p[i] == (float)i);
        refuse = !refuse;  // allocated again, the other way
        s.alloc(2 * n);
        CHECK(s.p && s.pinned == !refuse && held == !refuse);
        s.p[2 * n - 1] = 1;
    }
    CHECK(held == 0);
    return 0;
}
"""


def test_plain_memory_where_none_can_be_pinned(tmp_path):
    """A plan whose staging cannot be pinned gets ordinary memory, as all host
    calls had before there was pinned staging; each kind is given back."""
    (tmp_path / "s.cpp").write_text(SRC)
    exe = str(tmp_path / "s")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    "-I" + os.path.join(ROOT, "maos_amd", "csrc", "hip"), str(tmp_path / "s.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
