"""CPU test of the growth of the launcher's temporary buffers (csrc/grown_buffer.h)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include "%s"
#include <cstdio>
#include <cstdlib>
#include <vector>
#define CHECK(x) do { if (!(x)) { printf("line %%d: %%s\\n", __LINE__, #x); return 1; } } while (0)
int main() {
    size_t room = 1000, asked = 0;
    int calls = 0;
    auto alloc = [&](void **p, size_t bytes) -> int {
        calls++;
        asked = bytes;
        if (bytes > room) return 2;
        *p = malloc(bytes);
        return 0;
    };
    float *buf = nullptr;
    size_t have = 0;
    std::vector<void *> retired;
    CHECK(rf::grow_buffer(buf, have, 2000, retired, alloc) == 2 && !buf && have == 0 && retired.empty());
    CHECK(rf::grow_buffer(buf, have, 400, retired, alloc) == 0 && buf && have == 400 && retired.empty());
    float *const first = buf;
    // no memory for the large plan's sums, time and again: the small plan's stay where they are
    for (int i = 0; i < 3; i++) {
        CHECK(rf::grow_buffer(buf, have, 5000, retired, alloc) == 2);
        CHECK(buf == first && have == 400 && retired.empty());
        const int before = calls;
        CHECK(rf::grow_buffer(buf, have, 400, retired, alloc) == 0 && buf == first && calls == before);
    }
    room = 100000;
    CHECK(rf::grow_buffer(buf, have, 401, retired, alloc) == 0 && asked == 600 && have == 600);
    CHECK(buf != first && retired.size() == 1 && retired[0] == first);
    CHECK(rf::grow_buffer(buf, have, 5000, retired, alloc) == 0 && asked == 5000 && have == 5000 && retired.size() == 2);
    // a plan that can do without: a size that was refused is asked for once in 64 calls, a smaller one at once
    rf::RefusedGrowth r;
    CHECK(r.ask(9000));
    r.answer(9000, false);
    for (int round = 0; round < 3; round++) {
        for (int i = 0; i < 63; i++) CHECK(!r.ask(round == 1 ? 20000 : 9000));
        CHECK(r.ask(9000));
        r.answer(9000, false);
    }
    CHECK(r.ask(8999));
    r.answer(8999, false);
    CHECK(!r.ask(9000) && r.ask(8998));
    for (int i = 0; i < 62; i++) CHECK(!r.ask(9000));
    CHECK(r.ask(9000));
    r.answer(9000, true);
    CHECK(r.ask(9000) && r.ask(1u << 30));
    return 0;
}
"""


def test_a_growth_that_fails_leaves_the_buffer_in_use(tmp_path):
    src, exe = tmp_path / "grow.cpp", str(tmp_path / "grow")
    src.write_text(PROGRAM % os.path.join(ROOT, "radeonflow_kernels_amd", "csrc", "grown_buffer.h"))
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-o", exe, str(src)], check=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
