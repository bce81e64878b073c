"""The pool of idle memory (csrc/pool.cpp) on the CPU, with stubs that record what is freed:
the bound, the order in which blocks go, their age, and that a program can have it all back."""
import os
import subprocess

import pytest

from conftest import PKG, ROOT

MAIN = r"""
#include <chrono>
static double now_s = 0.0;
namespace std { namespace chrono {
struct test_clock {                        // stands in for the steady clock: a time that the test sets
    using rep = double;
    using period = std::ratio<1>;
    using duration = std::chrono::duration<double>;
    using time_point = std::chrono::time_point<test_clock>;
    static time_point now() { return time_point(duration(now_s)); }
};
} }
#define steady_clock test_clock
#include "pool.cpp"
#include <cstdio>
#include <cstring>
using namespace dtc;
static std::vector<size_t> freed, freed_host;
extern "C" hipError_t hipFree(void* p) { freed.push_back((size_t)p); return hipSuccess; }
extern "C" hipError_t hipHostFree(void* p) { freed_host.push_back((size_t)p); return hipSuccess; }
static void* at(size_t v) { return (void*)v; }
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
constexpr size_t MB = (size_t)1 << 20;

static int bound() {                       // 16 GiB in blocks of 256 MiB: 16 stay, the oldest go first
    for (size_t k = 1; k <= 64; ++k) {
        pool_put(at(k), 256 * MB, 0);
        CHECK(freed.size() == (k > 16 ? k - 16 : 0));
    }
    for (size_t k = 0; k < freed.size(); ++k) CHECK(freed[k] == k + 1);
    // unlike sizes: every block that goes leaves room, none is lost or freed twice
    size_t held = 16 * 256;
    for (size_t k = 100; k < 160; ++k) { pool_put(at(k), (k - 60) * MB, 0); held += k - 60; }
    for (size_t f : freed) if (f > 48) held -= f < 100 ? 256 : f - 60;
    CHECK(held * MB <= POOL_BYTES);
    std::vector<size_t> s = freed;
    for (size_t a = 0; a < s.size(); ++a) for (size_t b = 0; b < a; ++b) CHECK(s[a] != s[b]);
    return 0;
}
static int large() {                       // a block over a quarter of the bound is not kept
    pool_put(at(1), POOL_BYTES / 4 + 4096, 0);
    CHECK(freed.size() == 1 && freed[0] == 1);
    pool_put(at(2), POOL_BYTES / 4, 0);
    CHECK(freed.size() == 1 && pool_take(POOL_BYTES / 4, 0) == at(2) && !pool_take(POOL_BYTES / 4, 0));
    return 0;
}
static int age() {                         // gone at the next use after POOL_SECONDS
    pool_put(at(1), 4096, 0);
    now_s = POOL_SECONDS - 1.0;
    pool_put(at(2), 8192, 0);
    CHECK(freed.empty());
    now_s = POOL_SECONDS + 1.0;
    CHECK(!pool_take(1 << 20, 0) && freed.size() == 1 && freed[0] == 1);
    CHECK(pool_take(8192, 0) == at(2));
    return 0;
}
static int device() {                      // a block is handed out on its own GPU, at its own size
    pool_put(at(1), 4096, 0);
    CHECK(!pool_take(4096, 1) && !pool_take(8192, 0) && pool_take(4096, 0) == at(1));
    return 0;
}
static int release() {                     // everything idle, device and page-locked, each once
    for (size_t k = 1; k <= 9; ++k) pool_put(at(k), k * MB, (int)(k % 2));
    for (size_t k = 1; k <= 3; ++k) pool_put_pinned(at(100 + k), 4096);
    CHECK(pool_take(5 * MB, 1) == at(5));
    CHECK(dtc_release_memory() == DTC_OK);
    CHECK(freed.size() == 8 && freed_host.size() == 3);
    for (size_t f : freed) CHECK(f != 5);
    for (size_t k = 1; k <= 9; ++k) CHECK(!pool_take(k * MB, (int)(k % 2)));
    CHECK(!pool_take_pinned(4096) && dtc_release_memory() == DTC_OK && freed.size() == 8);
    pool_put(at(5), 5 * MB, 1);            // and it goes on as before
    CHECK(pool_take(5 * MB, 1) == at(5));
    return 0;
}
static int words() {                       // page-locked words: a fixed number stays whatever their sizes, the oldest go first
    const size_t N = POOL_PINNED;
    for (size_t k = 1; k <= N; ++k) pool_put_pinned(at(k), 4096 * (k + 1));       // sizes that never come back
    CHECK(freed_host.empty());
    pool_put_pinned(at(N + 1), 4096);
    CHECK(freed_host.size() == 1 && freed_host[0] == 1);
    CHECK(pool_take_pinned(4096) == at(N + 1) && !pool_take_pinned(4096));        // the next call of that size finds it
    pool_put_pinned(at(N + 2), 4096);
    pool_put_pinned(at(N + 3), ((size_t)1 << 20) + 4096);                         // larger than 1 MiB: not kept
    CHECK(freed_host.size() == 2 && freed_host[1] == N + 3);
    return 0;
}
static int words_age() {
    pool_put_pinned(at(1), 4096);
    now_s = POOL_SECONDS - 1.0;
    pool_put_pinned(at(2), 8192);
    CHECK(freed_host.empty());
    now_s = POOL_SECONDS + 1.0;
    CHECK(pool_take_pinned(8192) == at(2) && freed_host.size() == 1 && freed_host[0] == 1);
    return 0;
}
int main(int, char** argv) {
    const std::string t = argv[1];
    return t == "bound" ? bound() : t == "large" ? large() : t == "age" ? age() : t == "device" ? device()
         : t == "release" ? release() : t == "words" ? words() : t == "words_age" ? words_age() : 2;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("pool")
    (d / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I",
                    os.path.join(PKG, "csrc"), "-I", os.path.join(ROOT, "include"), str(d / "m.cpp"), "-o", str(d / "m")],
                   check=True)
    return str(d / "m")


@pytest.mark.parametrize("what", ["bound", "large", "age", "device", "release", "words", "words_age"])
def test_pool(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_release_without_a_device():
    """Nothing is kept: the entry point makes no call to the runtime."""
    import dtc_amd as dtc
    dtc.release_memory()
