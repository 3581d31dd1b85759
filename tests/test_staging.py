"""Host work of a prefill shared out over threads (host/staging.h): every task once, groups announced in order, errors thrown."""
import os
import subprocess

import pytest

from util import ROOT

PROGRAM = r'''
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>
#include "model.h"
// the header's atomics take their time after a read: what two reads one after the other may see in between shows
namespace std {
template <typename T> struct slow_atomic : atomic<T> {
    using atomic<T>::atomic;
    using atomic<T>::operator=;
    operator T() const {
        const T v = atomic<T>::load();
        this_thread::sleep_for(chrono::microseconds(SLOW_US));
        return v;
    }
};
}
#define atomic slow_atomic
#include "staging.h"
#undef atomic
namespace vla { int default_cpu_threads() { return 8; } }
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)
int main() {
    for (int threads : {1, 2, 8, 16})
        for (const std::vector<int>& first : {std::vector<int>{0, 1}, {0, 3, 6, 9, 12}, {0, 0, 5}, {0, 500}, {0, 7, 8}})
            for (int rep = 0; rep < 20; ++rep) {
                std::vector<std::atomic<int>> ran(first.back());
                for (auto& r : ran) r = 0;
                std::vector<int> order;
                vla::run_staged(first, threads, [&](int t) { ran[t]++; }, [&](int g) {
                    for (int t = first[g]; t < first[g + 1]; ++t) CHECK(ran[t] == 1);
                    order.push_back(g);
                });
                CHECK(order.size() + 1 == first.size());
                for (size_t g = 0; g < order.size(); ++g) CHECK(order[g] == (int)g);
                for (auto& r : ran) CHECK(r == 1);
            }
    for (int threads : {1, 4}) {  // a task that throws: thrown here, later groups not announced, all threads back
        std::vector<int> order;
        bool thrown = false;
        try {
            vla::run_staged({0, 4, 8, 12}, threads, [](int t) { if (t == 6) throw std::runtime_error("task 6"); }, [&](int g) { order.push_back(g); });
        } catch (const std::runtime_error& e) { thrown = std::string(e.what()) == "task 6"; }
        CHECK(thrown && order.size() <= 1);
    }
    // the group of a task that throws is never announced, however long a look at the state takes
    for (int rep = 0; rep < 40; ++rep) {
        bool announced = false, thrown = false;
        try {
            vla::run_staged({0, 2}, 2, [](int t) {
                if (t == 0) return;
                std::this_thread::sleep_for(std::chrono::microseconds(1200));
                throw std::out_of_range("task 1");
            }, [&](int) { announced = true; });
        } catch (const std::out_of_range&) { thrown = true; }
        CHECK(thrown && !announced);
    }
    {  // no task starts behind an announcement that throws, whose exception comes back as it is
        std::atomic<int> ran{0};
        bool thrown = false;
        try {
            vla::run_staged({0, 1, 2000}, 2, [&](int) { ran++; std::this_thread::sleep_for(std::chrono::microseconds(100)); }, [](int) { throw std::invalid_argument("copy"); });
        } catch (const std::invalid_argument&) { thrown = true; }
        CHECK(thrown && ran < 1000);
    }
    bool thrown = false;  // an announcement that throws
    try { vla::run_staged({0, 4, 8}, 4, [](int) {}, [](int) { throw std::runtime_error("copy"); }); } catch (const std::runtime_error&) { thrown = true; }
    CHECK(thrown);
    CHECK(vla::stage_pieces(0) == 1 && vla::stage_pieces(5 << 20) == 5 && vla::stage_threads(100, false) == 8 && vla::stage_threads(7, false) == 2 && vla::stage_threads(4, false) == 1 && vla::stage_threads(7, true) == 7 && vla::stage_threads(1, true) == 1);
    std::printf("ok\n");
}
'''


@pytest.mark.parametrize("slow_us", [0, 300])
def test_staged_work(tmp_path, slow_us):
    src, exe = str(tmp_path / "staged.cpp"), str(tmp_path / "staged")
    with open(src, "w") as f:
        f.write(PROGRAM)
    host = os.path.join(ROOT, "vla.cpp_amd", "host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-DSLOW_US=%d" % slow_us, "-I", host, "-I", os.path.join(ROOT, "include"), src, "-o", exe, "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr[-2000:]
