"""The kept graphs' cache (tomos_amd/csrc/shared_cache.hpp) with objects that
count themselves, compiled for the host: an entry that another call's insert
evicts lives on until the last call that found it lets go."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cassert>
#include <thread>
#include "shared_cache.hpp"
static std::atomic<int> alive{0};
struct Exec {
    int use = 1;
    Exec() { ++alive; }
    ~Exec() { use = 0; --alive; }
};
int main() {
    tomos_hip::SharedCache<int, Exec> c(8);
    for (int k = 0; k < 8; ++k) c.insert(k, std::make_shared<Exec>());
    std::shared_ptr<Exec> held = c.find(0);
    assert(held && c.find(7) && !c.find(8) && alive == 8);
    for (int k = 8; k < 16; ++k) c.insert(k, std::make_shared<Exec>());
    assert(!c.find(0) && !c.find(7) && c.find(8) && alive == 9 && held->use == 1);  // evicted, but held
    held.reset();
    assert(alive == 8);
    std::thread t[4];
    for (int i = 0; i < 4; ++i)
        t[i] = std::thread([&c, i] {
            for (int k = 0; k < 20000; ++k) {
                std::shared_ptr<Exec> e = c.find(k % 24);
                if (!e) c.insert(k % 24, e = std::make_shared<Exec>());
                assert(e->use == 1);
            }
        });
    for (auto& x : t) x.join();
    assert(alive == 8);
}
"""


def test_evicted_entry_lives_until_released(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text("#include <atomic>\n" + SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-fsanitize=address,undefined", "-I",
                    os.path.join(ROOT, "tomos_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True, timeout=60)
