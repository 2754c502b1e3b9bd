"""ResidentTurn (malaga_amd/csrc/resident_turn.hpp): one decode call per device has the resident
launch, until everything it launched has finished, also where the call fails on the way, and
none while other contexts decode batches there."""
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "malaga_amd" / "csrc"

PROGRAM = r"""
#include <cstdio>
#include <stdexcept>
#include <thread>
#include <vector>
#include "resident_turn.hpp"
using mlg::OtherDecode;
using mlg::ResidentTurn;

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

static bool free_for_another(int device) {
    ResidentTurn t(device, [] {});
    const bool got = t.take();
    t.done();
    return got;
}

int main() {
    int drains = 0;
    {   // held until done(), which is told that the stream is drained already
        ResidentTurn a(0, [&] { ++drains; });
        CHECK(free_for_another(0));
        CHECK(a.take());
        CHECK(!free_for_another(0));
        CHECK(free_for_another(1));
        a.done();
        CHECK(free_for_another(0));
    }
    CHECK(drains == 0);
    {   // a call that never had it waits for nothing and frees nothing
        ResidentTurn a(0, [&] { ++drains; });
        CHECK(a.take());
        {
            ResidentTurn b(0, [&] { ++drains; });
            CHECK(!b.take());
        }
        CHECK(drains == 0 && !free_for_another(0));
        a.done();
    }
    // a call that fails: its launches are waited for while it still has the turn
    bool held_while_draining = false;
    try {
        ResidentTurn a(0, [&] {
            ++drains;
            held_while_draining = !free_for_another(0);
        });
        CHECK(a.take());
        throw std::runtime_error("out of memory after the first launches");
    } catch (const std::runtime_error &) {
    }
    CHECK(drains == 1 && held_while_draining && free_for_another(0));
    // none beside the batches of other contexts on the device
    {
        const OtherDecode batch(0);
        {
            const OtherDecode beam(0);
            CHECK(!free_for_another(0) && free_for_another(1));
        }
        CHECK(!free_for_another(0));
    }
    CHECK(free_for_another(0));
    // several threads: never two at once
    std::atomic<int> in{0}, most{0}, got{0};
    std::vector<std::thread> ts;
    for (int i = 0; i < 4; ++i)
        ts.emplace_back([&] {
            for (int k = 0; k < 20000; ++k) {
                ResidentTurn t(2, [&] { in.fetch_sub(1); });
                if (!t.take()) continue;
                const int n = in.fetch_add(1) + 1;
                if (n > most.load()) most.store(n);
                ++got;
                if (k & 1) continue;  // left to the destructor
                in.fetch_sub(1);
                t.done();
            }
        });
    for (auto &t : ts) t.join();
    CHECK(most.load() == 1 && got.load() > 0 && free_for_another(2));
    return 0;
}
"""


def test_turn_is_held_until_the_launches_have_finished(tmp_path):
    src, exe = tmp_path / "turn.cpp", tmp_path / "turn"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
