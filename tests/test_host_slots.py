"""The rules of the pinned slots that copies to the host go through
(csrc/host_slots.hpp, plain C++, compiled here with g++): a first small copy
pins nothing, slots are earned by what is copied, bounded, kept for later
copies, given back with the last owner, and counted right when pinning fails
or many threads take them at once."""
import subprocess

from oxidizedmlx_amd import build

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include "host_slots.hpp"
using mlxhip::HostSlots;
static std::atomic<int> pinned{0}, most{0}, refuse{0};
static char* pin() {
    if (refuse.load()) return nullptr;
    const int n = ++pinned;
    for (int m = most.load(); n > m && !most.compare_exchange_weak(m, n);) {}
    return static_cast<char*>(std::malloc(16));
}
static void unpin(char* p) { --pinned; std::free(p); }
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s (pinned %d)\n", __LINE__, #c, pinned.load()); return 1; } } while (0)
int main() {
    constexpr size_t E = HostSlots::EARN, MIB = 1 << 20;
    HostSlots h(pin, unpin);
    char* s[HostSlots::MAX];
    // An owner per small copy: nothing is pinned, copy after copy, until one slot is earned.
    size_t copied = 0;
    for (; copied + MIB < E; copied += MIB) {
        h.retain();
        CHECK(h.take(MIB, 1, 1, s) == 0 && pinned == 0);
        h.release();
    }
    h.retain();
    CHECK(h.take(MIB, 1, 1, s) == 1 && pinned == 1);
    h.give(s, 1);
    h.release();
    CHECK(pinned == 1);  // within KEPT
    // A copy of several chunks pins nothing before it can have what it needs.
    h.retain();
    CHECK(h.take(2 * E, 8, 4, s) == 0 && pinned == 1);
    CHECK(h.take(E, 8, 4, s) == 4 && pinned == 4);
    h.give(s, 4);
    h.release();
    CHECK(pinned == HostSlots::KEPT);
    // Further ones need as much from one owner's time: not 16 MiB a job.
    for (int i = 0; i < 20; ++i) {
        h.retain();
        CHECK(h.take(2 * E, 8, 4, s) == 4 && pinned == 4);
        h.give(s, 4);
        h.release();
    }
    h.retain();
    CHECK(h.take(MIB, 8, 4, s) == 4 && pinned == 4);
    // Kept ones in use: another copy at the same time has none of them.
    char* t[HostSlots::MAX];
    CHECK(h.take(MIB, 8, 4, t) == 0 && h.take(MIB, 1, 1, t) == 0 && pinned == 4);
    h.give(s, 4);
    // A large copy earns its slots at once; pinning may fail.
    refuse = 1;
    CHECK(h.take(8 * E, 8, 5, s) == 0 && pinned == 4);
    CHECK(h.take(MIB, 8, 4, s) == 4 && pinned == 4);
    h.give(s, 4);
    refuse = 0;
    CHECK(h.take(MIB, 8, 4, s) == 8 && pinned == 8);
    h.give(s, 8);
    // The last owner goes while a copy of its own is still out.
    CHECK(h.take(MIB, 8, 4, s) == 8);
    h.release();
    CHECK(pinned == 8);
    h.give(s, 8);
    CHECK(pinned == HostSlots::KEPT);
    h.retain();
    CHECK(h.take(MIB, 8, 4, s) == 4 && pinned == 4);  // beyond KEPT to be earned again
    h.give(s, 4);
    // Threads with owners of their own.
    std::vector<std::thread> th;
    for (int i = 0; i < 6; ++i)
        th.emplace_back([&h] {
            for (int k = 0; k < 3000; ++k) {
                char* q[8];
                h.retain();
                const int n = h.take(8 * MIB, 8, 4, q);
                for (int j = 0; j < n; ++j) q[j][0] = (char)j;
                if (n) h.give(q, n);
                h.release();
            }
        });
    for (auto& x : th) x.join();
    CHECK(most <= HostSlots::MAX);
    h.release();
    CHECK(pinned == HostSlots::KEPT);
    std::puts("ok");
    return 0;
}
"""


def test_slots_are_earned_bounded_and_given_back(tmp_path):
    (tmp_path / "p.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", build.CSRC, "-o", str(tmp_path / "p"), str(tmp_path / "p.cpp"), "-pthread"],
                   check=True)
    r = subprocess.run([str(tmp_path / "p")], capture_output=True, text=True, timeout=120)
    assert r.stdout.strip() == "ok" and r.returncode == 0, r.stdout + r.stderr
