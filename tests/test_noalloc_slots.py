"""The slots of sgemm_launch_noalloc's scratch (csrc/noalloc_slots.hpp) against a
model of streams, without a GPU: random calls, captures, forks and closed
streams, and for every two launches that share a slot one that waits for the
other, or a replay that the caller orders."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amdgpu-arch-gemm_amd", "csrc")

MODEL = r"""
#include "noalloc_slots.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <set>
#include <vector>
using namespace noalloc;

constexpr int kNamed = 99;        // the per-thread name
struct Launch { int first, end; uint64_t capture; };

struct Model {
    typedef int Stream;
    int now = 1;                                  // the calling thread
    std::map<int, std::set<int>> before;          // launches that later work of a stream follows
    std::map<int, uint64_t> in_capture;
    std::map<int, std::set<int>> nodes;           // of the capture, the same
    std::set<int> marks[kSlots], ended;
    std::vector<Launch> launches;
    int orders = 0;
    int begins_capture = 0;                       // a stream that does while it is recorded on
    uint64_t captures = 0;

    int real(int s) const { return s == kNamed ? 1000 + now : s; }
    bool capturing(int s, uint64_t* id) {
        auto it = in_capture.find(real(s));
        if (it == in_capture.end()) return false;
        *id = it->second;
        return true;
    }
    bool per_thread(int s) { return s == kNamed; }
    uint64_t thread() { return (uint64_t)now; }
    int order(int b, int a) {
        ++orders;
        uint64_t x = 0, y = 0;
        if (b == begins_capture) { in_capture[real(b)] = ++captures; nodes[real(b)].clear(); begins_capture = 0; }
        const bool cb = capturing(b, &x), ca = capturing(a, &y);
        if (cb && ca && x == y) { nodes[real(a)].insert(nodes[real(b)].begin(), nodes[real(b)].end()); return 0; }
        if (cb) return kBusy;
        if (ca) die("a captured call waits for eager work");
        before[real(a)].insert(before[real(b)].begin(), before[real(b)].end());
        return 0;
    }
    int mark(int q, int s) { marks[q] = before[real(s)]; return 0; }
    int wait(int q, int s) { before[real(s)].insert(marks[q].begin(), marks[q].end()); return 0; }
    int sync(int s) { ended.insert(before[real(s)].begin(), before[real(s)].end()); return 0; }

    void die(const char* what) { std::printf("%s\n", what); std::exit(1); }
    void launch(int s, int first, int end) {
        uint64_t id = 0;
        const bool captured = capturing(s, &id);
        std::set<int>& seen = captured ? nodes[real(s)] : before[real(s)];
        for (int p = 0; p < (int)launches.size(); ++p) {
            const Launch& o = launches[p];
            if (o.capture != id || o.first >= end || first >= o.end || ended.count(p) || seen.count(p)) continue;
            std::printf("launch %d on stream %d (slots %d..%d) does not wait for launch %d (slots %d..%d)%s\n",
                        (int)launches.size(), real(s), first, end - 1, p, o.first, o.end - 1, captured ? ", captured" : "");
            std::exit(1);
        }
        seen.insert((int)launches.size());
        launches.push_back({first, end, id});
    }
};

int main(int argc, char** argv) {
    auto on = [&](const char* what) { for (int i = 1; i < argc; ++i) if (!std::strcmp(argv[i], what)) return true; return false; };
    int busy = 0, all_calls = 0, runs = 0;
    for (unsigned seed = 0; seed < 3000; ++seed) {
        std::mt19937 rng(seed);
        Model m;
        Slots<Model> slots;
        auto call = [&](int s, bool all) {
            int first = 0;
            bool fresh = false, captured = false;
            const int e = slots.take(m, s, all, &first, &fresh, &captured);
            ++runs;
            all_calls += all;
            if (e == kBusy) {
                ++busy;
                if (m.in_capture.empty()) m.die("refused without a capture");
                return;
            }
            if (e) m.die("error");
            m.launch(s, first, all ? kSlots : first + 1);
            slots.done(m, s, all, first);
        };
        const int streams = 2 + (int)(rng() % 11);
        for (int step = 0; step < 120; ++step) {
            m.now = 1 + (int)(rng() % 2);
            const int s = on("per_thread") && rng() % 4 == 0 ? kNamed : 1 + (int)(rng() % streams);
            const unsigned what = rng() % 20;
            if (what < 12) {
                if (on("captures_race") && rng() % 8 == 0) {
                    const int other = 1 + (int)(rng() % streams);
                    uint64_t id = 0;
                    if (other != s && !m.capturing(other, &id)) m.begins_capture = other;
                }
                call(s, rng() % 4 == 0);
                m.begins_capture = 0;
            } else if (what < 14 && on("captures")) {
                uint64_t id = 0;
                // without "eager_before" only idle streams capture: their eager work has ended
                if (!m.capturing(s, &id)) {
                    if (!on("eager_before")) m.sync(s);
                    m.in_capture[m.real(s)] = ++m.captures;
                    m.nodes[m.real(s)].clear();
                }
            } else if (what < 16 && on("forks")) {
                uint64_t id = 0, other = 0;
                const int t = 1 + (int)(rng() % streams);
                if (m.capturing(s, &id) && !m.capturing(t, &other) && t != s) {
                    if (!on("eager_before")) m.sync(t);
                    m.in_capture[m.real(t)] = id;
                    m.nodes[m.real(t)] = m.nodes[m.real(s)];
                }
            } else if (what < 18) {
                uint64_t id = 0;
                if (m.capturing(s, &id))
                    for (auto it = m.in_capture.begin(); it != m.in_capture.end();) it = it->second == id ? m.in_capture.erase(it) : std::next(it);
            } else if (on("leaves") && s != kNamed) {
                uint64_t id = 0;
                if (!m.capturing(s, &id)) {
                    slots.forget(m, s);          // one of several handles leaves the stream ...
                    if (rng() % 2) m.before[m.real(s)].clear();   // ... or it is destroyed and its name comes back
                }
            }
        }
    }
    // side by side: eight streams' small calls wait for nobody
    Model m;
    Slots<Model> slots;
    for (int round = 0; round < 3; ++round)
        for (int s = 1; s <= kSlots; ++s) {
            int first = 0;
            bool fresh = false, captured = false;
            if (slots.take(m, s, false, &first, &fresh, &captured) || fresh != (round == 0) || m.orders) m.die("not side by side");
        }
    std::printf("%d calls, %d of all slots, %d without scratch\n", runs, all_calls, busy);
    return 0;
}
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = tmp_path_factory.mktemp("slots")
    (d / "model.cpp").write_text(MODEL)
    exe = d / "model"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=undefined", "-I", CSRC, str(d / "model.cpp"),
                    "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("events", [
    [],
    ["captures"],                                     # a captured call leaves the eager owners alone
    ["captures", "forks"],                            # two branches of one capture meet in a slot
    ["captures", "eager_before"],                     # an owner captures while its eager calls still run
    ["captures", "captures_race"],                    # ... or begins to while it is recorded on
    ["leaves"],                                       # a stream shared by two handles, one of which leaves it
    ["per_thread"],                                   # one name, a stream in every thread
    ["captures", "forks", "eager_before", "captures_race", "leaves", "per_thread"],
])
def test_launches_that_share_a_slot_are_ordered(model, events):
    ret = subprocess.run([model] + events, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=120)
    out = ret.stdout.decode()
    print(out)
    assert ret.returncode == 0, out
