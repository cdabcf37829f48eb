"""Which repeated calls get a captured graph (host code only): every key of a
cycle that fits the table comes back to its count, however long the cycle; a
failed capture waits; graphs are bounded and give way only to keys that last;
captures that are not replayed end."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cstdio>
#include <iterator>
#include <set>
#include "mpm_recurring.hpp"
using namespace mpm;
using R = RecurringCalls<int, int*>;
static int bad = 0, box[1 << 16];
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); bad++; } } while (0)
struct Run {
    R r;
    std::multiset<int*> live;
    int replays = 0, captures = 0, destroyed = 0;
    void step(int key) {
        auto& e = r.call(key);
        if (e.graph) { CHECK(live.count(e.graph) == 1); replays++; return; }
        auto gone = [&](int* g) { CHECK(live.erase(g) == 1); destroyed++; };
        if (r.due(e, gone)) {
            int* g = box + captures++ % (1 << 16);
            live.insert(g);
            r.keep(e, g);
        }
        CHECK(r.graphs() == live.size() && r.graphs() <= R::GRAPHS && r.keys() <= R::KEYS);
    }
};
int main() {
    // cycles of a steady state: each key is captured at its fifth call, the
    // first GRAPHS of them, and none is given up
    for (int len : {1, 4, 63, 64, 65, 100, 226, 511, 512}) {
        Run u;
        const int rounds = 40, kept = len < int(R::GRAPHS) ? len : int(R::GRAPHS);
        for (int k = 0; k < rounds * len; ++k) u.step(k % len);
        CHECK(u.captures == kept && u.destroyed == 0 && u.replays == kept * (rounds - 5));
        int n = 0;
        u.r.clear([&](int*) { n++; });
        CHECK(n == kept && u.r.graphs() == 0 && u.r.keys() == 0);
    }
    {  // the same between keys that come once: they never push the cycle out
        Run u;
        for (int k = 0; k < 20000; ++k) { u.step(k % 100); u.step(1000 + k); }
        CHECK(u.captures == int(R::GRAPHS) && u.replays > 64 * 190);
    }
    {  // keys that last fewer than REPLACE_CALLS calls: captured while there is room, then eager
        Run u;
        for (int k = 0; k < 400 * 20; ++k) u.step(k / 20);
        CHECK(u.captures == int(R::GRAPHS) && u.destroyed == 0);
    }
    {  // keys that last replace graphs idle for more calls than any counted cycle
        Run u;
        for (int k = 0; k < 400 * 200; ++k) u.step(k / 200);
        CHECK(u.captures > 300 && u.destroyed == u.captures - int(R::GRAPHS) && u.replays > 400 * 150);
    }
    {  // cycles beyond the table are left alone
        Run u;
        for (int k = 0; k < 30000; ++k) u.step(k % 3000);
        CHECK(u.captures == 0);
    }
    // everything is dropped every `len` calls of a cycle of 4 keys, as where
    // particles are loaded anew: captures that do not pay end, others go on
    for (int len : {24, 30, 60, 100, 400}) {
        Run u;
        for (int ep = 0; ep < 2000; ++ep) {
            for (int k = 0; k < len; ++k) u.step(k % 4);
            u.r.clear([&](int* g) { CHECK(u.live.erase(g) == 1); });
        }
        CHECK(u.captures <= int(R::GRAPHS) + u.replays / int(R::CAPTURE_COST));
        if (len >= 100) CHECK(u.captures == 4 * 2000 && u.replays == 2000 * (len - 20));
    }
    {  // a failed capture waits for its calls again
        R r;
        int asked = 0;
        for (int k = 0; k < 25; ++k)
            if (r.due(r.call(7), [](int*) {})) { asked++; r.failed(7); }
        CHECK(asked == 5 && r.graphs() == 0);
        for (int k = 0; k < 5000; ++k)
            if (r.due(r.call(7), [](int*) {})) { asked++; r.failed(7); }
        CHECK(asked == int(R::GRAPHS));  // and not for ever
    }
    return bad != 0;
}
"""


def test_counts_and_graphs_of_repeated_calls(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "molla_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
