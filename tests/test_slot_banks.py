"""The slot banks through which a replica's workgroups exchange partial sums
(remc_slots.h, compiled for the host): for every sequence of windows and moves
that exchange everything, some or nothing, no order in which the members get
along leaves one waiting for a value that another has overwritten.  The model
takes every interleaving; with a count that advances at windows without an
exchange it must find one that gets stuck."""
import os
import subprocess

import pytest

from conftest import REPO

MODEL = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>
#include "remc_slots.h"

// What the members do one after the other: a window of `slots` slots, `still` of
// them without a partial (a large move: one slot that exchanges).
struct Event { int slots, still; };
static const Event kinds[] = {{1, 0}, {3, 1}, {1, 1}, {4, 4}};
static bool count_all; // the planted mistake

static unsigned next(unsigned n, const Event &e)
{
    return count_all ? n + 1u : remc_exchanges_after_window(n, e.slots, e.still);
}

struct Member { unsigned n; int at, polls; };
struct World {
    std::vector<Member> m;
    std::vector<int> bank; // 2 x members: the event whose partial is held
    bool operator<(const World &o) const
    {
        for (size_t k = 0; k < m.size(); ++k) {
            if (m[k].at != o.m[k].at) return m[k].at < o.m[k].at;
            if (m[k].polls != o.m[k].polls) return m[k].polls < o.m[k].polls;
        }
        return bank < o.bank;
    }
};

// true if some interleaving gets stuck
static bool stuck(const World &w, const std::vector<Event> &ev, std::set<World> &seen)
{
    if (!seen.insert(w).second) return false;
    const int M = (int)w.m.size();
    bool moved = false, done = true;
    for (int k = 0; k < M; ++k) {
        const Member &a = w.m[k];
        if (a.at == (int)ev.size()) continue;
        done = false;
        const Event &e = ev[a.at];
        World v = w;
        Member &b = v.m[k];
        if (!a.polls && e.still < e.slots) { // publishes, then waits
            v.bank[(a.n & 1u) * M + k] = a.at;
            b.polls = 1;
        } else {
            bool all = true; // a poll succeeds where it finds every member's partial
            if (a.polls)
                for (int q = 0; q < M; ++q) all = all && w.bank[(a.n & 1u) * M + q] == a.at;
            if (!all) continue;
            b.polls = 0;
            b.n = next(a.n, e);
            ++b.at;
        }
        moved = true;
        if (stuck(v, ev, seen)) return true;
    }
    return !done && !moved;
}

int main(int argc, char **argv)
{
    const int members = std::atoi(argv[1]), length = std::atoi(argv[2]);
    count_all = std::atoi(argv[3]) != 0;
    long sequences = 1, bad = 0;
    for (int k = 0; k < length; ++k) sequences *= 4;
    for (long s = 0; s < sequences; ++s) {
        std::vector<Event> ev;
        long c = s;
        for (int k = 0; k < length; ++k, c /= 4) ev.push_back(kinds[c % 4]);
        World w;
        w.m.assign(members, Member{0u, 0, 0});
        w.bank.assign(2 * members, -1);
        std::set<World> seen;
        bad += stuck(w, ev, seen);
    }
    std::printf("%ld %ld\n", sequences, bad);
    return 0;
}
"""


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("slots"))
    src, exe = os.path.join(d, "m.cpp"), os.path.join(d, "m")
    with open(src, "w") as f:
        f.write(MODEL)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas",
                    "-I", os.path.join(REPO, "remcdockingsimulator_amd", "csrc"), src, "-o", exe], check=True)

    def run(members, length, count_all=False):
        out = subprocess.run([exe, str(members), str(length), "1" if count_all else "0"], capture_output=True, text=True,
                             check=True).stdout.split()
        return int(out[0]), int(out[1])

    return run


@pytest.mark.parametrize("members,length", [(2, 6), (3, 5), (4, 4)])
def test_no_interleaving_gets_stuck(model, members, length):
    sequences, bad = model(members, length)
    assert sequences == 4 ** length and bad == 0


@pytest.mark.parametrize("members,length", [(2, 3), (3, 4)])
def test_the_model_finds_a_bank_reused_without_an_exchange(model, members, length):
    assert model(members, length, count_all=True)[1] > 0
