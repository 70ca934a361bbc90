"""The blocks' helping of the plain model calls, on the CPU: a model of its counters and
postings in C++, with the kernel's own test of when a helper leaves (plain_help.hpp).

Blocks start as room falls free, in any order, take steps in any order, post groups of
segments, take segments of each other's and wait as the kernel does; the host's base may
differ from the counters (a launch that ran but was reported as failed leaves it
behind).  Every call has to end, with every segment run once.  Equality with the number
of blocks as the helpers' first test, which a base that is behind steps over, is run
as well, to show that the model does tell the two apart."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MODEL = r'''
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
#include "plain_help.hpp"
struct Block { int state = 0, groups = 0, held = -1, own = 0; };  // 0 waits for room, 1 own work, 2 owner waits, 3 helps, 4 gone
int main(int argc, char** argv) {
    const bool equality = argv[1][0] == 'e';
    const uint32_t blocks = atoi(argv[2]), room = atoi(argv[3]), drift = (uint32_t)atoll(argv[4]);
    std::mt19937 rng(atoi(argv[5]));
    const uint32_t base0 = rng();
    uint32_t started = base0, ended = base0;
    const uint32_t base = base0 + drift;
    std::vector<Block> b(blocks);
    std::vector<int> avail(blocks, 0), finished(blocks, 0), total(blocks, 0);
    long run = 0, posted = 0;
    uint32_t running = 0, gone = 0;
    for (auto& x : b) x.groups = rng() % 3;
    for (long step = 0; step < 400000; step++) {
        if (gone == blocks) { printf("ended %ld %ld\n", run, posted); return 0; }
        const uint32_t i = rng() % blocks;
        Block& x = b[i];
        auto claim = [&](uint32_t s) { if (avail[s] <= 0) return false; avail[s]--; x.held = (int)s; return true; };
        if (x.state == 0) { if (running < room) { running++; started++; x.state = 1; } continue; }
        if (x.state == 4) continue;
        if (x.held >= 0) { finished[x.held]++; run++; x.held = -1; continue; }
        if (x.state == 1) {
            if (!x.groups) { ended++; x.state = 3; continue; }
            x.groups--;
            total[i] = 1 + rng() % 8; posted += total[i]; finished[i] = 0; avail[i] = total[i]; x.state = 2;
        } else if (x.state == 2) {
            if (claim(i)) continue;
            if (finished[i] == total[i]) x.state = 1;
        } else {
            const uint32_t s = rng() % blocks;
            if (claim(s)) continue;
            const bool leave = equality ? ended - base == blocks || started - base < blocks
                                        : nmlmc::helper_leaves(started, ended, base, blocks);
            if (leave) { x.state = 4; running--; gone++; }
        }
    }
    printf("waits %ld %ld\n", run, posted);
    return 0;
}
'''


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    d = tmp_path_factory.mktemp("help")
    src, exe = d / "model.cpp", d / "model"
    src.write_text(MODEL)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "nested-risk-mlmc_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)

    def run(test, blocks, room, drift, seed):
        return subprocess.run([str(exe), test, str(blocks), str(room), str(drift), str(seed)], check=True, timeout=60,
                              capture_output=True, text=True).stdout.split()
    return run


@pytest.mark.parametrize("blocks, room", [(1, 1), (2, 1), (7, 7), (7, 3), (40, 64), (40, 9)])
def test_every_call_ends(model, blocks, room):
    for drift in (0, -1, -3, -blocks, -2 * blocks - 1, 1, blocks, 1 << 31, -(1 << 31)):
        for seed in range(4):
            word, run, posted = model("kernel", blocks, room, drift, seed)
            assert word == "ended" and run == posted, (drift, seed)


def test_equality_would_wait(model):
    """A base behind by one, all blocks running: they wait for a count already passed."""
    assert any(model("equality", 7, 7, -1, seed)[0] == "waits" for seed in range(8))
    assert all(model("equality", 7, 7, 0, seed)[0] == "ended" for seed in range(8))
