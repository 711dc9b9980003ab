"""The decisions of the one-pass form's workgroups (fused_walk.hpp, the code
the kernel runs), compiled for the host and run over many solves of which only
some workgroups are there, one after the other or their steps mixed at random:
every tile of those that are there is solved, with no other's help."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MODEL = r'''
#include <cstdio>
#include <random>
#include <vector>
#include "fused_walk.hpp"
using namespace tprh;

struct Solve {
    int bps, nsys, total;
    std::vector<char> tile, group, result, x;  // published words, stored answers
    std::vector<int> link;
    bool spoiled = false;  // published from inputs that an answer had taken the place of (x stored over d)
    int ngroups() const { return bps / kFusedGroup; }
    Solve(int b, int s) : bps(b), nsys(s), total(b * s), tile(total), group(total), result(total), x(total), link(total) {}
};

// What a workgroup sees of one system (fused_look's x).
struct Words {
    Solve& s;
    int base;
    unsigned long long tiles(int g, int) const {
        unsigned long long m = 0;
        for (int k = 0; k < kFusedGroup; k++) m |= (unsigned long long)!s.tile[base + g * kFusedGroup + k] << k;
        return m;
    }
    unsigned long long groups(int) const {
        unsigned long long m = 0;
        for (int g = 0; g < s.ngroups(); g++) m |= (unsigned long long)!s.group[base + g] << g;
        return m;
    }
    void publish(int g) { s.group[base + g] = 1; }
};

struct Group {  // a workgroup
    int own, stride, tile, kind = kFusedOwn, missing = -1, step = 0;
    bool fresh = false, seen = false;  // what was loaded were inputs; the tile was published after that
    FusedWalk walk;
    Group(int first, int st) : own(first), stride(st), tile(first) {}
    bool done(const Solve& s) const { return tile < 0 || tile >= s.total; }

    // One step: loading the tile, asking whether it is published, publishing
    // it, or looking and going on.  patient: an own tile's first wait goes on
    // rather than give up.
    void run(Solve& s, int limit, bool patient) {
        if (step < 3) {
            if (step == 0) fresh = !s.x[tile];
            if (step == 1) seen = s.tile[tile];
            if (step == 2 && fused_publishes(kind, seen)) {
                s.tile[tile] = 1;
                if (!fresh) s.spoiled = true;
            }
            step++;
            return;
        }
        const int ti = tile % s.bps, base = tile - ti;
        Words w{s, base};
        bool ok;
        if (s.bps <= kFusedGroup) {
            unsigned long long m = w.tiles(0, 0) & ((1ull << s.bps) - 1);
            ok = m == 0;
            if (!ok) missing = base + fused_pick(m, ti);
        } else if (ti % kFusedGroup != 0 && kind == kFusedOwn) {
            ok = s.result[tile];
        } else {
            const int g = ti / kFusedGroup, lost = kind != kFusedOwn ? fused_look(w, ti, 0) : -1;
            ok = lost < 0 && w.tiles(g, 0) == 0;
            if (ok) {
                w.publish(g);
                ok = w.groups(0) == 0;
            }
            missing = base + lost;
            if (ok) for (int k = 0; k < kFusedGroup; k++) s.result[tile / kFusedGroup * kFusedGroup + k] = 1;
        }
        if (!ok && kind == kFusedOwn && patient) return;
        step = 0;
        if (!ok && kind == kFusedAgain && walk.lost(limit)) ok = true;  // x becomes NaN
        if (ok && kind != kFusedHelp) s.x[tile] = 1;
        const int next = own + stride < s.total ? own + stride : -1;
        const FusedTask t = walk.next(tile, kind, ok, missing, next, limit, [&](int k) -> int& { return s.link[k]; });
        tile = t.tile;
        kind = t.kind;
        if (kind == kFusedOwn) own = tile;
    }
};

// The workgroups `there` of `stride`, and no other: in turn, or with their
// steps mixed (seed > 0).  Returns the most tasks one took beyond its own
// tiles, or -1 if a tile of theirs is left or was published from what x had
// been stored over.
int solve(int bps, int nsys, int stride, const std::vector<int>& there, int limit, unsigned seed) {
    Solve s(bps, nsys);
    for (int& k : s.link) k = -2;
    std::vector<Group> g;
    for (int k : there) g.emplace_back(k, stride);
    int most = 0;
    long long steps = 0;
    if (seed == 0) {
        for (Group& w : g)
            while (!w.done(s)) w.run(s, limit, false), steps++;
    } else {
        std::mt19937 rng(seed);
        std::vector<int> live;
        for (int i = 0; i < (int)g.size(); i++)
            if (!g[i].done(s)) live.push_back(i);
        while (!live.empty()) {
            const int at = (int)(rng() % live.size());
            Group& w = g[live[at]];
            for (int k = (int)(rng() % 4); k >= 0 && !w.done(s); k--) w.run(s, limit, rng() % 3 != 0), steps++;
            if (w.done(s)) live[at] = live.back(), live.pop_back();
        }
    }
    if (s.spoiled) return -1;
    for (Group& w : g) most = w.walk.tries > most ? w.walk.tries : most;
    for (int k : there)
        for (int t = k; t < s.total; t += stride)
            if (!s.x[t]) return -1;
    return most;
}

std::vector<int> range(int a, int b, int by = 1) {
    std::vector<int> v;
    for (int k = a; k < b; k += by) v.push_back(k);
    return v;
}
'''


def run(tmp_path, main):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(MODEL + main)
    p = subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-I" + os.path.join(ROOT, "tpr_amd", "csrc"), str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


@pytest.mark.parametrize("seeds", [[0], [1, 2, 3], [4, 5, 6]])
def test_every_tile_of_those_there_is_solved(tmp_path, seeds):
    out = run(tmp_path, r'''
int main() {
    int n = 0;
    for (unsigned seed : {%s})
        for (int bps : {8, 16, 32, 128, 256, 512})
            for (int nsys : {1, 3}) {
                const int total = bps * nsys;
                for (int stride : {total, bps, 16, 5, bps / 2 + 3}) {
                    const int G = stride;
                    const std::vector<std::vector<int>> sets = {
                        range(0, 1), range(G - 1, G), range(0, (G + 1) / 2), range(G / 2, G), range(0, G, 2),
                        range(G > 16 ? 16 : 0, G), range(0, G > 16 ? G - 16 : G), range(0, G, 17), range(0, G)};
                    for (const auto& v : sets) {
                        if (solve(bps, nsys, stride, v, 1 << 14, seed) < 0) {
                            printf("tiles left: %%d tiles, %%d systems, stride %%d, %%d there, seed %%u\n", bps, nsys,
                                   stride, (int)v.size(), seed);
                            return 1;
                        }
                        n++;
                    }
                }
            }
    printf("%%d", n);
}
''' % ", ".join("%du" % k for k in seeds))
    assert int(out) == len(seeds) * 6 * 2 * 5 * 9


def test_the_bound_on_tasks_is_never_reached(tmp_path):
    """Many systems per workgroup and few workgroups there: none needs more
    tasks than the launch allows it."""
    out = run(tmp_path, r'''
int main() {
    int n = 0;
    for (int bps : {8, 64, 1024})
        for (int nsys : {1, 16, 64})
            for (int stride : {bps, 1024}) {
                const int total = bps * nsys;
                if (stride > total) continue;
                const int limit = fused_task_limit(total, stride, bps);
                for (const auto& v : {range(0, 1), range(stride - 1, stride), range(0, 16), range(0, stride, 97)}) {
                    if ((int)v.size() > stride || v.back() >= stride) continue;
                    const int most = solve(bps, nsys, stride, v, limit, 0);
                    if (most < 0 || most > limit) {
                        printf("%d tiles, %d systems, stride %d, %d there: %d of %d tasks\n", bps, nsys, stride,
                               (int)v.size(), most, limit);
                        return 1;
                    }
                    n++;
                }
            }
    printf("%d", n);
}
''')
    assert int(out) >= 40


def test_a_workgroup_out_of_tasks_leaves_no_tile_as_it_was(tmp_path):
    """With too low a bound (which words changed by another launch could make
    it): every own tile ends solved or marked as lost."""
    run(tmp_path, r'''
int main() {
    for (int more : {0, 1, 2, 7, 40})
        for (int bps : {8, 16, 64})
            for (int stride : {bps, 5, 3 * bps}) {
                const int limit = (3 * bps + stride - 1) / stride + more;  // own tiles and a few
                if (solve(bps, 3, stride, range(0, 2), limit, 0) < 0) {
                    printf("limit %d: %d tiles, stride %d\n", limit, bps, stride);
                    return 1;
                }
            }
}
''')
