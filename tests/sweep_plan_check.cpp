// Host check of the sweep plans (voluma_amd/csrc/sweep_plan.hpp), built and run by
// test_sweep_plan.py with the address and undefined-behaviour sanitizers.
//   limit <n>   a chain of n cells, one row per level: its chunks, steps and wait limit
#include "sweep_plan.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

using namespace vol;

namespace {

struct Graph {
    int n = 0;
    std::vector<int> l, u;  // face f joins l[f] < u[f]
};

// Rows in face order; the source is face << 1 | side.
void rows(const Graph& g, std::vector<int>& off, std::vector<int>& col, std::vector<int>& src) {
    const int nf = int(g.l.size());
    off.assign(g.n + 1, 0);
    for (int f = 0; f < nf; ++f) {
        ++off[g.l[f] + 1];
        ++off[g.u[f] + 1];
    }
    for (int c = 0; c < g.n; ++c) off[c + 1] += off[c];
    std::vector<int> fill(off.begin(), off.end() - 1);
    col.resize(2 * size_t(nf));
    src.resize(2 * size_t(nf));
    for (int f = 0; f < nf; ++f) {
        col[fill[g.l[f]]] = g.u[f];
        src[fill[g.l[f]]++] = f << 1;
        col[fill[g.u[f]]] = g.l[f];
        src[fill[g.u[f]]++] = f << 1 | 1;
    }
}

int limit(int n) {
    Graph g;
    g.n = n;
    for (int c = 0; c + 1 < n; ++c) {
        g.l.push_back(c);
        g.u.push_back(c + 1);
    }
    std::vector<int> off(n + 1), perm(n), ro, rc, rs;
    for (int c = 0; c < n; ++c) off[c + 1] = perm[c] = c;  // level c holds cell c
    for (int c = 0; c <= n; ++c) off[c] = c;
    rows(g, ro, rc, rs);
    const SweepPlanHost P = buildSweepPlan(n, off, perm, ro, rc, rs, sweepChunks(n, off, perm, false), 1, true);
    std::printf("chunks %d steps %zu polls %u\n", P.nChunks, P.steps.size(), sweepPolls(P.serial, 1));
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc == 3 && !std::strcmp(argv[1], "limit")) return limit(std::atoi(argv[2]));
    return 2;
}
