// Host check of the sweep plans (voluma_amd/csrc/sweep_plan.hpp), built and run by
// test_sweep_plan.py with the address and undefined-behaviour sanitizers.
//   limit <n>   a chain of n cells, one row per level: its chunks, steps and wait limit
//   sweep <faces> <backward> <sweeps> <chunks> <old>
//               sweeps x_c = (b_c − Σ a·x) / d_c over the graph in the file (n, then l and u of
//               each face) worked through as the kernels do, chunks 0: as many as they take,
//               against the sequential loop. old 1: values of the other side as they were
//               (Gauss–Seidel); 0: only the entries already swept (a substitution)
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

// Levels of k consecutive sweeps: a cell follows its neighbours already swept, its
// neighbours' and its own sweep before.
void levels(const Graph& g, bool backward, int k, std::vector<int>& off, std::vector<int>& perm) {
    std::vector<std::vector<int>> before(g.n), after(g.n);
    for (size_t f = 0; f < g.l.size(); ++f) {
        const int a = backward ? g.u[f] : g.l[f], b = backward ? g.l[f] : g.u[f];
        before[b].push_back(a);
        after[a].push_back(b);
    }
    std::vector<int> prev(g.n, -1), cur(g.n, 0);
    std::vector<std::vector<int>> cells;
    for (int s = 0; s < k; ++s, prev = cur)
        for (int t = 0; t < g.n; ++t) {
            const int c = backward ? g.n - 1 - t : t;
            int L = prev[c] + 1;
            for (int j : before[c]) L = std::max(L, cur[j] + 1);
            for (int j : after[c]) L = std::max(L, prev[j] + 1);
            cur[c] = L;
            if (size_t(L) >= cells.size()) cells.resize(L + 1);
            cells[L].push_back(c);
        }
    off.assign(1, 0);
    perm.clear();
    for (auto& v : cells) {
        std::sort(v.begin(), v.end());
        perm.insert(perm.end(), v.begin(), v.end());
        off.push_back(int(perm.size()));
    }
}

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

[[noreturn]] void fail(const char* what, long long a = 0, long long b = 0) {
    std::printf("%s (%lld, %lld)\n", what, a, b);
    std::exit(1);
}

struct Value {
    double v = 0.0;
    bool there = false;
};

// What k_sweep_one and k_sweep_chunks do with a plan, chunk by chunk. early: every chunk's
// x and halo are copied before the first chunk works, else each when its turn comes;
// reversed: the steps of a level and the rows of a step from the last to the first (they
// must not depend on each other).
std::vector<double> workThrough(const SweepPlanHost& P, const std::vector<double>& a, const std::vector<double>& b,
                                const std::vector<double>& d, std::vector<double> x, bool backward, int launchSweeps,
                                bool early, bool reversed) {
    const int n = P.n, nc = P.nChunks;
    std::vector<Value> mail(nc > 1 ? size_t(n) * launchSweeps : 0);
    auto fill = [&](int k) {
        const int c0 = P.chunkOff.at(k), size = P.chunkOff.at(k + 1) - c0;
        std::vector<Value> xs(size + P.haloOff.at(k + 1) - P.haloOff.at(k) + 1);
        for (int q = 0; q < size; ++q) xs.at(q) = {x.at(c0 + q), true};
        for (int h = P.haloOff.at(k); h < P.haloOff.at(k + 1); ++h)
            xs.at(size + h - P.haloOff.at(k)) = {x.at(P.halo.at(h)), true};
        xs.back() = {0.0, true};
        return xs;
    };
    std::vector<std::vector<Value>> start(nc);
    for (int k = 0; early && k < nc; ++k) start[k] = fill(k);
    for (int sweep = 0; sweep < launchSweeps; ++sweep)
        for (int i = 0; i < nc; ++i) {
            const int k = backward ? nc - 1 - i : i;
            const int c0 = P.chunkOff.at(k), size = P.chunkOff.at(k + 1) - c0;
            std::vector<Value> xs;
            if (sweep == 0) xs = early ? start[k] : fill(k);
            else {
                xs.resize(size + P.haloOff.at(k + 1) - P.haloOff.at(k) + 1);
                xs.back() = {0.0, true};
            }
            const std::vector<int>& places = sweep > 0 ? P.col2 : P.col;
            const int s0 = P.stepOff.at(k), s1 = P.stepOff.at(k + 1);
            for (int s = s0; s < s1;) {  // the steps of one level: those with the same need
                int e = s;
                const int need = P.steps.at(s).rowsNeed >> SWEEP_ROWS_BITS;
                while (e < s1 && P.steps.at(e).rowsNeed >> SWEEP_ROWS_BITS == need) ++e;
                if (need != s - s0) fail("a level waits for another count than the steps before it", need, s - s0);
                for (int q = 0; q < e - s; ++q) {
                    const SweepStep& st = P.steps.at(reversed ? e - 1 - q : s + q);
                    const int rows = st.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1);
                    if (rows < 1 || rows > SWEEP_STEP || st.width % SWEEP_GROUP) fail("shape of a step", rows, st.width);
                    for (int w = 0; w < rows; ++w) {
                        const int t = reversed ? rows - 1 - w : w;
                        const int c = P.cell.at(st.pos + t);
                        double acc = b.at(c);
                        for (int g = 0; g < st.width; ++g) {
                            const size_t at = size_t(st.base) + size_t(g) * rows + t;
                            const int place = places.at(at), src = P.src.at(at);
                            const double f = src < 0 ? 0.0 : a.at(src);
                            double v;
                            if (place >= 0) {
                                if (!xs.at(place).there) fail("a slot read before it is written", c, place);
                                v = xs.at(place).v;
                            } else if (~place < 2 * n) {
                                const Value& m = mail.at(size_t(sweep) * n + ~place - n);
                                if (!m.there) fail("a value not sent by an earlier chunk or sweep", c, ~place);
                                v = m.v;
                            } else {
                                if (sweep > 0) fail("x read in a later sweep", c, ~place);
                                v = x.at(~place - 2 * n);
                            }
                            acc = acc - f * v;
                        }
                        acc = acc / d.at(c);
                        xs.at(c - c0) = {acc, true};
                        if (nc > 1) mail.at(size_t(sweep) * n + st.pos + t) = {acc, true};
                    }
                }
                s = e;
            }
            if (sweep + 1 == launchSweeps)
                for (int q = 0; q < size; ++q) {
                    if (!xs.at(q).there) fail("a cell that was not swept", c0 + q);
                    x.at(c0 + q) = xs.at(q).v;
                }
        }
    return x;
}

int sweep(const char* file, bool backward, int sweeps, int nChunks, bool old) {
    Graph g;
    std::FILE* in = std::fopen(file, "rb");
    int nf = 0;
    if (!in || std::fread(&g.n, 4, 1, in) != 1 || std::fread(&nf, 4, 1, in) != 1) return 2;
    g.l.resize(nf);
    g.u.resize(nf);
    if (std::fread(g.l.data(), 4, nf, in) != size_t(nf) || std::fread(g.u.data(), 4, nf, in) != size_t(nf)) return 2;
    std::fclose(in);
    std::vector<int> off, perm, ro, rc, rs;
    rows(g, ro, rc, rs);
    if (!old) {  // only the entries on the side already swept
        std::vector<int> o(1, 0), c2, s2;
        for (int c = 0; c < g.n; ++c) {
            for (int q = ro[c]; q < ro[c + 1]; ++q)
                if (backward ? rc[q] > c : rc[q] < c) {
                    c2.push_back(rc[q]);
                    s2.push_back(rs[q]);
                }
            o.push_back(int(c2.size()));
        }
        ro = o;
        rc = c2;
        rs = s2;
    }
    levels(g, backward, 1, off, perm);
    int width = 0;
    for (int c = 0; c < g.n; ++c) width = std::max(width, ro[c + 1] - ro[c]);
    if (!nChunks) nChunks = sweepChunks(g.n, off, perm, width > 8);
    const bool one = nChunks == 1;
    if (one) levels(g, backward, sweeps, off, perm);
    const SweepPlanHost P =
        buildSweepPlan(g.n, off, perm, ro, rc, rs, nChunks, !old ? 0 : backward ? -1 : 1, sweeps > 1);
    unsigned long long r = 88172645463325252ull;
    auto uniform = [&] {  // xorshift
        r ^= r << 13;
        r ^= r >> 7;
        r ^= r << 17;
        return double(r >> 11) * 0x1p-53;
    };
    std::vector<double> a(2 * size_t(nf)), b(g.n), d(g.n), x(g.n);
    for (double& v : a) v = uniform() - 1.5;
    for (double& v : b) v = 2.0 * uniform() - 1.0;
    for (double& v : x) v = 2.0 * uniform() - 1.0;
    for (int c = 0; c < g.n; ++c) {
        d[c] = 0.1;
        for (int q = ro[c]; q < ro[c + 1]; ++q) d[c] += -a[rs[q]];
    }
    std::vector<double> want = x;
    for (int s = 0; s < sweeps; ++s)
        for (int t = 0; t < g.n; ++t) {
            const int c = backward ? g.n - 1 - t : t;
            double acc = b[c];
            for (int q = ro[c]; q < ro[c + 1]; ++q) acc = acc - a[rs[q]] * want[rc[q]];
            want[c] = acc / d[c];
        }
    for (bool early : {false, true})
        for (bool reversed : {false, true}) {
            const std::vector<double> got = workThrough(P, a, b, d, x, backward, one ? 1 : sweeps, early, reversed);
            for (int c = 0; c < g.n; ++c)
                if (std::memcmp(&got[c], &want[c], 8)) fail("another value", c, reversed);
        }
    long long mailed = 0, fromX = 0;
    for (int p : P.col) {
        mailed += p < 0 && ~p < 2 * g.n;
        fromX += p < 0 && ~p >= 2 * g.n;
    }
    std::printf("chunks %d slots %d width %d halo %zu mailed %lld fromx %lld\n", P.nChunks, P.maxSlots, P.maxWidth,
                P.halo.size(), mailed, fromX);
    return P.maxSlots <= SWEEP_MAX_SLOTS ? 0 : 1;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc == 3 && !std::strcmp(argv[1], "limit")) return limit(std::atoi(argv[2]));
    if (argc == 7 && !std::strcmp(argv[1], "sweep"))
        return sweep(argv[2], std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6]));
    return 2;
}
