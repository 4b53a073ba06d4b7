// Work order of a triangular sweep (sweep_kernels.hip), built on the host from a level
// order of its rows: no HIP in here.
//
// The cells are cut into chunks of consecutive indices; a workgroup takes a chunk and
// keeps its part of x in LDS. A chunk's rows are in level order, in steps of at most 64
// rows of one level (one wavefront each). A step may start once every step of the
// chunk's earlier levels is done (`need`, a count of steps); rows of one level never
// depend on each other. Dependencies between chunks go by the values themselves, and
// only from a chunk swept earlier in index order (later, for a backward sweep). Values of
// other chunks that a sweep reads as they were before it (Gauss–Seidel: the neighbours on
// the side not yet swept) are copied into LDS with the chunk: its halo.
//
// An entry names where its value lies: the LDS slot (a chunk's cells from 0, then its
// halo, then one slot for padding), or ~i for a value to be read from memory. Values go
// from chunk to chunk through a mailbox in row-position order, so that the 64 rows of a
// step write, and their neighbours' rows mostly read, a few whole cache lines: i = n +
// position for the neighbour's value of the same sweep and i = position for its value of
// the sweep before (`col2`, the sweeps after the first of one launch); i = 2n + cell is
// the neighbour's x before the first sweep, where the halo did not hold it. Rows are
// padded to a multiple of SWEEP_GROUP entries.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <vector>

namespace vol {

constexpr int SWEEP_STEP = 64;           // rows of a step
constexpr int SWEEP_GROUP = 4;           // entries are loaded and gathered in groups
constexpr int SWEEP_MAX_SLOTS = 20400;   // LDS slots besides the padding: 160 KB in FP64
constexpr int SWEEP_ROWS_BITS = 7;       // low bits of SweepStep::rowsNeed

struct SweepStep {
    int pos;       // first row position
    int base;      // entry k of the step's row t is base + k·rows + t
    int width;     // entries per row, padded to whole groups
    int rowsNeed;  // rows | need << SWEEP_ROWS_BITS
};

struct SweepPlanHost {
    int n = 0, nChunks = 0, maxSlots = 0, maxWidth = 0;
    int64_t serial = 0;         // Σ 1 + entry groups over the steps: the work if they ran in turn
    std::vector<int> chunkOff;  // first cell of each chunk (nChunks + 1)
    std::vector<int> stepOff;   // first step of each chunk (nChunks + 1)
    std::vector<int> haloOff, halo;  // cells of each chunk's halo
    std::vector<SweepStep> steps;
    std::vector<int> cell;      // per row position
    std::vector<int> col, src;  // per entry: place of the value, coefficient source (−1: padding)
    std::vector<int> col2;      // places in the sweeps after the first
};

// Chunks of a sweep over n cells by levels off/perm. Up to SWEEP_ONE_CELLS cells one chunk:
// every dependence stays in LDS, and several sweeps run as one pipelined schedule (two
// Gauss–Seidel sweeps over 4,096 box cells 28 µs against 30 in 4 chunks, over 10,260
// agglomerated cells of 16 neighbours 105 against 108, but over 16,384 box cells 92 against
// 55 in 8: one CU streams its rows at about 30 GB/s). Above, a chunk holds as many cells as
// keep its levels at 128 rows on average, two steps of each level at a time (373,920 tets,
// 158 levels: 18 of them in 6144 cells, 8 in 1536, where two sweeps take 340 and 200 µs;
// 64³ hexes, whose chunks all see about 128 of the 190 levels: 188 and 261); fewer cells
// only add hops between chunks. Long rows (coarse GAMG levels, few rows a level): 4096.
// Where that makes at most SWEEP_FEW_CHUNKS chunks, twice as many: a step less per level and
// chunk is then worth more than the hops (two sweeps, as given and doubled: 16,384 box cells
// in 3 chunks 54 → 44 µs, 65,536 in 11: 91 → 85, 24,000 agglomerated cells in 6: 206 → 170,
// 10,000 in 3: 79 → 65; but 93,000 agglomerated cells in 23: 175 → 203, 262,144 box cells in
// 43: 150 → 204).
constexpr int SWEEP_ONE_CELLS = 8192;
constexpr int SWEEP_FEW_CHUNKS = 12;
inline int sweepChunks(int n, const std::vector<int>& off, const std::vector<int>& perm, bool longRows) {
    if (n <= SWEEP_ONE_CELLS) return 1;
    auto chunks = [n](int cells) {
        const int nc = (n + cells - 1) / cells;
        return nc <= SWEEP_FEW_CHUNKS ? 2 * nc : nc;
    };
    if (longRows) return chunks(4096);
    for (int cells : {6144, 3072}) {
        const int nc = (n + cells - 1) / cells;
        int64_t runs = 0;  // (level, chunk) pairs
        for (size_t L = 0; L + 1 < off.size(); ++L)
            for (int i = off[L], last = -1; i < off[L + 1]; ++i) {
                const int k = int(int64_t(perm[i]) * nc / n);
                runs += k != last;
                last = k;
            }
        if (runs * 128 >= n) return chunks(cells);
    }
    return chunks(1536);
}

// Polls of one value after which a wait of `sweeps` sweeps counts as failed. The earliest
// unfinished chunk always proceeds, so a wait lasts at most as long as all steps one after
// the other: 0.4 µs each when the rows are held (a chain of cells: every step a level), 2
// µs per entry group past those. A poll is a memory round trip (0.3 µs at the least, 0.7
// measured), so SWEEP_STEP_POLLS per step and group are over ten times that, and
// SWEEP_BASE_POLLS (0.1–0.2 s) cover what does not grow with the plan. A fixed limit of
// the base alone ended sweeps over a chain of two million cells (0.8 s) with an error.
constexpr int64_t SWEEP_BASE_POLLS = int64_t(1) << 18, SWEEP_STEP_POLLS = 16;
inline uint32_t sweepPolls(int64_t serial, int sweeps) {
    return uint32_t(std::min<int64_t>(SWEEP_BASE_POLLS + SWEEP_STEP_POLLS * serial * sweeps, 0xfffffff0));
}

// off/perm: cells by level (levels off[L] .. off[L+1], ascending cells within a level;
// one chunk may list a cell several times, once per sweep of a pipelined schedule);
// rowOff/rowCol/rowSrc: the rows in the order of their sums. oldSide: neighbours whose
// value before the sweep is read (1: higher-numbered ones, −1: lower-numbered, 0: none).
// again: the plan is also used for sweeps after the first of a launch (one pass over the
// cells in perm).
inline SweepPlanHost buildSweepPlan(int n, const std::vector<int>& off, const std::vector<int>& perm,
                                    const std::vector<int>& rowOff, const std::vector<int>& rowCol,
                                    const std::vector<int>& rowSrc, int nChunks, int oldSide, bool again) {
    SweepPlanHost P;
    P.n = n;
    P.nChunks = std::max(1, std::min(nChunks, std::max(n, 1)));
    const int nc = P.nChunks, nl = int(off.size()) - 1;
    P.chunkOff.resize(nc + 1);
    for (int k = 0; k <= nc; ++k) P.chunkOff[k] = int(int64_t(n) * k / nc);
    // a level's ascending cells fall into runs of one chunk each: count, then place
    std::vector<int> posOff(nc + 1, 0), stepCnt(nc, 0);
    auto runs = [&](auto&& f) {
        for (int L = 0; L < nl; ++L)
            for (int i = off[L], k = 0; i < off[L + 1];) {
                while (perm[i] >= P.chunkOff[k + 1]) ++k;
                int e = i;
                if (nc == 1) e = off[L + 1];
                else
                    while (e < off[L + 1] && perm[e] < P.chunkOff[k + 1]) ++e;
                f(k, i, e);
                i = e;
            }
    };
    runs([&](int k, int i, int e) {
        posOff[k + 1] += e - i;
        stepCnt[k] += (e - i + SWEEP_STEP - 1) / SWEEP_STEP;
    });
    P.stepOff.assign(nc + 1, 0);
    for (int k = 0; k < nc; ++k) {
        posOff[k + 1] += posOff[k];
        P.stepOff[k + 1] = P.stepOff[k] + stepCnt[k];
        if (stepCnt[k] >= (1 << (31 - SWEEP_ROWS_BITS))) throw std::length_error("sweep chunk has too many steps");
    }
    P.cell.resize(perm.size());
    P.steps.resize(P.stepOff[nc]);
    std::vector<int> pf(posOff.begin(), posOff.end() - 1), sf(P.stepOff.begin(), P.stepOff.end() - 1);
    runs([&](int k, int i, int e) {
        const int need = sf[k] - P.stepOff[k];  // every step of the earlier levels
        for (; i < e; i += SWEEP_STEP) {
            const int rows = std::min(SWEEP_STEP, e - i);
            int w = 0;
            for (int q = 0; q < rows; ++q) {
                const int c = perm[i + q];
                P.cell[pf[k] + q] = c;
                w = std::max(w, rowOff[c + 1] - rowOff[c]);
            }
            w = (w + SWEEP_GROUP - 1) / SWEEP_GROUP * SWEEP_GROUP;
            P.steps[sf[k]++] = SweepStep{pf[k], 0, w, rows | (need << SWEEP_ROWS_BITS)};
            pf[k] += rows;
        }
    });
    size_t total = 0;
    for (SweepStep& s : P.steps) {
        s.base = int(total);
        total += size_t(s.width) * size_t(s.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1));
        P.maxWidth = std::max(P.maxWidth, s.width);
        P.serial += 1 + s.width / SWEEP_GROUP;
        if (total >= (size_t(1) << 31)) throw std::length_error("sweep rows exceed 2^31 entries");
    }
    again = again && nc > 1;
    P.col.assign(std::max<size_t>(total, 1), 0);
    P.src.assign(std::max<size_t>(total, 1), -1);
    if (again) P.col2.assign(P.col.size(), 0);
    P.haloOff.assign(nc + 1, 0);
    std::vector<int> slot(nc > 1 ? n : 0, -1), posOf(nc > 1 ? n : 0);  // slot: of this chunk's halo cells
    if (nc > 1) {
        if (n > (1 << 29)) throw std::length_error("sweep over too many cells");
        for (size_t q = 0; q < P.cell.size(); ++q) posOf[P.cell[q]] = int(q);
    }
    for (int k = 0; k < nc; ++k) {
        const int c0 = P.chunkOff[k], size = P.chunkOff[k + 1] - c0;
        if (size > SWEEP_MAX_SLOTS) throw std::length_error("sweep chunk exceeds the LDS slots");
        for (int s = P.stepOff[k]; s < P.stepOff[k + 1]; ++s) {
            const SweepStep& st = P.steps[s];
            const int rows = st.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1);
            for (int t = 0; t < rows; ++t) {
                const int c = P.cell[st.pos + t];
                size_t e = size_t(st.base) + t;
                for (int q = rowOff[c]; q < rowOff[c + 1]; ++q, e += rows) {
                    const int j = rowCol[q];
                    P.src[e] = rowSrc[q];
                    const bool old = oldSide > 0 ? j > c : oldSide < 0 && j < c;
                    const bool inside = unsigned(j - c0) < unsigned(size);
                    if (again) P.col2[e] = old ? ~posOf[j] : inside ? j - c0 : ~(n + posOf[j]);
                    if (inside) {
                        P.col[e] = j - c0;
                        continue;
                    }
                    const int held = int(P.halo.size()) - P.haloOff[k];
                    if (old && slot[j] < 0 && size + held < SWEEP_MAX_SLOTS) {
                        slot[j] = size + held;
                        P.halo.push_back(j);
                    }
                    P.col[e] = !old ? ~(n + posOf[j]) : slot[j] >= 0 ? slot[j] : ~(2 * n + j);
                }
            }
        }
        P.haloOff[k + 1] = int(P.halo.size());
        const int pad = size + P.haloOff[k + 1] - P.haloOff[k];
        P.maxSlots = std::max(P.maxSlots, pad);
        for (int h = P.haloOff[k]; h < P.haloOff[k + 1]; ++h) slot[P.halo[h]] = -1;
        if (P.stepOff[k] < P.stepOff[k + 1]) {
            const size_t e0 = P.steps[P.stepOff[k]].base;
            const SweepStep& l = P.steps[P.stepOff[k + 1] - 1];
            const size_t e1 = l.base + size_t(l.width) * (l.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1));
            for (size_t e = e0; e < e1; ++e)
                if (P.src[e] < 0) {
                    P.col[e] = pad;
                    if (again) P.col2[e] = pad;
                }
        }
    }
    return P;
}

}  // namespace vol
