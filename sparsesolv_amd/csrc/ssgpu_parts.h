// Partitioned triangular sweeps: the layout of a sweep cut into parts, one
// workgroup per part (k_sweep_part).  Plain C++
// (host), shared by the library and its CPU checks.
//
// Every input of a row lies in its own part or in a part with a smaller
// number (part_choice).  Inside a part the rows are ordered by level and grouped into steps of at most 64 rows of one level.
// A step's inputs from its own part are read from the part's results in LDS;
// its inputs from earlier parts (its externals, each listed once per step) are
// polled in device memory and staged in LDS.  Every input of an entry is thus
// one LDS slot:
//   slot 0                       zero (padding entries)
//   1 + w * ext_cap + j          external j of a step taken by wave w
//   1 + waves * ext_cap + q      result of the part's row q
// and wave w of the workgroup takes the part's steps w, w + waves, ...
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <memory>
#include <new>
#include <thread>
#include <vector>

#include "ssgpu_threads.h"

namespace ssgpu {

constexpr int kPartExt = 256;     // externals of one step (a step closes before it would exceed them)
constexpr int kPartStepRows = 64; // rows of one step: one lane each
constexpr int kPartLate = 2;      // an input is late if its level is among the last this many below the row's
constexpr int kPartNear = 4;       // levels ahead of its own that a step's externals are polled
constexpr int kPartPad = 4 * kPartStepRows;   // entries 0..: a quad of zeros for every lane

// Waves of a part's workgroup, by value type and longest row (registers: 168
// a lane with 12 waves, 256 with 8, 512 with 4).
constexpr int part_waves(bool cplx, int kmax) { return cplx ? (kmax <= 20 ? 8 : 4) : (kmax <= 20 ? 12 : 8); }
constexpr int kPartMaxLen = 32;   // longest row the partitioned sweep takes

// Entries are kept in quads, so that a lane loads its row with 16-byte accesses
// (one 8-byte access for the four slots): entry 4 q + j of row l of a step is
// at ent + 4 (q cnt + l) + j, rows padded to `quads` quads.  A forward sweep's
// rows are aligned at their ends, a backward sweep's at their starts, because
// that is where their late inputs lie: rows of the part solved at most
// kPartLate levels before the row's own.  The last (forward) or first
// (backward) `late` entries hold all of a step's late inputs; the others need
// only the part's first `need0` steps, so they are gathered while the levels
// in between are still being solved.
// 32 bytes, read by a wave as one uniform load.
struct PartStep {
    int pos0;                        // first position (part-major, then level order) of the step's rows
    int lpos;                        // the same within the part
    unsigned char cnt, quads, late;  // rows; quads of the longest row; entries that may be late
    unsigned char near;              // its externals are polled once need - near steps are done
    int next;                        // externals
    int need;                        // steps of the part at lower levels: done before the late entries are read
    int need0;                       // steps more than kPartLate levels below: done before the others are
    int ent;                         // first entry
    int ext0;                        // first external
};

struct PartLayout {
    int nparts = 0, waves = 0, rows = 0;
    int64_t nent = 0;                     // entries, the first kPartPad of them padding (slot 0)
    std::vector<int> order;               // position -> row
    std::vector<int> part_step;           // nparts + 1
    std::vector<PartStep> steps;
    std::vector<unsigned short> slot;     // per entry
    std::vector<int> src;                 // per entry: index into the row arrays' entries, -1 for padding
    std::vector<int> ext;                 // positions of the externals
    int slots() const { return 1 + waves * kPartExt + rows; }   // LDS slots of a part
};

// Parts of a sweep: a part number per row, parts numbered so that a row reads
// only its own part and lower ones, and the largest part's rows.
struct PartChoice {
    int nparts = 0, most = 0;
    bool cells = false;   // grid cells (part_cells); otherwise intervals
    std::vector<int> part;
};

// A matrix numbered line by line and plane by plane (a 3-D grid) has index
// distances in three groups: rows of one line, of neighbouring lines, of
// neighbouring planes.  Looked for in a sample of the rows; not found for
// other numberings.
struct PartGrid {
    int near = 0, far = 0;     // largest distance within a line; to a neighbouring line
    int line = 0, plane = 0;   // rows of a line and of a plane
    bool found() const { return far > near; }
};
inline PartGrid part_grid(int n, const int* off, const int* col) {
    PartGrid g;
    std::vector<int> d;
    const int sample = std::min(n, 512);
    for (int q = 0; q < sample; ++q) {
        const int i = (int)((int64_t)n * q / sample);
        for (int k = off[i]; k < off[i + 1]; ++k) d.push_back(std::abs(i - col[k]));
    }
    if (d.empty()) return g;
    std::sort(d.begin(), d.end());
    std::vector<size_t> cut{0};   // a distance at least 3 times the one before starts a new group
    for (size_t k = 1; k < d.size(); ++k)
        if ((int64_t)d[k] >= 3 * (int64_t)std::max(d[k - 1], 4)) cut.push_back(k);
    cut.push_back(d.size());
    if (cut.size() != 4) return g;
    auto mid = [&](int c) { return d[(cut[c] + cut[c + 1]) / 2]; };
    if (mid(2) < 4 * (int64_t)mid(1)) return g;
    g.near = d[cut[1] - 1];
    g.far = d[cut[2] - 1];
    g.line = mid(1);
    g.plane = mid(2);
    return g;
}

// Cells of a grid numbering: bands of k planes (an interval of the row index)
// cut at every k-th value of u, the most steps to a neighbouring line on a
// path to the row.  u grows by one from line to line and, because a row reads
// the next line of the plane before, by one from plane to plane.  Neither the
// index nor u falls from an input to the row that reads it, so the cells are
// parts, and a path crosses few of them (at 95^3 with k = 6: 46 crossings,
// against 162 of as many intervals of the row index).
inline PartChoice part_cells(int n, const int* off, const int* col, bool forward, const PartGrid& g, int k) {
    PartChoice c;
    std::vector<int> u(n);
    int umax = 0;
    for (int q = 0; q < n; ++q) {
        const int i = forward ? q : n - 1 - q;
        int m = 0;
        for (int e = off[i]; e < off[i + 1]; ++e) {
            const int j = col[e], dist = std::abs(i - j);
            m = std::max(m, u[j] + (dist > g.near && dist <= g.far));
        }
        u[i] = m;
        umax = std::max(umax, m);
    }
    const int64_t band = (int64_t)k * g.plane;
    const int64_t nb = (n + band - 1) / band, nu = umax / k + 1;
    if (nb * nu > n) return c;
    std::vector<int> count((size_t)(nb * nu), 0);
    c.part.resize(n);
    for (int i = 0; i < n; ++i) {
        c.part[i] = (int)((forward ? i : n - 1 - i) / band * nu + u[i] / k);
        ++count[c.part[i]];
    }
    // Cells that hold rows, numbered by diagonals of (band, u): the order in
    // which the levels reach them, so that the workgroups running at any time
    // are those of the cells being solved.
    for (int64_t diag = 0; diag < nb + nu - 1; ++diag)
        for (int64_t b = std::max<int64_t>(0, diag - nu + 1); b <= std::min(diag, nb - 1); ++b) {
            int& x = count[(size_t)(b * nu + diag - b)];
            if (x == 0) continue;
            c.most = std::max(c.most, x);
            x = c.nparts++;
        }
    for (int i = 0; i < n; ++i) c.part[i] = count[c.part[i]];
    c.cells = true;
    return c;
}

// Intervals of the row index of at most `rows` rows, of even size.
inline PartChoice part_intervals(int n, bool forward, int rows) {
    PartChoice c;
    const int P = (n + rows - 1) / rows;
    c.most = (n + P - 1) / P;
    c.nparts = (n + c.most - 1) / c.most;
    c.part.resize(n);
    for (int i = 0; i < n; ++i) c.part[i] = (forward ? i : n - 1 - i) / c.most;
    return c;
}

// The same parts for the sweep over the transposed triangle: its rows read
// where the first sweep's rows are read from, so the parts in reverse order.
inline PartChoice part_reverse(PartChoice c) {
    for (int& p : c.part) p = c.nparts - 1 - p;
    return c;
}

// off/col: off-diagonal entries of each row on the solved side, in summation
// order; lev: level of each row.  ch.most <= 65535 - waves * kPartExt - 1.
inline PartLayout part_layout(int n, const int* off, const int* col, const int* lev, bool forward,
                              const PartChoice& ch, int waves) {
    PartLayout L;
    const int P = ch.nparts;
    L.rows = ch.most;
    L.waves = waves;
    L.nparts = P;
    L.order.resize(n);
    std::vector<int> pos(n), first(P + 1, 0), list(n);
    for (int i = 0; i < n; ++i) ++first[ch.part[i] + 1];
    for (int q = 0; q < P; ++q) first[q + 1] += first[q];
    {   // the rows of each part, in the sweep's index order
        std::vector<int> fill(first.begin(), first.end() - 1);
        for (int k = 0; k < n; ++k) {
            const int i = forward ? k : n - 1 - k;
            list[fill[ch.part[i]]++] = i;
        }
    }
    struct Piece {
        std::vector<PartStep> steps;
        std::vector<unsigned short> slot;
        std::vector<int> src, ext;
    };
    std::vector<Piece> piece(P);
    const int hw = (int)std::thread::hardware_concurrency();
    const int nt = std::max(1, std::min({hw > 0 ? hw : 1, 16, P, n / 2048 + 1}));
    auto each_part = [&](auto&& f) { each_share(P, nt, f); };   // f(part, thread)
    // positions: rows of a part by level, in the sweep's index order within one
    each_part([&](int q, int) {
        const int p0 = first[q], m = first[q + 1] - p0;
        auto row = [&](int k) { return list[p0 + k]; };
        int lo = lev[row(0)], hi = lo;
        for (int k = 1; k < m; ++k) {
            lo = std::min(lo, lev[row(k)]);
            hi = std::max(hi, lev[row(k)]);
        }
        if ((int64_t)hi - lo < 8 * (int64_t)m + 1024) {
            std::vector<int> cnt(hi - lo + 2, 0);
            for (int k = 0; k < m; ++k) cnt[lev[row(k)] - lo + 1]++;
            for (int l = 0; l <= hi - lo; ++l) cnt[l + 1] += cnt[l];
            for (int k = 0; k < m; ++k) L.order[p0 + cnt[lev[row(k)] - lo]++] = row(k);
        } else {
            for (int k = 0; k < m; ++k) L.order[p0 + k] = row(k);
            std::stable_sort(L.order.begin() + p0, L.order.begin() + p0 + m,
                             [&](int a, int b) { return lev[a] < lev[b]; });
        }
        for (int k = 0; k < m; ++k) pos[L.order[p0 + k]] = p0 + k;
    });
    // steps: consecutive positions of one level, cut at 64 rows and at kPartExt externals
    struct Free {
        void operator()(int* p) const { std::free(p); }
    };
    struct Mark {   // per thread: the step that last listed a position, and its place in the list
        std::unique_ptr<int, Free> seen, at;
    };
    std::vector<Mark> mark(nt);
    each_part([&](int q, int t) {
        Mark& M = mark[t];
        if (!M.seen) {
            M.seen.reset(static_cast<int*>(std::calloc((size_t)n, sizeof(int))));
            M.at.reset(static_cast<int*>(std::malloc((size_t)n * sizeof(int))));
        }
        if (!M.seen || !M.at) throw std::bad_alloc();
        int* seen = M.seen.get();
        int* at = M.at.get();
        Piece& pc = piece[q];
        const int p0 = first[q], p1 = first[q + 1];
        const int xbase = 1 + waves * kPartExt - p0;
        {
            size_t e = 0;
            for (int p = p0; p < p1; ++p) e += off[L.order[p] + 1] - off[L.order[p]];
            pc.slot.reserve(e + e / 4);
            pc.src.reserve(e + e / 4);
        }
        // first steps of the level, of the lowest late level, of the lowest level whose completion starts the polls
        int level_first = 0, level = lev[L.order[p0]], early = 0, polls = 0;
        for (int p = p0; p < p1;) {
            const int st = (int)pc.steps.size();
            if (lev[L.order[p]] != level) {
                level = lev[L.order[p]];
                level_first = st;
                while (early < st && lev[L.order[pc.steps[early].pos0]] < level - kPartLate) ++early;
                while (polls < st && lev[L.order[pc.steps[polls].pos0]] < level - kPartNear) ++polls;
            }
            PartStep s{};
            s.pos0 = p;
            s.lpos = p - p0;
            s.need = level_first;
            s.need0 = early;
            s.near = (unsigned char)std::min(255, level_first - polls);
            s.ext0 = (int)pc.ext.size();
            s.ent = (int)pc.slot.size();
            const int stamp = p + 1;   // of this thread's steps, each has its own first position
            const int wbase = 1 + (st % waves) * kPartExt;
            int e = p, longest = 0;
            for (; e < p1 && e - p < kPartStepRows && lev[L.order[e]] == level; ++e) {
                const int i = L.order[e];
                int fresh = 0;   // externals this row adds (a row lists a column once)
                for (int k = off[i]; k < off[i + 1]; ++k) {
                    const int c = pos[col[k]];
                    if ((c < p0 || c >= p1) && seen[c] != stamp) ++fresh;
                }
                if (e > p && s.next + fresh > kPartExt) break;
                for (int k = off[i]; k < off[i + 1]; ++k) {
                    const int c = pos[col[k]];
                    if ((c < p0 || c >= p1) && seen[c] != stamp) {
                        seen[c] = stamp;
                        at[c] = s.next++;
                        pc.ext.push_back(c);
                    }
                }
                longest = std::max(longest, off[i + 1] - off[i]);
            }
            s.cnt = (unsigned char)(e - p);
            s.quads = (unsigned char)((longest + 3) / 4);
            const int len = 4 * s.quads;
            pc.slot.resize(pc.slot.size() + (size_t)s.cnt * len, 0);
            pc.src.resize(pc.src.size() + (size_t)s.cnt * len, -1);
            for (int l = 0; l < s.cnt; ++l) {
                const int i = L.order[p + l];
                const int shift = forward ? len - (off[i + 1] - off[i]) : 0;
                for (int k = off[i]; k < off[i + 1]; ++k) {
                    const int c = pos[col[k]];
                    const int at_k = k - off[i] + shift;
                    const size_t d = (size_t)s.ent + 4 * ((size_t)(at_k / 4) * s.cnt + l) + at_k % 4;
                    pc.src[d] = k;
                    if (c >= p0 && c < p1 && lev[col[k]] >= level - kPartLate)
                        s.late = (unsigned char)std::max<int>(s.late, forward ? len - at_k : at_k + 1);
                    pc.slot[d] = (unsigned short)((c < p0 || c >= p1) ? wbase + at[c] : xbase + c);
                }
            }
            pc.steps.push_back(s);
            p = e;
        }
    });
    // one array of each kind, the padding entries first
    L.part_step.assign(P + 1, 0);
    std::vector<int64_t> ent(P + 1, kPartPad), ext(P + 1, 0);
    for (int q = 0; q < P; ++q) {
        L.part_step[q + 1] = L.part_step[q] + (int)piece[q].steps.size();
        ent[q + 1] = ent[q] + (int64_t)piece[q].slot.size();
        ext[q + 1] = ext[q] + (int64_t)piece[q].ext.size();
    }
    L.nent = ent[P];
    if (L.nent > INT32_MAX || ext[P] > INT32_MAX) {   // beyond the steps' 32-bit offsets: no layout
        L.nparts = 0;
        return L;
    }
    L.steps.resize(L.part_step[P]);
    L.slot.resize(L.nent);
    L.src.resize(L.nent);
    L.ext.resize(std::max<int64_t>(ext[P], 1));
    std::fill(L.slot.begin(), L.slot.begin() + kPartPad, (unsigned short)0);
    std::fill(L.src.begin(), L.src.begin() + kPartPad, -1);
    each_part([&](int q, int) {
        Piece& pc = piece[q];
        for (size_t k = 0; k < pc.steps.size(); ++k) {
            PartStep s = pc.steps[k];
            s.ent += (int)ent[q];
            s.ext0 += (int)ext[q];
            L.steps[L.part_step[q] + k] = s;
        }
        std::copy(pc.slot.begin(), pc.slot.end(), L.slot.begin() + ent[q]);
        std::copy(pc.src.begin(), pc.src.end(), L.src.begin() + ent[q]);
        std::copy(pc.ext.begin(), pc.ext.end(), L.ext.begin() + ext[q]);
        pc = Piece();
    });
    return L;
}

}  // namespace ssgpu
