// Runs a partitioned sweep's layout (ssgpu_parts.h) on the CPU the way the
// kernel does, one part after another and one step after another, and checks
// every index it would use.  Built as a shared library by the test.
#include <cmath>
#include <vector>

#include "ssgpu_parts.h"

using namespace ssgpu;

// rows > 0: intervals of that many rows; cell > 0: grid cells (7 when the
// matrix has no grid numbering); rows < 0: the parts of the transposed sweep.  x receives the solution of the triangular
// system (lower for forward, upper otherwise) with right-hand side r; info:
// parts, largest part, steps, externals, most externals of a step.
// Returns 0, or the number of the check that failed.
extern "C" int part_layout_run(int n, const int* rp, const int* ci, const double* v, int forward, int rows, int cell,
                               int waves, const double* r, double* x, int* info) {
    std::vector<int> off(n + 1, 0), col, lev(n, 0);
    std::vector<double> val, d(n, 1.0);
    for (int i = 0; i < n; ++i) {
        for (int k = rp[i]; k < rp[i + 1]; ++k) {
            if (ci[k] == i) d[i] = v[k];
            else if ((ci[k] < i) == (forward != 0)) {
                col.push_back(ci[k]);
                val.push_back(v[k]);
            }
        }
        off[i + 1] = (int)col.size();
    }
    for (int q = 0; q < n; ++q) {
        const int i = forward ? q : n - 1 - q;
        for (int k = off[i]; k < off[i + 1]; ++k) lev[i] = std::max(lev[i], lev[col[k]] + 1);
    }
    auto choice = [&](const std::vector<int>& o, const std::vector<int>& c, bool fwd, int most) {
        if (cell == 0) return part_intervals(n, fwd, most);
        const PartGrid g = part_grid(n, o.data(), c.data());
        return g.found() ? part_cells(n, o.data(), c.data(), fwd, g, cell) : PartChoice();
    };
    PartChoice ch;
    if (rows >= 0) {
        ch = choice(off, col, forward != 0, rows);
    } else {   // the parts of the transposed triangle's sweep, reversed
        std::vector<int> toff(n + 1, 0), tcol(col.size());
        for (int j : col) ++toff[j + 1];
        for (int i = 0; i < n; ++i) toff[i + 1] += toff[i];
        std::vector<int> fill(toff.begin(), toff.end() - 1);
        for (int i = 0; i < n; ++i)
            for (int k = off[i]; k < off[i + 1]; ++k) tcol[fill[col[k]]++] = i;
        ch = part_reverse(choice(toff, tcol, forward == 0, -rows));
    }
    if (ch.nparts == 0) return 7;
    const PartLayout L = part_layout(n, off.data(), col.data(), lev.data(), forward != 0, ch, waves);
    std::vector<double> xp(n, NAN), lds(L.slots());
    std::vector<int> step_of(L.rows);
    int most_ext = 0;
    for (int q = 0; q < L.nparts; ++q) {
        std::fill(lds.begin(), lds.end(), NAN);
        lds[0] = 0.0;
        const int xb = 1 + waves * kPartExt, first = L.steps[L.part_step[q]].pos0;
        for (int st = L.part_step[q]; st < L.part_step[q + 1]; ++st)
            for (int l = 0; l < L.steps[st].cnt; ++l) step_of[L.steps[st].lpos + l] = st - L.part_step[q];
        for (int st = L.part_step[q]; st < L.part_step[q + 1]; ++st) {
            const PartStep& s = L.steps[st];
            const int rel = st - L.part_step[q];
            if (s.cnt < 1 || s.cnt > kPartStepRows || s.next > kPartExt || s.late > 4 * s.quads) return 1;
            if (s.need > rel || s.need0 > s.need || s.near > s.need || s.lpos + s.cnt > L.rows) return 2;
            most_ext = std::max(most_ext, s.next);
            for (int j = 0; j < s.next; ++j) {
                const int p = L.ext[s.ext0 + j];
                if (p < 0 || p >= first || std::isnan(xp[p])) return 3;   // solved by an earlier part
                lds[1 + (rel % waves) * kPartExt + j] = xp[p];
            }
            std::vector<double> out(s.cnt);
            for (int l = 0; l < s.cnt; ++l) {
                const int i = L.order[s.pos0 + l];
                double acc = r[i];
                for (int k = 0; k < 4 * s.quads; ++k) {
                    const bool late = forward ? k >= 4 * s.quads - s.late : k < s.late;
                    const long e = (long)s.ent + 4 * ((long)(k / 4) * s.cnt + l) + k % 4;
                    if (e < kPartPad || e >= L.nent) return 4;
                    const int slot = L.slot[e];
                    if (slot >= L.slots() || std::isnan(lds[slot])) return 5;
                    if (slot >= xb && step_of[slot - xb] >= (late ? s.need : s.need0)) return 6;
                    acc -= (L.src[e] < 0 ? 0.0 : val[L.src[e]]) * lds[slot];
                }
                out[l] = acc / d[i];
            }
            for (int l = 0; l < s.cnt; ++l) {
                lds[xb + s.lpos + l] = xp[s.pos0 + l] = out[l];
                x[L.order[s.pos0 + l]] = out[l];
            }
        }
    }
    info[0] = L.nparts;
    info[1] = L.rows;
    info[2] = (int)L.steps.size();
    info[3] = L.part_step.back() ? (int)L.ext.size() : 0;
    info[4] = most_ext;
    return 0;
}

// the quotient the kernel forms with a reciprocal known in advance (its plain
// operands: neither |s| nor |d| beyond 2^400 nor below 2^-400, or s = 0)
extern "C" void part_quotients(long n, const double* s, const double* d, double* q) {
    for (long i = 0; i < n; ++i) {
        const double y = 1.0 / d[i], q0 = s[i] * y;
        const double q1 = std::fma(std::fma(-q0, d[i], s[i]), y, q0);
        q[i] = std::copysign(std::fma(std::fma(-q1, d[i], s[i]), y, q1), q0);
    }
}
