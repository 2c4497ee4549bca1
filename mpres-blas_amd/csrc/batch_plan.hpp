// Host side of the batched form: checks the problems as their single calls do,
// splits them into work items and lays out the items' scratch. Pure C++ (no HIP
// calls), so the host tests compile it as it is.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/mpres_hip.h"
#include "ops.hpp"

namespace mph {

inline SoA soa_view(const mp_array_t *a) {
    SoA s;
    s.d = a->digits;
    s.s = a->sign;
    s.e = a->exp;
    s.ev = (ErMem *)a->eval;
    s.lenp = a->len;
    s.len = 0;
    return s;
}

struct BatchLayout {
    std::vector<BatchItem> items;  // in launch order (descending work)
    size_t ws_bytes = 0;
    double fmas = 0;               // multiply-accumulates of the batch
    std::string err;
};

constexpr size_t BATCH_WS_ALIGN = 256;

// Rows per item of a gemv of ly outputs, lx terms each, in block3 chains, where the plan chooses them
// (at most cap): an item is to be no more than 1 / BATCH_PARTS of the batch's multiply-accumulates,
// so that its slowest item does not outlast the others (about two items a compute unit), but gives each
// group of lanes of its workgroup (groups) a chain; the rows are split evenly. Every item forms
// alpha * x again, which costs it lx products beside rows * lx. One gemv of 1024^2 over 16 moduli,
// before in items of 128 rows: 17.2 -> 2.2 ms; 512 gemvs of 48 rows keep one item each (0.26 ms;
// two each 0.34). Every item also holds its own copy of alpha * x: where a batch's copies, beyond those of
// items of cap rows, would take more than BATCH_SPARE (wide gemvs: 512 x 32768 at 106 bits, an
// item a row, 1.2 GB, as much as A), the parts are halved until they do not (parts).
constexpr int BATCH_PARTS = 512;
constexpr double BATCH_SPARE = 256.0 * (1 << 20);
inline int batch_rows(double fmas, int parts_of, int lx, int ly, int block3, int groups, int cap) {
    const double fair = std::ceil(fmas / parts_of / lx);
    const int least = 1 + (groups - 1) / block3;
    int rows = fair < cap ? std::max((int)fair, least) : cap;
    rows = std::min(rows, cap);
    const int parts = 1 + (ly - 1) / rows;
    return 1 + (ly - 1) / parts;
}
// multiply-accumulates of a batch; wide: those of its gemvs with more chains than a workgroup has lanes
inline double batch_fmas(const mpres_batch_problem_t *probs, int count, double &wide) {
    double sum = 0;
    wide = 0;
    for (int i = 0; probs && i < count; i++) {
        const mpres_batch_problem_t &p = probs[i];
        const bool dot = p.op == MPRES_BATCH_DOT;
        const double f = dot ? (p.n > 0 ? p.n : 0) : (p.m > 0 && p.n > 0 ? (double)p.m * p.n : 0);
        sum += f;
        if (!dot && (double)(p.trans == MPRES_NO_TRANS ? p.m : p.n) * p.block3 > 256) wide += f;
    }
    return sum;
}
// Whether a batch over 16 moduli runs one lane a number, its roundings positional: where such gemvs are
// nearly all of it (over 7/8). 1024 dots and gemvs of 32 to 1024 rows 11.9 ms with one lane, 23.7 with 4; 64
// gemvs of 200 rows 0.52 and 0.83 ms (operands that seldom round 0.22 and 0.28). A dot of few chains leaves most
// lanes of its workgroup idle and runs longer for one lane a number: 512 dots of 1 x 64 chains and one gemv of
// 200 rows 0.64 and 0.27 ms, 1024 of them and 512 gemvs of 100 rows (0.77 of the work) 0.96 and 0.57 (rounding
// 1.28 and 1.40).
inline bool batch_one_lane(const mpres_batch_problem_t *probs, int count) {
    double wide;
    const double sum = batch_fmas(probs, count, wide);
    return sum > 0 && wide > 0.875 * sum;
}

// Returns MPRES_OK, or MPRES_ERR_ARG with layout.err naming the first bad problem.
// Problems the single call would skip (dot n <= 0, gemv m or n <= 0) give no item.
// groups > 0: gemv_rows is the most that batch_rows may choose, for workgroups of that many groups
inline int batch_layout(const mpres_batch_problem_t *probs, int count, int n_moduli, int gemv_rows,
                        BatchLayout &out, int groups = 0) {
    out = BatchLayout{};
    const long long S = 4LL * n_moduli + 40;
    char buf[160];
    auto bad = [&](int i, const char *what) {
        std::snprintf(buf, sizeof buf, "batch problem %d: %s", i, what);
        out.err = buf;
        return MPRES_ERR_ARG;
    };
    if (count < 0 || (count > 0 && !probs)) {
        out.err = "invalid problem list";
        return MPRES_ERR_ARG;
    }
    if (gemv_rows <= 0) {
        out.err = "gemv rows per item must be positive";
        return MPRES_ERR_ARG;
    }
    struct Work {
        BatchItem it;
        double work;
        size_t bytes;
    };
    std::vector<Work> v;
    double wide;
    const double total = batch_fmas(probs, count, wide);
    int parts = BATCH_PARTS;
    for (; groups > 0 && parts > 1; parts /= 2) {
        double spare = 0;
        for (int i = 0; i < count; i++) {
            const mpres_batch_problem_t &p = probs[i];
            if (p.op != MPRES_BATCH_GEMV || p.m <= 0 || p.n <= 0 || p.block3 <= 0) continue;
            const bool tr = p.trans != MPRES_NO_TRANS;
            const int lx = tr ? p.m : p.n, ly = tr ? p.n : p.m;
            const auto items = [&](int rows) { return (double)(1 + (ly - 1) / rows); };
            spare += (items(batch_rows(total, parts, lx, ly, p.block3, groups, gemv_rows)) - items(gemv_rows)) * lx;
        }
        if (spare * S <= BATCH_SPARE) break;
    }
    for (int i = 0; i < count; i++) {
        const mpres_batch_problem_t &p = probs[i];
        if (p.op == MPRES_BATCH_DOT) {
            // mpres_dot: src/blas/dot.cuh:84-107
            if (!p.x || !p.y || !p.r) return bad(i, "null argument");
            if (p.n <= 0) continue;
            if (p.grid3 <= 0 || p.block3 <= 0) return bad(i, "invalid reduction shape");
            Work w{};
            w.it.kind = BATCH_DOT;
            w.it.n = p.n;
            w.it.incx = p.incx;
            w.it.incy = p.incy;
            w.it.g3 = p.grid3;
            w.it.b3 = p.block3;
            w.it.x = soa_view(p.x);
            w.it.y = soa_view(p.y);
            w.it.r = soa_view(p.r);
            const long long G = (long long)p.grid3 * p.block3;
            w.bytes = (size_t)((G + p.block3) * S);
            w.work = (double)p.n + (double)G + (double)p.block3;
            out.fmas += p.n;
            v.push_back(w);
        } else if (p.op == MPRES_BATCH_GEMV) {
            // mpres_gemv: src/blas/gemv.cuh:150-268
            if (!p.alpha || !p.A || !p.x || !p.beta || !p.y) return bad(i, "null argument");
            if (p.m <= 0 || p.n <= 0) continue;
            if (p.incx == 0 || p.incy == 0 || p.lda < std::max(1, p.m))
                return bad(i, "invalid increments or leading dimension");
            if (p.block3 <= 0) return bad(i, "invalid blockDim3");
            if (p.trans != MPRES_NO_TRANS && p.trans != MPRES_TRANS && p.trans != MPRES_CONJ_TRANS)
                return bad(i, "invalid trans");
            const bool tr = p.trans != MPRES_NO_TRANS;
            const int lx = tr ? p.m : p.n, ly = tr ? p.n : p.m;
            out.fmas += (double)p.m * p.n;
            const int rows = groups > 0 ? batch_rows(total, parts, lx, ly, p.block3, groups, gemv_rows) : gemv_rows;
            for (int r0 = 0; r0 < ly; r0 += rows) {
                const int r1 = ly - r0 > rows ? r0 + rows : ly, h = r1 - r0;
                Work w{};
                w.it.kind = tr ? BATCH_GEMV_T : BATCH_GEMV_N;
                w.it.r0 = r0;
                w.it.r1 = r1;
                w.it.m = p.m;
                w.it.n = p.n;
                w.it.lda = p.lda;
                w.it.incx = p.incx;
                w.it.incy = p.incy;
                w.it.b3 = p.block3;
                w.it.alpha = soa_view(p.alpha);
                w.it.A = soa_view(p.A);
                w.it.x = soa_view(p.x);
                w.it.beta = soa_view(p.beta);
                w.it.y = soa_view(p.y);
                w.bytes = (size_t)(((long long)lx + (long long)h * p.block3) * S);
                w.work = (double)h * lx + (double)lx + (double)h * p.block3;
                v.push_back(w);
            }
        } else {
            return bad(i, "unknown operation");
        }
    }
    std::stable_sort(v.begin(), v.end(), [](const Work &a, const Work &b) { return a.work > b.work; });
    size_t off = 0;
    out.items.reserve(v.size());
    for (auto &w : v) {
        w.it.ws = (long long)off;
        off += (w.bytes + BATCH_WS_ALIGN - 1) / BATCH_WS_ALIGN * BATCH_WS_ALIGN;
        out.items.push_back(w.it);
    }
    out.ws_bytes = off;
    return MPRES_OK;
}

}  // namespace mph
