// Reduction chains on positional integers.
//
// A chain acc = acc + x*y whose sums need rounding spends its time, in residues, on the
// power-of-two scaling (several mixed steps of 30 bits) and on a fresh interval evaluation
// per step. Both are functions of the integer X that the residues stand for: scaling is
// floor(X / 2^b), the new residues and the new evaluation follow from the scaled integer.
// So the chain here holds X as W = N/2 32-bit words (a rounded number is below
// 2^(log2 M / 2 + 1)) and takes every decision of the residue algorithm from it:
//   * whether and by how many bits a product or a sum is rounded, and whether an operand is
//     dropped, depend on the binary exponent of the evaluation's upper bound ev1 alone. ev1
//     lies within a known distance above X / M, so that exponent is the exponent of X / M
//     unless X / M is just below a power of two (about 1 in 10^6 decisions);
//   * the sign of a sum is the sign of the integers (the residue algorithm's interval test and
//     mixed-radix comparison give the same).
// The evaluation itself is needed only at the end of the chain and where a decision is too
// close to call. It is then rebuilt exactly (pos_replay): the evaluation of the last rounded
// X from its residues (rns_eval), then the interval additions of the steps since then, with
// the original operands' evaluations. Results equal the residue chain's bit for bit.
//
// Operands must be normalised as every operation leaves them: X / M below 2^(mp_h + 1) and
// the evaluation within a relative 2^-20 of X / M, residues not below zero. Chains with others (PosOp::bad) and chains
// that cancel exactly to zero are left to the residue arithmetic (kernels_pos.hpp).
#pragma once

#include "bigint.hpp"
#include "group.hpp"

namespace mph {

// an operand of a product
template <int W>
struct PosOp {
    uint32_t x[W];
    int e, s;
    double h;  // X rounded to a double
    bool bad;
};
// operands kept in memory: converted once where they are used by many chains
template <int W>
struct PosRec {
    uint32_t x[W];
    int e, sb;  // sb: sign, plus 2 for an operand that is not normalised
    double h;
};

// running sum, or a product: value (-1)^s X 2^e; le: exponent of the evaluation's upper bound;
// h: X as a double; ae: both bounds of the evaluation lie within ae / M of X / M; nz: the upper
// bound is not zero
template <int W>
struct PosNum {
    uint32_t x[W];
    int e, s, le;
    double h, ae;
    bool nz;
};
// the same with its evaluation
template <int W>
struct PosExact {
    Big<W> x;
    int e, s;
    Er ev0, ev1;
};

constexpr double POS_FRESH = 0x1p-22;  // relative distance of a computed evaluation (below 1e-7 by its accuracy constant)
constexpr double POS_GIVEN = 0x1p-20;  // of an operand's
constexpr double POS_PROD = 0x1.01p-19;  // of a product of two such operands

__device__ __forceinline__ int pos_ilogb(double v) {  // floor(log2 v), v > 0 normal
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_frexp_exp(v) - 1;
#else
    int e;
    frexp(v, &e);
    return e - 1;
#endif
}
template <int W>
__device__ __forceinline__ double pos_double(const uint32_t *x) {
    double h = (double)x[W - 1];
#pragma unroll
    for (int i = W - 2; i >= 0; i--) h = fma(h, 0x1p32, (double)x[i]);
    return h;
}
// x << s, s >= 0, the result below 2^(32 W)
template <int W>
__device__ __forceinline__ void pos_shl(uint32_t *r, const uint32_t *x, int s) {
    const int q = s >> 5, b = s & 31;
#pragma unroll
    for (int i = 0; i < W; i++) r[i] = x[i];
#pragma unroll
    for (int k = 1; k < W; k <<= 1) {
        const bool on = (q & k) != 0;
#pragma unroll
        for (int i = W - 1; i >= 0; i--) r[i] = on ? (i >= k ? r[i - k] : 0u) : r[i];
    }
#pragma unroll
    for (int i = W - 1; i >= 0; i--) {
        const uint32_t lo = i > 0 ? r[i - 1] : 0u;
        r[i] = (uint32_t)(((((uint64_t)r[i] << 32) | lo) << b) >> 32);
    }
}

// the same; U: in registers (the end of a chain), or with rolled loops, for the rare
// out-of-line calls
template <int N, bool U>
__device__ __forceinline__ void pos_eval(const DevConsts *__restrict__ C, const uint32_t *x, Er &lo, Er &up) {
    if constexpr (U) {
        pos_eval_fast<N>(C, x, lo, up);
    } else {
        int d[N];
        loop<N, false>([&](int i) { d[i] = pos_residue<N, Pos<N>::W>(C, x, i); });
        Core<N, 1> k{C, C->pow2, 0};
        k.load();
        rns_eval<N, 1, false, false>(k, d, lo, up, false);
    }
}

// an operand from its residues and scalar fields
template <int N>
__device__ __forceinline__ void pos_operand(const DevConsts *__restrict__ C, const int *d, int s, int e, Er e0, Er e1,
                                            PosOp<Pos<N>::W> &o) {
    constexpr int W = Pos<N>::W;
    uint32_t any = 0;  // its top bit: a residue below zero, which pos_from_digits does not take
#pragma unroll
    for (int r = 0; r < N; r++) any |= (uint32_t)d[r];
    pos_from_digits<N, W, true>(C, d, o.x);
    o.e = e;
    o.s = s;
    o.h = pos_double<W>(o.x);
    const double f = o.h * pos_const(C->pinv);
    const double u = ldexp(e1.frac, e1.exp), l = ldexp(e0.frac, e0.exp);
    const bool zero = o.h == 0;
    const bool fits = e1.exp <= pos_const(C->mp_h) && u >= f * (1 - 0x1p-44) && u <= f * (1 + POS_GIVEN) &&
                      l <= f * (1 + 0x1p-44) && l >= f * (1 - POS_GIVEN);
    o.bad = (int)any < 0 || (zero ? (e1.frac != 0 || e0.frac != 0) : !fits);
}
template <int W>
__device__ __forceinline__ PosOp<W> pos_unpack(const PosRec<W> &r) {
    PosOp<W> o;
#pragma unroll
    for (int i = 0; i < W; i++) o.x[i] = r.x[i];
    o.e = r.e;
    o.s = r.sb & 1;
    o.h = r.h;
    o.bad = (r.sb & 2) != 0;
    return o;
}

// p = x * y rounded as cuda::mp_mul rounds it; false when a decision is too close to call
template <int N>
__device__ __forceinline__ bool pos_mul(const DevConsts *__restrict__ C, const PosOp<Pos<N>::W> &x,
                                        const PosOp<Pos<N>::W> &y, PosNum<Pos<N>::W> &p) {
    constexpr int W = Pos<N>::W;
    p.s = x.s ^ y.s;
    p.e = x.e + y.e;
    const double h = x.h * y.h;
    p.nz = h != 0;
    const double g = h * pos_const(C->pinv);
    int le = p.nz ? pos_ilogb(g * (1 + POS_PROD)) : -(1 << 28);
    bool sure = !p.nz || pos_ilogb(g * (1 - 0x1p-46)) == le;
    int b = le - pos_const(C->mp_h) + 1;
    b = (b > 0) ? b : 0;
    // the 2W-word product
    uint32_t z[2 * W];
#pragma unroll
    for (int i = 0; i < 2 * W; i++) z[i] = 0;
#pragma unroll
    for (int i = 0; i < W; i++) {
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < W; j++) {
            c += (uint64_t)x.x[i] * y.x[j] + z[i + j];
            z[i + j] = (uint32_t)c;
            c >>= 32;
        }
        z[i + W] = (uint32_t)c;
    }
    if (b > 0) {
        bool dr;
        uint32_t t[2 * W];
        pos_shr<2 * W>(t, z, b, dr);
#pragma unroll
        for (int i = 0; i < W; i++) p.x[i] = t[i];
        p.e += b;
        p.h = pos_double<W>(p.x);
        p.ae = p.h * POS_FRESH;
        const double f = p.h * pos_const(C->pinv);
        le = pos_ilogb(f * (1 + POS_FRESH));
        sure = sure && pos_ilogb(f * (1 - 0x1p-46)) == le;
    } else {
#pragma unroll
        for (int i = 0; i < W; i++) p.x[i] = z[i];
        p.h = h;
        p.ae = h * POS_PROD;
    }
    p.le = le;
    return sure;
}

template <int W>
__device__ __forceinline__ void pos_zero(PosNum<W> &a) {
#pragma unroll
    for (int i = 0; i < W; i++) a.x[i] = 0;
    a.e = a.s = 0;
    a.le = -(1 << 28);
    a.h = a.ae = 0.0;
    a.nz = false;
}

// acc = acc + p as cuda::mp_add (alignment, drop rules, rounding). 0: done without rounding,
// 1: done and rounded (acc's evaluation is that of its integer alone), -1: a decision is too
// close to call, acc unchanged.
template <int N>
__device__ __forceinline__ int pos_add(const DevConsts *__restrict__ C, PosNum<Pos<N>::W> &acc,
                                       const PosNum<Pos<N>::W> &p) {
    constexpr int W = Pos<N>::W;
    const int dexp = acc.e - p.e;
    int ga = dexp > 0 ? dexp : 0, th = dexp < 0 ? -dexp : 0;
    const int mpj = pos_const(C->mp_j);
    const bool nzx = !p.nz || th + p.le < mpj;      // acc kept
    const bool nzy = !acc.nz || ga + acc.le < mpj;  // p kept
    ga = nzy ? ga : 0;
    th = nzx ? th : 0;
    const int ex = nzx ? acc.e - ga : 0, ey = nzy ? p.e - th : 0;
    const int E = ex == 0 ? ey : ex;
    // the shifted operand A and the other, B (at most one shift is nonzero)
    const bool sw = ga > 0;  // acc is shifted
    const int sh = ga + th;
    uint32_t a[W], b[W];
    const uint32_t ka = nzx ? ~0u : 0u, kp = nzy ? ~0u : 0u;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint32_t u = acc.x[i] & ka, v = p.x[i] & kp;
        a[i] = sw ? u : v;
        b[i] = sw ? v : u;
    }
    const double hx = nzx ? acc.h : 0.0, hp = nzy ? p.h : 0.0, axe = nzx ? acc.ae : 0.0, ape = nzy ? p.ae : 0.0;
    const double hA = ldexp(sw ? hx : hp, sh), hB = sw ? hp : hx;
    const double err = ldexp(sw ? axe : ape, sh) + (sw ? ape : axe);
    const bool sub = acc.s != p.s;
    const double sum = hA + hB, base = sub ? fabs(hA - hB) : sum;
    const bool zero = sum == 0 && !acc.nz && !p.nz;  // both operands zero
    const double tot = err + sum * 0x1p-49;
    if (!(base > 2 * tot) && !zero) return -1;  // near-cancellation: the interval may straddle zero
    const double pinv = pos_const(C->pinv);
    int le = pos_ilogb((base + tot) * pinv * (1 + 0x1p-46));
    if (pos_ilogb((base - sum * 0x1p-49) * pinv * (1 - 0x1p-46)) != le && !zero) return -1;
    int r = le - pos_const(C->mp_h) + 1;
    r = (r > 0 && !zero) ? r : 0;
    const int s1 = r < sh ? r : sh;
    bool rem;
    uint32_t bq[W], a1[W], t[W];
    pos_shr<W>(bq, b, s1, rem);
    pos_shl<W>(a1, a, sh - s1);
    const bool neg = sub && hA < hB;
    // floor of the magnitude: A + B, A - ceil(B) or floor(B) - A at the scale 2^s1
    uint32_t carry = (sub && (neg || !rem)) ? 1u : 0u;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint32_t u = neg ? bq[i] : a1[i];
        uint32_t v = neg ? a1[i] : bq[i];
        v = sub ? ~v : v;
        const uint64_t q = (uint64_t)u + v + carry;
        t[i] = (uint32_t)q;
        carry = (uint32_t)(q >> 32);
    }
    const int s2 = r - s1;  // below 32: both operands are normalised
    uint32_t y[W];
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint32_t hi = i + 1 < W ? t[i + 1] : 0u;
        y[i] = (uint32_t)((((uint64_t)hi << 32) | t[i]) >> s2);
    }
    const double h = pos_double<W>(y);
    double ae = tot;
    if (r > 0) {
        const double f = h * pinv;
        le = pos_ilogb(f * (1 + POS_FRESH));
        if (pos_ilogb(f * (1 - 0x1p-46)) != le) return -1;
        ae = h * POS_FRESH;
    }
    const int sa = sw ? acc.s : p.s, sb = sw ? p.s : acc.s;
    // a dropped or zero operand leaves the other's sign
    acc.s = zero ? 0 : (sub ? (neg ? sb : sa) : sa);
#pragma unroll
    for (int i = 0; i < W; i++) acc.x[i] = y[i];
    acc.e = E + r;
    acc.le = zero ? -(1 << 28) : le;
    acc.h = h;
    acc.ae = zero ? 0.0 : ae;
    acc.nz = !zero;
    return r > 0 ? 1 : 0;
}

// ---------------------------------------------------------------- exact steps
// acc = acc + p with the evaluations (Grp::add on integers)
template <int N, bool U>
__device__ __forceinline__ void pos_add_exact(const DevConsts *__restrict__ C, PosExact<Pos<N>::W> &acc,
                                              const PosExact<Pos<N>::W> &p) {
    constexpr int W = Pos<N>::W;
    const Align a = align_sc(pos_const(C->mp_j), acc.s, acc.e, acc.ev0, acc.ev1, p.s, p.e, p.ev0, p.ev1);
    Er e0, e1;
    er_add_pair(a.sx ? a.x1 : a.x0, a.sy ? a.y1 : a.y0, a.sx ? a.x0 : a.x1, a.sy ? a.y0 : a.y1, e0, e1);
    Big<2 * W> x = big_widen<2 * W>(acc.x), y = big_widen<2 * W>(p.x);
    if (!a.nzx) big_zero(x);
    if (!a.nzy) big_zero(y);
    x = big_shl(x, a.gamma);
    y = big_shl(y, a.theta);
    int ts;  // true sign of the sum
    if (a.sx == a.sy) {
        big_add(x, y);
        ts = a.sx;
    } else {
        const int c = big_cmp(x, y);
        ts = c < 0 ? a.sy : a.sx;
        if (c < 0) {
            big_sub(y, x);
            x = y;
        } else {
            big_sub(x, y);
        }
        if (c == 0) ts = 0;
    }
    int sign = e0.frac < 0;
    if (sign != (e1.frac < 0)) {  // the interval straddles zero: the integers decide
        sign = ts;
        const Er u{C->unit_low.frac * (double)(1 - 2 * sign), C->unit_low.exp};
        if (sign)
            e1 = u;
        else
            e0 = u;
    }
    acc.s = sign;
    acc.e = (a.ex == 0) ? a.ey : a.ex;
    if (sign) {
        acc.ev0 = Er{-e1.frac, e1.exp};
        acc.ev1 = Er{-1.0 * e0.frac, e0.exp};
    } else {
        acc.ev0 = e0;
        acc.ev1 = e1;
    }
    int bits = 0;
    if (acc.ev1.frac != 0 && acc.ev1.exp >= pos_const(C->mp_h)) bits = acc.ev1.exp - pos_const(C->mp_h) + 1;
    x = big_shr(x, bits);
#pragma unroll
    for (int i = 0; i < W; i++) acc.x.l[i] = x.l[i];
    if (bits) {
        acc.e += bits;
        pos_eval<N, U>(C, acc.x.l, acc.ev0, acc.ev1);
    }
}
// p = x * y with the evaluation (cuda::mp_mul)
template <int N, bool U>
__device__ __forceinline__ void pos_mul_exact(const DevConsts *__restrict__ C, const PosOp<Pos<N>::W> &x, Er x0, Er x1,
                                              const PosOp<Pos<N>::W> &y, Er y0, Er y1, PosExact<Pos<N>::W> &p) {
    constexpr int W = Pos<N>::W;
    const ScC K = sc_consts(C);
    Sc q;
    sc_mul(K, q, x.s, x.e, x0, x1, y.s, y.e, y0, y1);
    Big<W> a, b;
#pragma unroll
    for (int i = 0; i < W; i++) {
        a.l[i] = x.x[i];
        b.l[i] = y.x[i];
    }
    Big<2 * W> z = big_mul(a, b);
    p.s = q.sign;
    p.e = q.exp;
    p.ev0 = q.ev0;
    p.ev1 = q.ev1;
    int bits = 0;
    if (sc_needs_round(K, q.ev1)) bits = q.ev1.exp - K.mp_h + 1;
    z = big_shr(z, bits);
#pragma unroll
    for (int i = 0; i < W; i++) p.x.l[i] = z.l[i];
    if (bits) {
        p.e += bits;
        pos_eval<N, U>(C, p.x.l, p.ev0, p.ev1);
    }
}
// the fast state of an exact number
template <int N>
__device__ __forceinline__ void pos_from_exact(const DevConsts *__restrict__ C, const PosExact<Pos<N>::W> &v,
                                               PosNum<Pos<N>::W> &a) {
    constexpr int W = Pos<N>::W;
#pragma unroll
    for (int i = 0; i < W; i++) a.x[i] = v.x.l[i];
    a.e = v.e;
    a.s = v.s;
    a.nz = v.ev1.frac != 0;
    a.le = a.nz ? v.ev1.exp : -(1 << 28);
    a.h = pos_double<W>(a.x);
    const double f = a.h * pos_const(C->pinv);
    const double du = fabs(ldexp(v.ev1.frac, v.ev1.exp) - f), dl = fabs(f - ldexp(v.ev0.frac, v.ev0.exp));
    a.ae = a.nz ? (du > dl ? du : dl) * pos_const(C->pmod) * (1 + 0x1p-40) + a.h * 0x1p-45 : 0.0;
}

// The last state of a chain whose evaluation is known, after `at` terms: sign, exponent and
// evaluation (lazy: the evaluation is pos_eval of x)
template <int W>
struct PosSnap {
    uint32_t x[W];
    Sc v;
    long long at;
    bool lazy;
};
template <int W>
__device__ __forceinline__ void pos_snap_zero(PosSnap<W> &s) {
#pragma unroll
    for (int i = 0; i < W; i++) s.x[i] = 0;
    s.v = Sc{0, 0, Er{0.0, 0}, Er{0.0, 0}};
    s.at = 0;
    s.lazy = false;
}
// The evaluation after `to` terms. The terms since the snapshot were added without rounding and
// without a straddling interval, so the scalar fields alone are replayed, each term's loaded a step ahead.
template <int N, bool U, class PV>
__device__ __forceinline__ void pos_replay(const DevConsts *__restrict__ C, const PV &pv, PosSnap<Pos<N>::W> &s,
                                        long long to) {
    if (s.lazy) {
        pos_eval<N, U>(C, s.x, s.v.ev0, s.v.ev1);
        s.lazy = false;
    }
    if (s.at >= to) return;
    typename PV::Scalars cur = pv.scalars(s.at);
    for (; s.at < to; s.at++) {
        const typename PV::Scalars nxt = pv.scalars(s.at + 1 < to ? s.at + 1 : s.at);
        Sc p;
        pv.template product<U>(C, s.at, cur, p);
        cur = nxt;
        const Align a = align_sc(pos_const(C->mp_j), s.v.sign, s.v.exp, s.v.ev0, s.v.ev1, p.sign, p.exp, p.ev0, p.ev1);
        Er e0, e1;
        er_add_pair(a.sx ? a.x1 : a.x0, a.sy ? a.y1 : a.y0, a.sx ? a.x0 : a.x1, a.sy ? a.y0 : a.y1, e0, e1);
        s.v.sign = e0.frac < 0;
        s.v.exp = (a.ex == 0) ? a.ey : a.ex;
        if (s.v.sign) {
            s.v.ev0 = Er{-e1.frac, e1.exp};
            s.v.ev1 = Er{-1.0 * e0.frac, e0.exp};
        } else {
            s.v.ev0 = e0;
            s.v.ev1 = e1;
        }
    }
}
// One step with every decision exact: acc (after `at` terms) plus term `at`. False after an
// exact cancellation: the residue algorithm keeps a positive lower bound for that zero and may
// later take a sum's sign from it, which the integers would not, so the chain is left to it.
// Out of line, with rolled loops: a rare call must not set the register count of the chains.
template <int N, class PV>
__device__ __noinline__ bool pos_step_exact(const DevConsts *__restrict__ C, const PV &pv, PosNum<Pos<N>::W> &acc,
                                            PosSnap<Pos<N>::W> &snap, long long at) {
    constexpr int W = Pos<N>::W;
    pos_replay<N, false>(C, pv, snap, at);
    PosExact<W> v, p;
#pragma unroll
    for (int i = 0; i < W; i++) v.x.l[i] = acc.x[i];
    v.s = snap.v.sign;
    v.e = snap.v.exp;
    v.ev0 = snap.v.ev0;
    v.ev1 = snap.v.ev1;
    pv.template exact<false>(C, at, p);
    pos_add_exact<N, false>(C, v, p);
    pos_from_exact<N>(C, v, acc);
#pragma unroll
    for (int i = 0; i < W; i++) snap.x[i] = acc.x[i];
    snap.v = Sc{v.s, v.e, v.ev0, v.ev1};
    snap.at = at + 1;
    snap.lazy = false;
    return acc.h != 0 || !acc.nz;
}

// one step of a chain: acc and its snapshot after adding term `at`; false: see pos_step_exact
template <int N, class PV>
__device__ __forceinline__ bool pos_step(const DevConsts *__restrict__ C, const PV &pv, PosNum<Pos<N>::W> &acc,
                                         PosSnap<Pos<N>::W> &snap, const PosNum<Pos<N>::W> &p, bool sure,
                                         long long at) {
    constexpr int W = Pos<N>::W;
    const int r = sure ? pos_add<N>(C, acc, p) : -1;
    if (r == 1) {
#pragma unroll
        for (int i = 0; i < W; i++) snap.x[i] = acc.x[i];
        snap.v.exp = acc.e;
        snap.v.sign = acc.s;
        snap.at = at + 1;
        snap.lazy = true;
    } else if (r < 0) {
        // copies, so that the chain's own state stays in registers
        PosNum<W> a = acc;
        PosSnap<W> s = snap;
        const PV v = pv;
        const bool ok = pos_step_exact<N>(C, v, a, s, at);
        acc = a;
        snap = s;
        return ok;
    }
    return true;
}

// ---------------------------------------------------------------- operands converted once
// records of the elements of an m x n operand (leading dimension ld; rec[i + m j])
template <int N, class VM>
__device__ __forceinline__ void pos_load(const DevConsts *__restrict__ C, const VM &X, long long idx,
                                         PosOp<Pos<N>::W> &o, Er &e0, Er &e1) {
    int s, e, d[N];
    scalars_of<N>(X, idx, s, e, e0, e1);
    const int *dp = digits_of<N>(X, idx);
#pragma unroll
    for (int r = 0; r < N; r++) d[r] = dp[r];
    pos_operand<N>(C, d, s, e, e0, e1, o);
}
template <int N, class VM>
__device__ __forceinline__ void pos_record(const DevConsts *__restrict__ C, const VM &X, long long idx,
                                           PosRec<Pos<N>::W> *out) {
    PosOp<Pos<N>::W> o;
    Er e0, e1;
    pos_load<N>(C, X, idx, o, e0, e1);
    PosRec<Pos<N>::W> r;
#pragma unroll
    for (int i = 0; i < Pos<N>::W; i++) r.x[i] = o.x[i];
    r.e = o.e;
    r.sb = o.s | (o.bad ? 2 : 0);
    r.h = o.h;
    *out = r;
}

// Terms of one chain: x from records (RX) or converted from X where it is used, y likewise. Term k
// of the chain is element x0 + k dx of X, record rx0 + k rdx, and so on.
template <int N, class V, bool REC>
struct PosRaw {  // an operand as it lies in memory
    int d[N], s, e;
    Er e0, e1;
};
template <int N, class V>
struct PosRaw<N, V, true> {
    PosRec<Pos<N>::W> r;
};
template <int N, class VX, class VY, bool RX, bool RY>
struct PosTerms {
    static constexpr int W = Pos<N>::W;
    struct Raw {
        PosRaw<N, VX, RX> x;
        PosRaw<N, VY, RY> y;
    };
    VX X;
    VY Y;
    const PosRec<W> *rx, *ry;
    long long x0, dx, y0, dy;      // element indices
    long long rx0, rdx, ry0, rdy;  // record indices
    template <class V, bool REC>
    __device__ __forceinline__ static void load1(const V &v, long long i, const PosRec<W> *rec, long long ri,
                                                 PosRaw<N, V, REC> &o) {
        if constexpr (REC) {
            o.r = rec[ri];
        } else {
            scalars_of<N>(v, i, o.s, o.e, o.e0, o.e1);
            const int *p = digits_of<N>(v, i);
#pragma unroll
            for (int r = 0; r < N; r++) o.d[r] = p[r];
        }
    }
    template <class V, bool REC>
    __device__ __forceinline__ static void convert1(const DevConsts *__restrict__ C, const PosRaw<N, V, REC> &o,
                                                    PosOp<W> &x) {
        if constexpr (REC)
            x = pos_unpack<W>(o.r);
        else
            pos_operand<N>(C, o.d, o.s, o.e, o.e0, o.e1, x);
    }
    // the same terms, the operands as they lie in memory
    __device__ __forceinline__ PosTerms<N, VX, VY, false, false> plain() const {
        return {X, Y, nullptr, nullptr, x0, dx, y0, dy, 0, 0, 0, 0};
    }
    __device__ __forceinline__ Raw load(long long k) const {
        Raw o;
        load1(X, x0 + k * dx, rx, rx0 + k * rdx, o.x);
        load1(Y, y0 + k * dy, ry, ry0 + k * rdy, o.y);
        return o;
    }
    __device__ __forceinline__ void convert(const DevConsts *__restrict__ C, const Raw &o, PosOp<W> &x,
                                            PosOp<W> &y) const {
        convert1(C, o.x, x);
        convert1(C, o.y, y);
    }
    __device__ __forceinline__ void ops(const DevConsts *__restrict__ C, long long k, PosOp<W> &x, PosOp<W> &y) const {
        convert(C, load(k), x, y);
    }
    template <bool U>
    __device__ __forceinline__ void exact(const DevConsts *__restrict__ C, long long k, PosExact<W> &p) const {
        PosOp<W> x, y;
        ops(C, k, x, y);
        int s, e;
        Er a0, a1, b0, b1;
        scalars_of<N>(X, x0 + k * dx, s, e, a0, a1);
        scalars_of<N>(Y, y0 + k * dy, s, e, b0, b1);
        pos_mul_exact<N, U>(C, x, a0, a1, y, b0, b1, p);
    }
    struct Scalars {
        int xs, xe, ys, ye;
        Er a0, a1, b0, b1;
    };
    __device__ __forceinline__ Scalars scalars(long long k) const {
        Scalars o;
        scalars_of<N>(X, x0 + k * dx, o.xs, o.xe, o.a0, o.a1);
        scalars_of<N>(Y, y0 + k * dy, o.ys, o.ye, o.b0, o.b1);
        return o;
    }
    // sign, exponent and evaluation of term k from its operands' fields
    template <bool U>
    __device__ __forceinline__ void product(const DevConsts *__restrict__ C, long long k, const Scalars &o,
                                            Sc &p) const {
        const ScC K = sc_consts(C);
        sc_mul(K, p, o.xs, o.xe, o.a0, o.a1, o.ys, o.ye, o.b0, o.b1);
        if (sc_needs_round(K, p.ev1)) {
            PosExact<W> q;
            exact<U>(C, k, q);
            p = Sc{q.s, q.e, q.ev0, q.ev1};
        }
    }
};

}  // namespace mph
