// Reduction kernels on positional integers (pos.hpp), one chain per group of G lanes.
//
// With G = 4 the four lanes of a quad each form the product of one of the chain's next four
// terms, and then add the four in order, each lane the same sum: the conversion of the
// operands, which is most of a step's work, runs in parallel, and the products reach the other
// lanes by quad permutations (DPP, no LDS). That serves calls with few chains. With G = 1 a
// lane does a whole chain, for calls with enough of them to fill the chip.
// What bounds them is the serial chain: 1560 vector instructions a wave for four terms of its quads
// (a product a lane, four sums), issued by one or two waves per SIMD. Against the residue chains over 8 moduli: dot of 2^24
// terms in 256 x 64 chains 6.12 -> 1.18 ms, A^T x of a 1501 x 777 matrix in 24864 chains
// 697 -> 150 us.
#pragma once

#include "kernels.hpp"
#include "pos.hpp"

namespace mph {

#if defined(__HIPCC__)
#define POS_WAVES(n) __attribute__((amdgpu_waves_per_eu(n)))
#else
#define POS_WAVES(n)
#endif

template <int U>
__device__ __forceinline__ int quad_lane(int v) {  // the value of lane U of the quad
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_update_dpp(0, v, U * 0x55, 0xF, 0xF, false);
#else
    return v;
#endif
}
template <int U>
__device__ __forceinline__ double quad_lane_d(double v) {
    const uint64_t u = d2u(v);
    return u2d(((uint64_t)(uint32_t)quad_lane<U>((int)(uint32_t)(u >> 32)) << 32) |
               (uint32_t)quad_lane<U>((int)(uint32_t)u));
}
// the constants through a pointer that the compiler must take as new: a loop's table entries
// are read from the scalar cache where they are used instead of being held (and spilled) in
// scalar registers over the whole chain
__device__ __forceinline__ const DevConsts *pos_fresh(const DevConsts *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(p));
#endif
    return p;
}
__device__ __forceinline__ bool wave_any(bool v) {  // of the lanes that are active
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ballot_w64(v) != 0;
#else
    return v;
#endif
}
// product of a term as the lanes of a group exchange it
template <int W>
struct PosTerm {
    PosNum<W> p;
    bool sure, bad;
};
template <int G, int U, int W>
__device__ __forceinline__ PosTerm<W> group_term(const PosTerm<W> &t) {
    if constexpr (G == 1) {
        return t;
    } else {
        PosTerm<W> r;
#pragma unroll
        for (int i = 0; i < W; i++) r.p.x[i] = (uint32_t)quad_lane<U>((int)t.p.x[i]);
        r.p.e = quad_lane<U>(t.p.e);
        r.p.le = quad_lane<U>(t.p.le);
        r.p.h = quad_lane_d<U>(t.p.h);
        r.p.ae = quad_lane_d<U>(t.p.ae);
        const int f = quad_lane<U>(t.p.s | (t.p.nz ? 2 : 0) | (t.sure ? 4 : 0) | (t.bad ? 8 : 0));
        r.p.s = f & 1;
        r.p.nz = (f & 2) != 0;
        r.sure = (f & 4) != 0;
        r.bad = (f & 8) != 0;
        return r;
    }
}

// a sum whose interval straddles zero: decided by mixed-radix digits, out of line
template <int N, int G>
__device__ __noinline__ void pos_straddle(const DevConsts *C, MP<N / G> *a, const MP<N / G> *p) {
    const Grp<N, G> g(uniform_ptr(C));
    MP<N / G> x = *a, y = *p, r;
    g.template add<false, false>(r, x, y);
    *a = r;
}
// The chain from its start in residues (the usual arithmetic, Grp), N / G residues a lane, up to the first
// step that rounds; the chains of a wave stop together (apart, they would take turns). As in the
// positional steps, a group's lanes form the products of its next G terms and then add them in order.
// The terms done: cnt when the chain ended (its result is in out[i]), otherwise the sum is in acc and its
// snapshot (unchanged for 0 terms). -1, and nothing done, for a chain that this and the positional steps cannot do: a rounding after
// an exact cancellation, or operands whose evaluations are not their numbers'; without PAST0, for every
// exact cancellation.
template <int N, int G, bool PAST0, class PV>
__device__ __forceinline__ long long pos_quiet(const DevConsts *__restrict__ C0, const PV &pv,
                                               PosNum<Pos<N>::W> &acc, PosSnap<Pos<N>::W> &snap, long long cnt,
                                               AoSRef<N> out, long long i) {
    constexpr int W = Pos<N>::W, R = N / G;
    const int l = G == 1 ? 0 : (int)(threadIdx.x & (G - 1));
    const Grp<N, G> g(C0);
    const Grp<N, 1> g1(C0);
    MP<R> a;
    g.zero(a);
    bool own = true;  // no exact cancellation yet: the evaluation is the sum's
    const auto pq = pv.plain();
    typename decltype(pq)::Raw cur = pq.load(l < cnt ? l : cnt - 1);
    for (long long k = 0; k < cnt; k += G) {
        const DevConsts *C = pos_fresh(C0);
        const long long kn = k + G + l;
        const typename decltype(pq)::Raw nxt = pq.load(kn < cnt ? kn : cnt - 1);
        // term k + l
        Sc q;
        int d[N];
        sc_mul(g1.K, q, cur.x.s, cur.x.e, cur.x.e0, cur.x.e1, cur.y.s, cur.y.e, cur.y.e0, cur.y.e1);
        g1.product(cur.x.d, cur.y.d, 0.0, false, C, [&](int r, int v) { d[r] = v; });
        int stop = -1;  // step of the group at which the chain leaves
        bool lost = false;
        auto step = [&](auto lane, int u) {
            constexpr int U = decltype(lane)::value;
            if (k + u >= cnt || stop >= 0 || lost) return;
            MP<R> p;
            if constexpr (G == 1) {
#pragma unroll
                for (int r = 0; r < R; r++) p.d[r] = d[r];
                p.sign = q.sign;
                p.exp = q.exp;
                p.ev0 = q.ev0;
                p.ev1 = q.ev1;
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    int v = quad_lane<U>(d[r]);
#pragma unroll
                    for (int t = 1; t < G; t++) {
                        const int o = quad_lane<U>(d[t * R + r]);
                        v = l == t ? o : v;
                    }
                    p.d[r] = v;
                }
                p.sign = quad_lane<U>(q.sign);
                p.exp = quad_lane<U>(q.exp);
                p.ev0 = Er{quad_lane_d<U>(q.ev0.frac), quad_lane<U>(q.ev0.exp)};
                p.ev1 = Er{quad_lane_d<U>(q.ev1.frac), quad_lane<U>(q.ev1.exp)};
            }
            const Align al = g.align(a, p);
            Er e0, e1;
            er_add_pair(al.sx ? al.x1 : al.x0, al.sy ? al.y1 : al.y0, al.sx ? al.x0 : al.x1, al.sy ? al.y0 : al.y1, e0,
                        e1);
            const int sign = e0.frac < 0;
            const bool straddles = sign != (e1.frac < 0);
            const bool rounds = g.needs_round(p) || (!straddles && sc_needs_round(g.K, sign ? e0 : e1));
            if (wave_any(rounds && own) && own) {
                stop = u;
                return;
            }
            lost = rounds;
            const bool shx = al.gamma > 0;
            const int sh = al.gamma + al.theta, row = g.prow(sh);
            const int fs = shx ? al.fx : al.fy, fo = shx ? al.fy : al.fx;
            int t[R];
            uint32_t any = 0;
#pragma unroll
            for (int r = 0; r < R; r++) {
                t[r] = g.combine(a.d[r], p.d[r], row, shx, sh != 0, fs, fo, straddles ? 0 : sign, r, C);
                any |= (uint32_t)t[r];
            }
            if (straddles && !rounds) {
                if constexpr (G == 4) any |= (uint32_t)xchg<1>((int)any), any |= (uint32_t)xchg<2>((int)any);
                if (any != 0) {
                    MP<R> x = a, y = p;
                    pos_straddle<N, G>(C0, &x, &y);
                    a = x;
                    lost = g.needs_round(a);
                    return;
                }
                // an exact cancellation (Grp::add): sign 0, the smallest lower bound
                e0 = g.unit_low();
                own = false;
                lost = !PAST0;
            }
#pragma unroll
            for (int r = 0; r < R; r++) a.d[r] = t[r];
            a.sign = straddles ? 0 : sign;
            a.exp = (al.ex == 0) ? al.ey : al.ex;
            a.ev0 = a.sign ? Er{-e1.frac, e1.exp} : e0;
            a.ev1 = a.sign ? Er{-1.0 * e0.frac, e0.exp} : e1;
            lost = lost || (straddles && g.needs_round(a));
        };
        step(std::integral_constant<int, 0>{}, 0);
        if constexpr (G == 4) {
            step(std::integral_constant<int, 1>{}, 1);
            step(std::integral_constant<int, 2>{}, 2);
            step(std::integral_constant<int, 3>{}, 3);
        }
        if (lost) return -1;
        if (stop >= 0) {
            if (k == 0) return 0;  // within the first terms: done again
            int t[N];
#pragma unroll
            for (int r = 0; r < R; r++) {
                if constexpr (G == 4) {
                    t[r] = quad_lane<0>(a.d[r]);
                    t[R + r] = quad_lane<1>(a.d[r]);
                    t[2 * R + r] = quad_lane<2>(a.d[r]);
                    t[3 * R + r] = quad_lane<3>(a.d[r]);
                } else {
                    t[r] = a.d[r];
                }
            }
            PosExact<W> v;
            pos_from_digits<N, W, true>(C, t, v.x.l);
            const double f = pos_double<W>(v.x.l) * pos_const(C->pinv);
            const double lo = ldexp(a.ev0.frac, a.ev0.exp), up = ldexp(a.ev1.frac, a.ev1.exp);
            if ((a.ev1.frac != 0 && a.ev1.exp > pos_const(C->mp_h)) || lo > f * (1 + 0x1p-44) || up < f * (1 - 0x1p-44))
                return -1;
#pragma unroll
            for (int w = 0; w < W; w++) snap.x[w] = v.x.l[w];
            v.s = a.sign;
            v.e = a.exp;
            v.ev0 = a.ev0;
            v.ev1 = a.ev1;
            pos_from_exact<N>(C, v, acc);
            snap.v = Sc{v.s, v.e, v.ev0, v.ev1};
            snap.at = k + stop;
            snap.lazy = false;
            return snap.at;
        }
        cur = nxt;
    }
    store_aos(g, a, out, i);
    return cnt;
}
// the rest of a chain, from its snapshot, in residues with every rounding, out of line
template <int N, int G, class PV>
__device__ __noinline__ void pos_finish(const DevConsts *C0, const PV &pv, PosSnap<Pos<N>::W> &snap, long long cnt,
                                        AoSRef<N> out, long long i) {
    constexpr int W = Pos<N>::W, R = N / G;
    const DevConsts *C = uniform_ptr(C0);
    const Grp<N, G> g(C);
    MP<R> a;
    uint32_t x[W];
#pragma unroll
    for (int q = 0; q < W; q++) x[q] = snap.x[q];
#pragma unroll
    for (int q = 0; q < N; q++) {  // the constants are read wave-uniformly: every lane forms all
        const int v = pos_residue<N, W>(C, x, q);
        if (q / R == g.lane()) a.d[q % R] = v;
    }
    a.sign = snap.v.sign;
    a.exp = snap.v.exp;
    a.ev0 = snap.v.ev0;
    a.ev1 = snap.v.ev1;
    if (snap.lazy) pos_eval<N, true>(C, x, a.ev0, a.ev1);
    for (long long k = snap.at; k < cnt; k++)
        g.template fma_step<true>(a, pv.X, pv.x0 + k * pv.dx, pv.Y, pv.y0 + k * pv.dy);
    store_aos(g, a, out, i);
}

// The chain of terms 0 .. cnt - 1 of pv by the group's lanes (all of them take part and hold the same
// state); its result to out[i]. PART POS_BOTH: it starts in residues (pos_quiet) and changes to positional steps where
// the first step rounds: sums that never round (integers, doubles of few bits, zeros) cost no more than a
// chain in residues, and their evaluation need not be replayed from the operands (dot of 2^22
// integers 2.10 -> 0.40 ms, in residues alone 0.38; of 2^22 numbers that round 0.40 -> 0.38, gemv of 2048^2
// 0.27 -> 0.285, where the chains read their first terms twice). A chain that neither can do, an operand outside the positional form, or an
// exact cancellation after the change: a quad finishes the chain in residues, a single lane marks it
// REDO for the residue kernels. With one lane a chain the two are kernels of their own, since in one the
// residues' registers leave room for half the waves: POS_QUIET, which marks a chain with a step that
// rounds REDO, then POS_ONLY over the chains marked.
enum { POS_BOTH, POS_QUIET, POS_ONLY };
template <int N, int G, int PART = POS_BOTH, class PV>
__device__ __forceinline__ void pos_group_chain(const DevConsts *__restrict__ C0, const PV &pv, long long cnt,
                                                AoSRef<N> out, long long i) {
    static_assert(G == 1 || G == 4, "a lane or a quad");
    constexpr int W = Pos<N>::W;
    const int l = G == 1 ? 0 : (int)(threadIdx.x & (G - 1));
    if (cnt <= 0) {  // an empty chain is zero
        if (l == 0) {
            int *p = (int *)(out.base + i * AoSRef<N>::STRIDE);
#pragma unroll
            for (int q = 0; q < N + 10; q++) p[q] = 0;
        }
        return;
    }
    PosNum<W> acc;
    PosSnap<W> snap;
    pos_zero(acc);
    pos_snap_zero(snap);
    long long k = 0;
    if constexpr (N <= 8 && PART != POS_ONLY) {
        k = pos_quiet<N, G, (G > 1 || PART == POS_QUIET)>(C0, pv, acc, snap, cnt, out, i);
        if (k >= cnt) return;
        if constexpr (PART == POS_QUIET) {
            if (l == 0) *out.sign(i) = REDO;
            return;
        }
    }
    bool ok = k >= 0;
    const long long k0 = (ok ? k : 0) + l;
    typename PV::Raw cur = pv.load(k0 < cnt ? k0 : cnt - 1);
    for (; ok && k < cnt; k += G) {
        const DevConsts *C = pos_fresh(C0);
        const long long kn = k + G + l;
        const typename PV::Raw nxt = pv.load(kn < cnt ? kn : cnt - 1);
        PosTerm<W> t;
        {
            PosOp<W> x, y;
            pv.convert(C, cur, x, y);
            t.bad = x.bad || y.bad;
            t.sure = pos_mul<N>(C, x, y, t.p);
        }
        auto step = [&](const PosTerm<W> &q, long long at) {
            if (!ok || at >= cnt) return;
            ok = !q.bad && pos_step<N>(C, pv, acc, snap, q.p, q.sure, at);
        };
        step(group_term<G, 0, W>(t), k);
        if constexpr (G == 4) {
            step(group_term<G, 1, W>(t), k + 1);
            step(group_term<G, 2, W>(t), k + 2);
            step(group_term<G, 3, W>(t), k + 3);
        }
        cur = nxt;
    }
    if (!ok) {
        if constexpr (G == 4) {
            PosSnap<W> s = snap;  // copies, so that the chain's own state stays in registers
            const PV v = pv;
            pos_finish<N, G>(C0, v, s, cnt, out, i);
        } else {
            *out.sign(i) = REDO;
        }
        return;
    }
    const DevConsts *C = pos_fresh(C0);
    pos_replay<N, true>(C, pv, snap, cnt);
    int *d = out.digits(i);
#pragma unroll
    for (int r = 0; r < N; r++)
        if (G == 1 || r % G == l) d[r] = pos_residue<N, W>(C, acc.x, r);
    if (l == 0) {
        *out.sign(i) = snap.v.sign;
        *out.exp(i) = snap.v.exp;
        ErMem *ev = out.eval(i);
        ev[0] = ErMem{snap.v.ev0.frac, (long long)snap.v.ev0.exp};
        ev[1] = ErMem{snap.v.ev1.frac, (long long)snap.v.ev1.exp};
    }
}

// records of count numbers: record i + rows j is element idx(i, j) of X
template <int N, class VM, int SIDE>
__global__ __launch_bounds__(BLK) void k_pos_records(const DevConsts *__restrict__ C, int cnt, int k, int t, VM X,
                                                     int ld, PosRec<Pos<N>::W> *out) {
    if constexpr (std::is_same<VM, SoA>::value) X = rd(X);
    const long long g = (long long)blockIdx.x * BLK + threadIdx.x;
    if (g >= (long long)cnt * k) return;
    // op(A): row j fastest; op(B): index i along k fastest
    const int j = SIDE == 0 ? (int)(g % cnt) : (int)(g / k), i = SIDE == 0 ? (int)(g / cnt) : (int)(g % k);
    pos_record<N>(C, X, op_index<SIDE>(t, j, i, ld), out + g);
}

// dot, first pass: chain v takes terms v, v + nvt, ... (k_fold). MODE 0: SoA with increments, 1: AoS
template <int N, int G, int MODE, int PART>
__global__ __launch_bounds__(BLK) POS_WAVES(2) void k_pos_fold(const DevConsts *__restrict__ C, long long cnt, long long nvt, SoA xs,
                                                  int incx, SoA ys, int incy, AoSRef<N> xa, AoSRef<N> ya,
                                                  AoSRef<N> out) {
    const long long v = ((long long)blockIdx.x * BLK + threadIdx.x) / G;
    if (v >= nvt) return;
    if (PART == POS_ONLY && *out.sign(v) != REDO) return;
    const long long n = v < cnt ? (cnt - v + nvt - 1) / nvt : 0;
    if constexpr (MODE == 0) {
        xs = rd(xs);
        ys = rd(ys);
        const PosTerms<N, SoA, SoA, false, false> pv{xs, ys, nullptr, nullptr, bidx(v, cnt, incx),
                                                     nvt * (long long)incx, bidx(v, cnt, incy),
                                                     nvt * (long long)incy, 0, 0, 0, 0};
        pos_group_chain<N, G, PART>(C, pv, n, out, v);
    } else {
        const PosTerms<N, AoSRef<N>, AoSRef<N>, false, false> pv{xa, ya, nullptr, nullptr, v, nvt, v, nvt, 0, 0, 0, 0};
        pos_group_chain<N, G, PART>(C, pv, n, out, v);
    }
}

// gemv partials (k_gemv_fold): RY: bx also as records
template <int N, int G, bool TRANS, bool RY, int PART>
__global__ __launch_bounds__(BLK) POS_WAVES(2) void k_pos_gemv(const DevConsts *__restrict__ C, int m, int n, SoA A, int lda,
                                                  AoSRef<N> bx, const PosRec<Pos<N>::W> *__restrict__ rb, int b3,
                                                  long long nvt, AoSRef<N> part) {
    A = rd(A);
    const long long gid = ((long long)blockIdx.x * BLK + threadIdx.x) / G;
    if (gid >= nvt) return;
    const long long ly = nvt / b3;
    const long long o = TRANS ? gid / b3 : gid % ly;
    const int t = (int)(TRANS ? gid % b3 : gid / ly);
    const long long v = o * b3 + t;
    if (PART == POS_ONLY && *part.sign(v) != REDO) return;
    const int len = TRANS ? m : n;
    const long long cnt = t < len ? ((long long)len - t + b3 - 1) / b3 : 0;
    const PosTerms<N, SoA, AoSRef<N>, false, RY> pv{A,
                                                    bx,
                                                    nullptr,
                                                    rb,
                                                    TRANS ? o * lda + t : (long long)t * lda + o,
                                                    TRANS ? (long long)b3 : (long long)b3 * lda,
                                                    t,
                                                    b3,
                                                    0,
                                                    0,
                                                    t,
                                                    b3};
    pos_group_chain<N, G, PART>(C, pv, cnt, part, v);
}

// gemm sums (k_gemm_sum): REC: operands from the records of op(A) (rows fastest) and op(B)
template <int N, int G, bool REC, int PART, class VM>
__global__ __launch_bounds__(BLK) POS_WAVES(PART == POS_ONLY ? 4 : 2) void k_pos_gemm(
    const DevConsts *__restrict__ C, int ta, int tb, int m, int n, int k, VM A, int lda, VM B, int ldb,
    const PosRec<Pos<N>::W> *__restrict__ ra, const PosRec<Pos<N>::W> *__restrict__ rb, AoSRef<N> sums) {
    if constexpr (std::is_same<VM, SoA>::value) {
        A = rd(A);
        B = rd(B);
    }
    const long long e = ((long long)blockIdx.x * BLK + threadIdx.x) / G;
    if (e >= (long long)m * n) return;
    if (PART == POS_ONLY && *sums.sign(e) != REDO) return;
    const int row = (int)(e % m), col = (int)(e / m);
    const long long a0 = op_index<0>(ta, row, 0, lda), b0 = op_index<1>(tb, col, 0, ldb);
    const PosTerms<N, VM, VM, REC, REC> pv{A,  B,  ra,
                                           rb, a0, ta ? 1LL : (long long)lda,
                                           b0, tb ? (long long)ldb : 1LL,
                                           row, m, (long long)col * k,
                                           1};
    pos_group_chain<N, G, PART>(C, pv, k, sums, e);
}

}  // namespace mph
