// Reduction kernels on positional integers (pos.hpp), one chain per group of G lanes.
//
// With G = 4 the four lanes of a quad each form the product of one of the chain's next four
// terms, and then add the four in order, each lane the same sum: the conversion of the
// operands, which is most of a step's work, runs in parallel, and the products reach the other
// lanes by quad permutations (DPP, no LDS). That serves calls with few chains. With G = 1 a
// lane does a whole chain, for calls with enough of them to fill the chip.
// What bounds them is the serial chain: about 290 vector instructions a sum and 190 a product,
// issued by one or two waves per SIMD. Against the residue chains over 8 moduli: dot of 2^24
// terms in 256 x 64 chains 6.12 -> 1.50 ms, A^T x of a 1501 x 777 matrix in 24864 chains
// 686 -> 126 us.
// FIX: only chains marked REDO in their output are done; chains that the positional form
// cannot do (pos.hpp) are marked REDO for the residue kernels.
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

// the chain of terms 0 .. cnt - 1 of pv by the group's lanes (all of them take part and hold
// the same state); its result, or REDO, to out[i]
template <int N, int G, class PV>
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
    bool ok = true;
    typename PV::Raw cur = pv.load(l < cnt ? l : cnt - 1);
    for (long long k = 0; k < cnt && ok; k += G) {
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
        if (l == 0) *out.sign(i) = REDO;
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
template <int N, int G, int MODE, bool FIX>
__global__ __launch_bounds__(BLK) POS_WAVES(2) void k_pos_fold(const DevConsts *__restrict__ C, long long cnt, long long nvt, SoA xs,
                                                  int incx, SoA ys, int incy, AoSRef<N> xa, AoSRef<N> ya,
                                                  AoSRef<N> out) {
    const long long v = ((long long)blockIdx.x * BLK + threadIdx.x) / G;
    if (v >= nvt) return;
    if (FIX && *out.sign(v) != REDO) return;
    const long long n = v < cnt ? (cnt - v + nvt - 1) / nvt : 0;
    if constexpr (MODE == 0) {
        xs = rd(xs);
        ys = rd(ys);
        const PosTerms<N, SoA, SoA, false, false> pv{xs, ys, nullptr, nullptr, bidx(v, cnt, incx),
                                                     nvt * (long long)incx, bidx(v, cnt, incy),
                                                     nvt * (long long)incy, 0, 0, 0, 0};
        pos_group_chain<N, G>(C, pv, n, out, v);
    } else {
        const PosTerms<N, AoSRef<N>, AoSRef<N>, false, false> pv{xa, ya, nullptr, nullptr, v, nvt, v, nvt, 0, 0, 0, 0};
        pos_group_chain<N, G>(C, pv, n, out, v);
    }
}

// gemv partials (k_gemv_fold): RY: bx also as records
template <int N, int G, bool TRANS, bool RY, bool FIX>
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
    if (FIX && *part.sign(v) != REDO) return;
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
    pos_group_chain<N, G>(C, pv, cnt, part, v);
}

// gemm sums (k_gemm_sum): REC: operands from the records of op(A) (rows fastest) and op(B)
template <int N, bool REC, bool FIX, class VM>
__global__ __launch_bounds__(BLK) POS_WAVES(N <= 8 ? 4 : 2) void k_pos_gemm(const DevConsts *__restrict__ C, int ta, int tb, int m, int n, int k,
                                                  VM A, int lda, VM B, int ldb, const PosRec<Pos<N>::W> *__restrict__ ra,
                                                  const PosRec<Pos<N>::W> *__restrict__ rb, AoSRef<N> sums) {
    if constexpr (std::is_same<VM, SoA>::value) {
        A = rd(A);
        B = rd(B);
    }
    const long long e = (long long)blockIdx.x * BLK + threadIdx.x;
    if (e >= (long long)m * n) return;
    if (FIX && *sums.sign(e) != REDO) return;
    const int row = (int)(e % m), col = (int)(e / m);
    const long long a0 = op_index<0>(ta, row, 0, lda), b0 = op_index<1>(tb, col, 0, ldb);
    const PosTerms<N, VM, VM, REC, REC> pv{A,  B,  ra,
                                           rb, a0, ta ? 1LL : (long long)lda,
                                           b0, tb ? (long long)ldb : 1LL,
                                           row, m, (long long)col * k,
                                           1};
    pos_group_chain<N, 1>(C, pv, k, sums, e);
}

}  // namespace mph
