// Residues to positional integers and back, and the interval evaluation of an integer, one thread
// per number: the parts that the positional reduction chains (pos.hpp) and the rounding of
// single numbers share.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "devconsts.hpp"
#include "numerics.hpp"
#include "rare.hpp"

namespace mph {

template <int N>
struct Pos {
    static constexpr int W = N / 2;  // words of a normalised number (at most 31 N / 2 + 2 bits)
};

// a value of the constants block, through the scalar cache: the address is wave-uniform and the
// block is never written while kernels run, which the constant address space states (a plain
// load behind calls and stores would be a vector load)
template <class T>
__device__ __forceinline__ T pos_const(const T &v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const __attribute__((address_space(4))) T *)(uintptr_t)&v;
#else
    return v;
#endif
}
// a wave-uniform pointer that reached a function through its arguments (vector registers), so
// that what it points to is read through the scalar cache again
__device__ __forceinline__ const DevConsts *uniform_ptr(const DevConsts *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const DevConsts *)(uintptr_t)((uint64_t)hi << 32 | lo);
#else
    return p;
#endif
}
// keeps the instructions before it ahead of those after it: bounds how many table entries are
// in registers at once
__device__ __forceinline__ void pos_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
}
// x >> s for any s >= 0; dropped: whether a nonzero bit was shifted out
template <int W>
__device__ __forceinline__ void pos_shr(uint32_t *r, const uint32_t *x, int s, bool &dropped) {
    uint32_t low = 0;
    const int b = s & 31;
    int q = s >> 5;
    q = q > W ? W : q;
#pragma unroll
    for (int i = 0; i < W; i++) r[i] = x[i];
#pragma unroll
    for (int k = 1; k <= W; k <<= 1) {
        const bool on = (q & k) != 0;
#pragma unroll
        for (int i = 0; i < W; i++) {
            if (i < k) low |= on ? r[i] : 0u;
            r[i] = on ? (i + k < W ? r[i + k] : 0u) : r[i];
        }
    }
    low |= b ? r[0] << ((32 - b) & 31) : 0u;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint32_t hi = i + 1 < W ? r[i + 1] : 0u;
        r[i] = (uint32_t)((((uint64_t)hi << 32) | r[i]) >> b);
    }
    dropped = low != 0;
}
// a residue in [0, m) of any int
__device__ __forceinline__ int pos_reduce(int d, int m) {
    if ((unsigned)d < (unsigned)m) return d;  // as every operation leaves it
    const int v = d % m;
    return v < 0 ? v + m : v;
}
// The integer of residues (any int from 0 of the class): X = sum c_i M/m_i - rank M with c_i = |x_i w_i| mod m_i, its low WX
// words. NORM: X / M below 2^-40, and rank the nearest integer of sum c_i / m_i; otherwise any
// X < M (WX = N: all of it): rank is the whole part of a sum that may be off by 2^-40, so the
// result is brought into [0, M). Columns of 28-bit limbs in 64 bits: at most 32 products
// below 1.43e9 2^28 (compute_consts), the rank's multiple of 2^K - M, below 2^33, and a carry below 2^36
// stay below 2^63.5.
template <int N, int WX, bool NORM>
__device__ __forceinline__ void pos_from_digits(const DevConsts *__restrict__ C, const int *d, uint32_t *x) {
    constexpr int LN = (32 * WX + 27) / 28;
    uint32_t c[N];
    double rk = 0.0;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const int v = mulmod_c((uint32_t)d[i], (uint32_t)pos_const(C->w[i]), pos_const(C->wq[i]),
                               (uint32_t)pos_const(C->m[i]));
        c[i] = (uint32_t)v;
        rk = fma((double)v, pos_const(C->minv[i]), rk);
    }
    const uint32_t rank = (uint32_t)(NORM ? rint(rk) : floor(rk + 0x1p-40));
    uint64_t carry = 0;
    uint32_t y[LN];
#pragma unroll
    for (int l = 0; l < LN; l++) {
        if (l % 2 == 0) pos_fence();
        uint64_t v = carry;
#pragma unroll
        for (int i = 0; i < N; i++) v += (uint64_t)c[i] * pos_const(C->mi28[l][i]);
        v += (uint64_t)rank * pos_const(C->mn28[l]);
        y[l] = (uint32_t)v & 0xfffffffu;
        carry = v >> 28;
    }
    // 28-bit limbs to words
#pragma unroll
    for (int w = 0; w < WX; w++) {
        const int l = 32 * w / 28, b = 32 * w % 28;
        uint32_t v = y[l] >> b;
        if (l + 1 < LN) v |= y[l + 1] << (28 - b);
        if (b > 24 && l + 2 < LN) v |= y[l + 2] << (56 - b);
        x[w] = v;
    }
    if constexpr (!NORM) {
        // rank one too large (X negative mod 2^K: above M) or one too small (X at or above M)
        const bool neg = (y[LN - 1] >> 27) != 0;
        uint32_t t[WX];
        uint32_t borrow = 0, cc = 0;
#pragma unroll
        for (int w = 0; w < WX; w++) {
            const uint64_t q = (uint64_t)x[w] - pos_const(C->m32[w]) - borrow;
            t[w] = (uint32_t)q;
            borrow = (uint32_t)(q >> 63);
        }
        const bool over = !neg && borrow == 0;
#pragma unroll
        for (int w = 0; w < WX; w++) {
            const uint64_t q = (uint64_t)x[w] + pos_const(C->m32[w]) + cc;
            cc = (uint32_t)(q >> 32);
            x[w] = neg ? (uint32_t)q : over ? t[w] : x[w];
        }
    }
}
// residue i of an integer of WX words
template <int N, int WX>
__device__ __forceinline__ int pos_residue(const DevConsts *__restrict__ C, const uint32_t *x, int i) {
    double v = 0.0;
#pragma unroll
    for (int l = 0; l < WX; l++) {
        v = fma((double)(x[l] & 0xffffu), pos_const(C->q16[i][2 * l]), v);
        v = fma((double)(x[l] >> 16), pos_const(C->q16[i][2 * l + 1]), v);
    }
    return modd(v, pos_const(C->md[i]), pos_const(C->minv[i]));
}
// ---- several directed operations under one setting of the rounding mode (numerics.hpp) ----
#if defined(__HIP_DEVICE_COMPILE__)
#define POS_DIR4(MODE, OP, BC)                                                                            \
    asm("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), " #MODE "\n\ts_nop 1\n\t" OP " %0, %4, %5\n\t" OP  \
        " %1, %6, %7\n\t" OP " %2, %8, %9\n\t" OP " %3, %10, %11\n\ts_nop 1\n\t"                         \
        "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 2, 2), 0\n\ts_nop 1"                                       \
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])                                              \
        : "v"(a[0]), BC(b[0]), "v"(a[1]), BC(b[1]), "v"(a[2]), BC(b[2]), "v"(a[3]), BC(b[3]))
#endif
// r[i] = a[i] + b[i] rounded up (UP) or down, i < CNT
template <int CNT, bool UP>
__device__ __forceinline__ void dir_add(double *r, const double *a, const double *b) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (CNT >= 4) {
        if constexpr (UP)
            POS_DIR4(1, "v_add_f64", "v");
        else
            POS_DIR4(2, "v_add_f64", "v");
        if constexpr (CNT > 4) dir_add<CNT - 4, UP>(r + 4, a + 4, b + 4);
        return;
    }
#endif
#pragma unroll
    for (int i = 0; i < CNT; i++) r[i] = UP ? add_ru(a[i], b[i]) : add_rd(a[i], b[i]);
}
// r[i] = x[i] * c[i] rounded up (UP) or down, i < CNT; c: constants of the block
template <int CNT, bool UP>
__device__ __forceinline__ void dir_mulc(double *r, const int *x, const double *c) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (CNT >= 4) {
        const double a[4] = {(double)x[0], (double)x[1], (double)x[2], (double)x[3]};
        const double b[4] = {pos_const(c[0]), pos_const(c[1]), pos_const(c[2]), pos_const(c[3])};
        if constexpr (UP)
            POS_DIR4(1, "v_mul_f64", "s");
        else
            POS_DIR4(2, "v_mul_f64", "s");
        if constexpr (CNT > 4) dir_mulc<CNT - 4, UP>(r + 4, x + 4, c + 4);
        return;
    }
#endif
#pragma unroll
    for (int i = 0; i < CNT; i++) r[i] = UP ? mul_ru((double)x[i], c[i]) : mul_rd((double)x[i], c[i]);
}
#undef POS_DIR4
// psum_arr's balanced tree over v[0 .. CNT-1], in place; the sum in v[0]
template <int CNT, bool UP>
__device__ __forceinline__ void dir_sum(double *v) {
    if constexpr (CNT > 1) {
        double a[CNT / 2], b[CNT / 2];
#pragma unroll
        for (int i = 0; i < CNT / 2; i++) {
            a[i] = v[2 * i];
            b[i] = v[2 * i + 1];
        }
        dir_add<CNT / 2, UP>(v, a, b);
        dir_sum<CNT / 2, UP>(v);
    }
}
// Interval evaluation of a rounded integer: rns_eval<FULL = false> on its residues, the
// directed operations of one kind issued together.
template <int N>
__device__ __forceinline__ void pos_eval_fast(const DevConsts *__restrict__ C, const uint32_t *x, Er &lo, Er &up) {
    int s[N];
    double f[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        s[i] = mulmod_c((uint32_t)pos_residue<N, Pos<N>::W>(C, x, i), (uint32_t)pos_const(C->w[i]),
                        pos_const(C->wq[i]), (uint32_t)pos_const(C->m[i]));
        if (i % 2 == 1) pos_fence();
    }
    auto sum = [&](auto upw, double &frac, unsigned &whole) {
        constexpr bool UP = decltype(upw)::value;
        dir_mulc<N, UP>(f, s, UP ? C->rru : C->rrd);
        dir_sum<N, UP>(f);
        whole = (unsigned)f[0];
        frac = f[0];
    };
    double sl, su;
    unsigned wl, wu;
    sum(std::false_type{}, sl, wl);
    sum(std::true_type{}, su, wu);
    if (sl == 0 && su == 0) {
        lo = Er{0.0, 0};
        up = Er{0.0, 0};
        return;
    }
    sl = sub_rd(sl, (double)wl);
    su = sub_ru(su, (double)wu);
    const double acc = pos_const(C->acc);
    int K = 0;
    if (su < acc) {
        const int ref = pos_const(C->ref_factor), kmax = pos_const(C->log2m);
        const int *p2 = pos_const(C->pow2);
        for (int it = 0; su < acc && it < EVAL_MAX_ITER; it++) {
            int kk = -(ceil_log2_rn(su) + 1);
            kk = kk > ref ? kk : ref;
            kk = kk < kmax ? kk : kmax;
            const int *row = p2 + (size_t)kk * N, *rowq = row + (size_t)(kmax + 1) * N;
#pragma unroll
            for (int i = 0; i < N; i++)
                s[i] = mulmod_c((uint32_t)s[i], (uint32_t)row[i], (uint32_t)rowq[i], (uint32_t)pos_const(C->m[i]));
            sum(std::true_type{}, su, wu);
            su = sub_ru(su, (double)wu);
            K += kk;
        }
        sum(std::false_type{}, sl, wl);
        sl = sub_rd(sl, (double)wl);
    }
    lo = er_set_d(sl);
    up = er_set_d(su);
    lo.exp -= K;
    up.exp -= K;
}

// mp_round of one number in one thread (mp_round_body): X = floor(X / 2^bits) on the integer, then
// the residues and the evaluation of the result. The residue algorithm scales in steps of 30
// bits, each with a rank and two passes over the residues; here the integer is formed once
// (exact for every X < M) and shifted. bits = ev1.exp - mp_h + 1 leaves X below 2^mp_h M, so the
// result fits W words. False, and nothing done, when it does not: the evaluation is then not the
// number's (a sum that the residue algorithm let wrap after an exact cancellation), and what
// the residue algorithm makes of it is its own.
template <int N>
__device__ __forceinline__ bool pos_round(const DevConsts *__restrict__ C, int *d, int &exp, Er &ev0, Er &ev1) {
    constexpr int W = Pos<N>::W;
    const int bits = ev1.exp - pos_const(C->mp_h) + 1;
    uint32_t x[N], y[N];
    pos_from_digits<N, N, false>(C, d, x);
    bool dropped;
    pos_shr<N>(y, x, bits, dropped);
    uint32_t high = 0;
#pragma unroll
    for (int i = W; i < N; i++) high |= y[i];
    if (high) return false;
    exp += bits;
#pragma unroll
    for (int i = 0; i < N; i++) {
        d[i] = pos_residue<N, W>(C, y, i);
        if (i % 2 == 1) pos_fence();
    }
    pos_eval_fast<N>(C, y, ev0, ev1);
    return true;
}

}  // namespace mph
