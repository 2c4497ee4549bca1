// Unsigned integers of W 32-bit limbs (least significant first), for the exact parts of
// the operations the reference runs on the host in MPFR: the division and square root
// of multiple-precision numbers (src/arith/div.cuh, src/arith/sqrt.cuh). These run one
// thread per number and are not on any hot path; every loop is bounded by W.
//
// __host__ __device__ so the same code is checked on the CPU against Python integers.
#pragma once

#include <stdint.h>

#include "numerics.hpp"

namespace mph {

template <int W>
struct Big {
    uint32_t l[W];
};

template <int W>
MPH_HD void big_zero(Big<W> &a) {
#pragma unroll
    for (int i = 0; i < W; i++) a.l[i] = 0;
}
template <int W>
MPH_HD bool big_is_zero(const Big<W> &a) {
    uint32_t o = 0;
#pragma unroll
    for (int i = 0; i < W; i++) o |= a.l[i];
    return o == 0;
}
MPH_HD int clz32(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __clz((int)v);
#else
    return v ? __builtin_clz(v) : 32;
#endif
}
MPH_HD int ctz32(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
    return v ? __ffs((int)v) - 1 : 32;
#else
    return v ? __builtin_ctz(v) : 32;
#endif
}
// Every index below is a compile-time constant (loops over limbs are unrolled, dynamic
// positions are resolved with selects), so a Big stays in registers: an array indexed
// with a run-time value would be placed in scratch memory.

// number of significant bits (0 for zero)
template <int W>
MPH_HD int big_bitlen(const Big<W> &a) {
    int r = 0;
#pragma unroll
    for (int i = 0; i < W; i++) r = a.l[i] ? 32 * i + 32 - clz32(a.l[i]) : r;
    return r;
}
// number of trailing zero bits (0 for zero)
template <int W>
MPH_HD int big_ctz(const Big<W> &a) {
    int r = 0;
#pragma unroll
    for (int i = W - 1; i >= 0; i--) r = a.l[i] ? 32 * i + ctz32(a.l[i]) : r;
    return r;
}
template <int W>
MPH_HD int big_bit(const Big<W> &a, int i) {
    const int q = i >> 5;
    uint32_t v = 0;
#pragma unroll
    for (int k = 0; k < W; k++) v = q == k ? a.l[k] : v;
    return (i >= 0 && i < 32 * W) ? (int)((v >> (i & 31)) & 1u) : 0;
}
// any nonzero bit below position i
template <int W>
MPH_HD bool big_any_below(const Big<W> &a, int i) {
    uint32_t o = 0;
#pragma unroll
    for (int q = 0; q < W; q++) {
        const int k = i - 32 * q;  // bits of limb q below position i
        const uint32_t mask = k >= 32 ? 0xffffffffu : (k <= 0 ? 0u : (1u << (k & 31)) - 1u);
        o |= a.l[q] & mask;
    }
    return o != 0;
}
// a << s for s >= 0, bits shifted beyond W limbs are lost: the whole-limb part as a
// barrel of conditional moves (1, 2, 4, ... limbs), then the bit part
template <int W>
MPH_HD Big<W> big_shl(const Big<W> &a, int s) {
    Big<W> r = a;
    const int q = s >> 5, b = s & 31;
#pragma unroll
    for (int k = 1; k < W; k <<= 1) {
        const bool on = (q & k) != 0;
#pragma unroll
        for (int i = W - 1; i >= 0; i--) r.l[i] = on ? (i >= k ? r.l[i - k] : 0u) : r.l[i];
    }
    const bool out = q >= W;
#pragma unroll
    for (int i = W - 1; i >= 0; i--) {
        const uint32_t lo = i > 0 ? r.l[i - 1] : 0u;
        r.l[i] = out ? 0u : (b ? (r.l[i] << b) | (lo >> ((32 - b) & 31)) : r.l[i]);
    }
    return r;
}
// a >> s for s >= 0
template <int W>
MPH_HD Big<W> big_shr(const Big<W> &a, int s) {
    Big<W> r = a;
    const int q = s >> 5, b = s & 31;
#pragma unroll
    for (int k = 1; k < W; k <<= 1) {
        const bool on = (q & k) != 0;
#pragma unroll
        for (int i = 0; i < W; i++) r.l[i] = on ? (i + k < W ? r.l[i + k] : 0u) : r.l[i];
    }
    const bool out = q >= W;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint32_t hi = i + 1 < W ? r.l[i + 1] : 0u;
        r.l[i] = out ? 0u : (b ? (r.l[i] >> b) | (hi << ((32 - b) & 31)) : r.l[i]);
    }
    return r;
}
template <int W>
MPH_HD int big_cmp(const Big<W> &a, const Big<W> &b) {
    int r = 0;
#pragma unroll
    for (int i = 0; i < W; i++) r = a.l[i] != b.l[i] ? (a.l[i] > b.l[i] ? 1 : -1) : r;
    return r;
}
// a -= b (a >= b)
template <int W>
MPH_HD void big_sub(Big<W> &a, const Big<W> &b) {
    uint64_t borrow = 0;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint64_t t = (uint64_t)a.l[i] - b.l[i] - borrow;
        a.l[i] = (uint32_t)t;
        borrow = (t >> 63) & 1u;
    }
}
// a += b
template <int W>
MPH_HD void big_add(Big<W> &a, const Big<W> &b) {
    uint64_t carry = 0;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint64_t t = (uint64_t)a.l[i] + b.l[i] + carry;
        a.l[i] = (uint32_t)t;
        carry = t >> 32;
    }
}
template <int W>
MPH_HD void big_add_u32(Big<W> &a, uint32_t v) {
    uint64_t carry = v;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const uint64_t t = (uint64_t)a.l[i] + carry;
        a.l[i] = (uint32_t)t;
        carry = t >> 32;
    }
}
// a * b, exactly
template <int A, int B>
MPH_HD Big<A + B> big_mul(const Big<A> &a, const Big<B> &b) {
    Big<A + B> r;
    big_zero(r);
#pragma unroll
    for (int i = 0; i < A; i++) {
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < B; j++) {
            const uint64_t t = (uint64_t)a.l[i] * b.l[j] + r.l[i + j] + c;
            r.l[i + j] = (uint32_t)t;
            c = t >> 32;
        }
        r.l[i + B] = (uint32_t)c;
    }
    return r;
}
// a in a wider (or equal) type
template <int WB, int WA>
MPH_HD Big<WB> big_widen(const Big<WA> &a) {
    static_assert(WB >= WA, "widen");
    Big<WB> r;
#pragma unroll
    for (int i = 0; i < WB; i++) r.l[i] = i < WA ? a.l[i] : 0u;
    return r;
}
// a mod m for a modulus below 2^31
template <int W>
MPH_HD uint32_t big_mod_u32(const Big<W> &a, uint32_t m) {
    uint64_t r = 0;
#pragma unroll
    for (int i = W - 1; i >= 0; i--) r = ((r << 32) | a.l[i]) % m;
    return (uint32_t)r;
}
// a mod m through exact FP64 steps (modd), 16 bits at a time: r 2^16 + digit < 2^47
template <int W>
MPH_HD int big_mod_d(const Big<W> &a, double m, double minv) {
    int r = 0;
#pragma unroll
    for (int i = W - 1; i >= 0; i--) {
        r = modd((double)r * 65536.0 + (double)(a.l[i] >> 16), m, minv);
        r = modd((double)r * 65536.0 + (double)(a.l[i] & 0xffffu), m, minv);
    }
    return r;
}
// a rounded to p significant bits, to nearest with ties to even (the value a * 2^e is
// kept: e grows by the bits dropped); the result may be 2^p
template <int W>
MPH_HD void big_round(Big<W> &a, int &e, int p) {
    const int b = big_bitlen(a);
    if (b <= p) return;
    const int sh = b - p;
    const int half = big_bit(a, sh - 1), sticky = big_any_below(a, sh - 1) ? 1 : 0;
    a = big_shr(a, sh);
    if (half && (sticky || (a.l[0] & 1u))) big_add_u32(a, 1u);
    e += sh;
}
// a top-aligned estimate: the leading 64 bits at and below limb W - 1 as a double
template <int W>
MPH_HD double big_top(const Big<W> &a) {
    return fma((double)a.l[W - 1], 0x1p32, (double)a.l[W - 2]) + (double)a.l[W - 3] * 0x1p-32;
}
// r - d * b, 0 <= d < 2^26, in two's complement
template <int W>
MPH_HD void big_submul(Big<W> &r, const Big<W> &b, uint32_t d) {
    uint64_t c = 0;
    uint32_t borrow = 0;
#pragma unroll
    for (int i = 0; i < W; i++) {
        c += (uint64_t)b.l[i] * d;
        const uint64_t t = (uint64_t)r.l[i] - (uint32_t)c - borrow;
        r.l[i] = (uint32_t)t;
        borrow = (uint32_t)(t >> 63);
        c >>= 32;
    }
}
// a << S for a constant 0 < S < 32
template <int S, int W>
MPH_HD void big_shl_const(Big<W> &a) {
#pragma unroll
    for (int i = W - 1; i >= 0; i--) a.l[i] = (a.l[i] << S) | (i > 0 ? a.l[i - 1] >> (32 - S) : 0u);
}
// floor(a / b * 2^(q - 1)) for a, b of equal bit length L (so 1/2 < a/b < 2), with
// W >= L + 2 bits, q <= 32 W; and whether the division left a remainder. Long division with
// digits of BIG_DIGIT bits, each estimated in double from the leading bits (off by one at most) and corrected.
constexpr int BIG_DIGIT = 24;
template <int W>
MPH_HD Big<W> big_div_bits(const Big<W> &a, const Big<W> &b, int q, bool &inexact) {
    // both operands at the top of limb W - 1, one limb of headroom
    const int up = 32 * W - big_bitlen(b);
    Big<W + 1> r = big_shl(big_widen<W + 1>(a), up), d = big_shl(big_widen<W + 1>(b), up);
    const double inv = 1.0 / big_top(d);
    Big<W> quo;
    big_zero(quo);
    if (big_cmp(r, d) >= 0) {
        big_sub(r, d);
        quo.l[0] = 1u;
    }
    const int digits = (q - 1 + BIG_DIGIT - 1) / BIG_DIGIT, extra = digits * BIG_DIGIT - (q - 1);
    bool lost = false;
#pragma nounroll
    for (int i = 0; i < digits; i++) {
        big_shl_const<BIG_DIGIT>(r);
        int t = (int)(big_top(r) * inv);
        big_submul(r, d, (uint32_t)t);
        if ((int)r.l[W] < 0) {  // one too many
            big_add(r, d);
            t--;
        } else if (big_cmp(r, d) >= 0) {
            big_sub(r, d);
            t++;
        }
        if (i + 1 < digits) {
            big_shl_const<BIG_DIGIT>(quo);
            quo.l[0] |= (uint32_t)t;
        } else {  // the last digit's bits below 2^-(q - 1) only tell whether there is a remainder
            quo = big_shl(quo, BIG_DIGIT - extra);
            quo.l[0] |= (uint32_t)t >> extra;
            lost = ((uint32_t)t & ((1u << extra) - 1u)) != 0;
        }
    }
    inexact = lost || !big_is_zero(r);
    return quo;
}
// s = floor(sqrt(a)), a below 2^(32 W - 48); inexact when s^2 != a. The root's digits of 24 bits: the
// first from a's leading 47 or 48 bits in double, each further one d from the remainder r
// (next two digits of a appended): the largest with d (2 s + d) <= r, estimated as r / (2 s) and
// corrected.
template <int W>
MPH_HD Big<W> big_isqrt(const Big<W> &a, bool &inexact) {
    Big<W> s;
    big_zero(s);
    const int len = big_bitlen(a);
    if (len == 0) {
        inexact = false;
        return s;
    }
    // a 4^z, of 48 digits - 1 or 48 digits bits, at the top of x: its 48-bit digits are taken from
    // there in turn, and the root comes out times 2^z
    const int digits = (len + 47) / 48, z = (48 * digits - len) / 2;
    Big<W> x = big_shl(a, 32 * W - 48 * digits + 2 * z);
    auto next = [&]() -> uint64_t {
        const uint64_t v = ((uint64_t)x.l[W - 1] << 16) | (x.l[W - 2] >> 16);
        big_shl_const<24>(x);
        big_shl_const<24>(x);
        return v;
    };
    uint64_t c = next();
    uint64_t s0 = (uint64_t)sqrt((double)c);
    Big<W> r;  // remainder, at most 2 s
    big_zero(r);
    r.l[0] = (uint32_t)(c - s0 * s0);
    r.l[1] = (uint32_t)((c - s0 * s0) >> 32);
    s.l[0] = (uint32_t)s0;
#pragma nounroll
    for (int i = 1; i < digits; i++) {
        c = next();
        big_shl_const<24>(r);
        big_shl_const<24>(r);
        r.l[0] |= (uint32_t)c;
        r.l[1] |= (uint32_t)(c >> 32);
        big_shl_const<24>(s);
        const Big<W> s2 = big_shl(s, 1);
        // estimate from the leading bits of 2 s
        const int k = big_bitlen(s2) > 64 ? big_bitlen(s2) - 64 : 0;
        const Big<W> st = big_shr(s2, k), rt = big_shr(r, k);
        const double sd = fma((double)st.l[1], 0x1p32, (double)st.l[0]);
        const double rd = fma(fma((double)rt.l[2], 0x1p32, (double)rt.l[1]), 0x1p32, (double)rt.l[0]);
        double e = rd / sd;
        e = e > 16777215.0 ? 16777215.0 : e;
        uint32_t d = (uint32_t)e;
        // r - d (2 s + d)
        Big<W> t = s2;
        t.l[0] |= d;  // 2 s is a multiple of 2^25
        big_submul(r, t, d);
        for (int j = 0; j < 2 && (int)r.l[W - 1] < 0; j++) {  // too many: add back (2 s + 2 d - 1)
            d--;
            Big<W> u = s2;
            big_add_u32(u, 2 * d + 1);
            big_add(r, u);
        }
        {  // one too few: r >= 2 s + 2 d + 1
            Big<W> u = s2;
            big_add_u32(u, 2 * d + 1);
            if (d < 16777215u && big_cmp(r, u) >= 0) {
                big_sub(r, u);
                d++;
            }
        }
        s.l[0] |= d;
    }
    inexact = !big_is_zero(r) || big_any_below(s, z);
    return big_shr(s, z);
}

}  // namespace mph
