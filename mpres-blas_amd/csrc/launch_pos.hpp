// Launchers of the positional reduction kernels (kernels_pos.hpp) for one moduli count.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_pos.hpp"

namespace mph {

// chains up to which a quad does a chain (kernels_pos.hpp); above, a lane each
constexpr long long POS_QUAD_CHAINS = 1 << 16;
// sums of a gemm up to which a quad does one: its products come from records, so that a quad saves
// less (64^3 84 us either way on rounding data and 92 against 195 on integers; 256^3, 65536 sums, 732 us
// on quads and 462 on single lanes)
constexpr long long POS_QUAD_SUMS = 1 << 14;

template <int N>
struct LaunchPos {
    using Rec = PosRec<Pos<N>::W>;
    static bool leaves(long long nvt) { return nvt > POS_QUAD_CHAINS; }
    static bool gemm_leaves(long long mn) { return mn > POS_QUAD_SUMS; }
    static unsigned blocks(long long threads) { return (unsigned)((threads + BLK - 1) / BLK); }
    template <int MODE>
    static void fold_m(const DevConsts *c, long long cnt, long long nvt, SoA xs, int incx, SoA ys, int incy,
                       AoSRef<N> xa, AoSRef<N> ya, AoSRef<N> out, hipStream_t st) {
        if (!leaves(nvt)) {
            hipLaunchKernelGGL((k_pos_fold<N, 4, MODE, POS_BOTH>), dim3(blocks(4 * nvt)), dim3(BLK), 0, st, c, cnt, nvt,
                               xs, incx, ys, incy, xa, ya, out);
            return;
        }
        hipLaunchKernelGGL((k_pos_fold<N, 1, MODE, POS_QUIET>), dim3(blocks(nvt)), dim3(BLK), 0, st, c, cnt, nvt, xs,
                           incx, ys, incy, xa, ya, out);
        hipLaunchKernelGGL((k_pos_fold<N, 1, MODE, POS_ONLY>), dim3(blocks(nvt)), dim3(BLK), 0, st, c, cnt, nvt, xs,
                           incx, ys, incy, xa, ya, out);
    }
    static hipError_t fold(const DevConsts *c, int mode, long long cnt, long long nvt, SoA xs, int incx, SoA ys,
                           int incy, const char *xa, const char *ya, char *out, hipStream_t st) {
        if (nvt <= 0) return hipSuccess;
        const AoSRef<N> X{(char *)xa}, Y{(char *)ya}, O{out};
        if (mode == 0)
            fold_m<0>(c, cnt, nvt, xs, incx, ys, incy, X, Y, O, st);
        else
            fold_m<1>(c, cnt, nvt, xs, incx, ys, incy, X, Y, O, st);
        return hipGetLastError();
    }
    static size_t rec_bytes(long long count) { return sizeof(Rec) * (size_t)count; }
    static hipError_t records(const DevConsts *c, int side, int t, int cnt, int k, SoA xs, const char *xa, bool soa,
                              int ld, char *rec, hipStream_t st) {
        if ((long long)cnt * k <= 0) return hipSuccess;
        const dim3 gr(blocks((long long)cnt * k)), bl(BLK);
        const AoSRef<N> X{(char *)xa};
        Rec *r = (Rec *)rec;
        if (soa && side == 0)
            hipLaunchKernelGGL((k_pos_records<N, SoA, 0>), gr, bl, 0, st, c, cnt, k, t, xs, ld, r);
        else if (soa)
            hipLaunchKernelGGL((k_pos_records<N, SoA, 1>), gr, bl, 0, st, c, cnt, k, t, xs, ld, r);
        else if (side == 0)
            hipLaunchKernelGGL((k_pos_records<N, AoSRef<N>, 0>), gr, bl, 0, st, c, cnt, k, t, X, ld, r);
        else
            hipLaunchKernelGGL((k_pos_records<N, AoSRef<N>, 1>), gr, bl, 0, st, c, cnt, k, t, X, ld, r);
        return hipGetLastError();
    }
    template <int G, bool TR, bool RY, int PART>
    static void gemv_g(const DevConsts *c, int m, int n, SoA A, int lda, AoSRef<N> bx, const Rec *rb, int b3,
                       long long nvt, AoSRef<N> part, hipStream_t st) {
        hipLaunchKernelGGL((k_pos_gemv<N, G, TR, RY, PART>), dim3(blocks(G * nvt)), dim3(BLK), 0, st, c, m, n, A, lda,
                           bx, rb, b3, nvt, part);
    }
    template <bool TR>
    static void gemv_t(const DevConsts *c, int m, int n, SoA A, int lda, AoSRef<N> bx, const Rec *rb, int b3,
                       long long nvt, AoSRef<N> part, hipStream_t st) {
        if (!leaves(nvt)) {
            if (rb)
                gemv_g<4, TR, true, POS_BOTH>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
            else
                gemv_g<4, TR, false, POS_BOTH>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
            return;
        }
        gemv_g<1, TR, false, POS_QUIET>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
        if (rb)
            gemv_g<1, TR, true, POS_ONLY>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
        else
            gemv_g<1, TR, false, POS_ONLY>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
    }
    static hipError_t gemv(const DevConsts *c, bool trans, int m, int n, SoA A, int lda, const char *bx,
                           const char *rec, int b3, long long nvt, char *part, hipStream_t st) {
        if (nvt <= 0) return hipSuccess;
        const AoSRef<N> B{(char *)bx}, P{part};
        const Rec *rb = (const Rec *)rec;
        if (trans)
            gemv_t<true>(c, m, n, A, lda, B, rb, b3, nvt, P, st);
        else
            gemv_t<false>(c, m, n, A, lda, B, rb, b3, nvt, P, st);
        return hipGetLastError();
    }
    template <int G, bool REC, int PART, class VM>
    static void gemm_g(const DevConsts *c, int ta, int tb, int m, int n, int k, VM A, int lda, VM B, int ldb,
                       const char *ra, const char *rb, AoSRef<N> sums, hipStream_t st) {
        hipLaunchKernelGGL((k_pos_gemm<N, G, REC, PART, VM>), dim3(blocks(G * (long long)m * n)), dim3(BLK), 0, st, c,
                           ta, tb, m, n, k, A, lda, B, ldb, (const Rec *)ra, (const Rec *)rb, sums);
    }
    template <class VM>
    static void gemm_v(const DevConsts *c, int ta, int tb, int m, int n, int k, VM A, int lda, VM B, int ldb,
                       const char *ra, const char *rb, AoSRef<N> sums, hipStream_t st) {
        if (!gemm_leaves((long long)m * n)) {
            if (ra)
                gemm_g<4, true, POS_BOTH, VM>(c, ta, tb, m, n, k, A, lda, B, ldb, ra, rb, sums, st);
            else
                gemm_g<4, false, POS_BOTH, VM>(c, ta, tb, m, n, k, A, lda, B, ldb, ra, rb, sums, st);
            return;
        }
        gemm_g<1, false, POS_QUIET, VM>(c, ta, tb, m, n, k, A, lda, B, ldb, ra, rb, sums, st);
        if (ra)
            gemm_g<1, true, POS_ONLY, VM>(c, ta, tb, m, n, k, A, lda, B, ldb, ra, rb, sums, st);
        else
            gemm_g<1, false, POS_ONLY, VM>(c, ta, tb, m, n, k, A, lda, B, ldb, ra, rb, sums, st);
    }
    static hipError_t gemm(const DevConsts *c, int ta, int tb, int m, int n, int k, SoA A, int lda, SoA B, int ldb,
                           const char *ra, const char *rb, char *sums, hipStream_t st) {
        if ((long long)m * n <= 0) return hipSuccess;
        gemm_v<SoA>(c, ta, tb, m, n, k, A, lda, B, ldb, ra, rb, AoSRef<N>{sums}, st);
        return hipGetLastError();
    }
    static hipError_t gemm_v2(const DevConsts *c, int ta, int tb, int m, int n, int k, const char *A, int lda,
                              const char *B, int ldb, const char *ra, const char *rb, char *sums, hipStream_t st) {
        if ((long long)m * n <= 0) return hipSuccess;
        gemm_v<AoSRef<N>>(c, ta, tb, m, n, k, AoSRef<N>{(char *)A}, lda, AoSRef<N>{(char *)B}, ldb, ra, rb,
                          AoSRef<N>{sums}, st);
        return hipGetLastError();
    }
    static PosOps table() {
        PosOps o;
        o.leaves = &leaves;
        o.gemm_leaves = &gemm_leaves;
        o.fold = &fold;
        o.rec_bytes = &rec_bytes;
        o.records = &records;
        o.gemv = &gemv;
        o.gemm = &gemm;
        o.gemm_v2 = &gemm_v2;
        return o;
    }
};

}  // namespace mph

#define MPH_INSTANTIATE_POS(N)                          \
    namespace mph {                                     \
    const PosOps *pos_ops_n##N() {                      \
        static const PosOps t = LaunchPos<N>::table();  \
        return &t;                                      \
    }                                                   \
    }
