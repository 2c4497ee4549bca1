// Launchers of the positional reduction kernels (kernels_pos.hpp) for one moduli count.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels_pos.hpp"

namespace mph {

// chains up to which a quad does a chain (kernels_pos.hpp); above, a lane each
constexpr long long POS_QUAD_CHAINS = 1 << 16;

template <int N>
struct LaunchPos {
    using Rec = PosRec<Pos<N>::W>;
    static unsigned blocks(long long threads) { return (unsigned)((threads + BLK - 1) / BLK); }
    template <int MODE, bool FIX>
    static void fold_m(const DevConsts *c, long long cnt, long long nvt, SoA xs, int incx, SoA ys, int incy,
                       AoSRef<N> xa, AoSRef<N> ya, AoSRef<N> out, hipStream_t st) {
        if (nvt <= POS_QUAD_CHAINS)
            hipLaunchKernelGGL((k_pos_fold<N, 4, MODE, FIX>), dim3(blocks(4 * nvt)), dim3(BLK), 0, st, c, cnt, nvt, xs,
                               incx, ys, incy, xa, ya, out);
        else
            hipLaunchKernelGGL((k_pos_fold<N, 1, MODE, FIX>), dim3(blocks(nvt)), dim3(BLK), 0, st, c, cnt, nvt, xs,
                               incx, ys, incy, xa, ya, out);
    }
    static hipError_t fold(const DevConsts *c, int mode, long long cnt, long long nvt, SoA xs, int incx, SoA ys,
                           int incy, const char *xa, const char *ya, char *out, hipStream_t st) {
        if (nvt <= 0) return hipSuccess;
        const AoSRef<N> X{(char *)xa}, Y{(char *)ya}, O{out};
        constexpr bool FIX = N > 8;  // above 8 moduli the residue kernel runs first
        if (mode == 0)
            fold_m<0, FIX>(c, cnt, nvt, xs, incx, ys, incy, X, Y, O, st);
        else
            fold_m<1, FIX>(c, cnt, nvt, xs, incx, ys, incy, X, Y, O, st);
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
    template <int G, bool TR, bool RY, bool FIX>
    static void gemv_g(const DevConsts *c, int m, int n, SoA A, int lda, AoSRef<N> bx, const Rec *rb, int b3,
                       long long nvt, AoSRef<N> part, hipStream_t st) {
        hipLaunchKernelGGL((k_pos_gemv<N, G, TR, RY, FIX>), dim3(blocks(G * nvt)), dim3(BLK), 0, st, c, m, n, A, lda,
                           bx, rb, b3, nvt, part);
    }
    template <bool TR>
    static void gemv_t(const DevConsts *c, int m, int n, SoA A, int lda, AoSRef<N> bx, const Rec *rb, int b3,
                       long long nvt, AoSRef<N> part, hipStream_t st) {
        constexpr bool FIX = N > 8;
        const bool quad = nvt <= POS_QUAD_CHAINS;
        if (rb && quad)
            gemv_g<4, TR, true, FIX>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
        else if (rb)
            gemv_g<1, TR, true, FIX>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
        else if (quad)
            gemv_g<4, TR, false, FIX>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
        else
            gemv_g<1, TR, false, FIX>(c, m, n, A, lda, bx, rb, b3, nvt, part, st);
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
    template <class VM>
    static void gemm_v(const DevConsts *c, int ta, int tb, int m, int n, int k, VM A, int lda, VM B, int ldb,
                       const char *ra, const char *rb, AoSRef<N> sums, hipStream_t st) {
        constexpr bool FIX = N > 8;
        const dim3 gr(blocks((long long)m * n)), bl(BLK);
        if (ra)
            hipLaunchKernelGGL((k_pos_gemm<N, true, FIX, VM>), gr, bl, 0, st, c, ta, tb, m, n, k, A, lda, B, ldb,
                               (const Rec *)ra, (const Rec *)rb, sums);
        else
            hipLaunchKernelGGL((k_pos_gemm<N, false, FIX, VM>), gr, bl, 0, st, c, ta, tb, m, n, k, A, lda, B, ldb,
                               (const Rec *)ra, (const Rec *)rb, sums);
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
