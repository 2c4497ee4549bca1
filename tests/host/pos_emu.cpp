// CPU emulation of the positional reduction chains (mpres-blas_amd/csrc/kernels_pos.hpp, one
// lane per chain) beside the residue chains of kernels.hpp they stand for. Built by
// tests/test_pos_cpu.py.
#include <vector>

#include "../../mpres-blas_amd/csrc/internal.hpp"
#include "../../mpres-blas_amd/csrc/kernels_pos.hpp"

using namespace mph;

namespace {

// chain c: terms x[c cnt + k] * y[c cnt + k], k < cnt. mode 0: the residue chain; 1: the positional
// chain; 2: its exact steps alone. Returns the chains left to the residue kernels.
template <int N>
int chains_n(const DevConsts &C, int mode, char *X, char *Y, int cnt, int chains, char *out) {
    constexpr int W = Pos<N>::W;
    const AoSRef<N> x{X}, y{Y}, o{out};
    int left = 0;
    for (long long c = 0; c < chains; c++) {
        if (mode == 0) {
            Grp<N, 1> g(&C);
            MP<N> acc;
            g.zero(acc);
            for (int k = 0; k < cnt; k++) g.template fma_step<true>(acc, x, c * cnt + k, y, c * cnt + k);
            store_aos(g, acc, o, c);
            continue;
        }
        const PosTerms<N, AoSRef<N>, AoSRef<N>, false, false> pv{x, y, nullptr, nullptr, c * cnt, 1,
                                                                 c * cnt, 1, 0, 0, 0, 0};
        if (mode == 1) {
            pos_group_chain<N, 1>(&C, pv, cnt, o, c);
            left += *o.sign(c) == REDO;
            continue;
        }
        PosNum<W> acc;
        PosSnap<W> snap;
        pos_zero(acc);
        pos_snap_zero(snap);
        bool ok = true;
        for (int k = 0; k < cnt && ok; k++) ok = pos_step_exact<N>(&C, pv, acc, snap, k);
        if (!ok) {
            *o.sign(c) = REDO;
            left++;
            continue;
        }
        for (int r = 0; r < N; r++) o.digits(c)[r] = pos_residue<N, W>(&C, acc.x, r);
        *o.sign(c) = snap.v.sign;
        *o.exp(c) = snap.v.exp;
        o.eval(c)[0] = ErMem{snap.v.ev0.frac, snap.v.ev0.exp};
        o.eval(c)[1] = ErMem{snap.v.ev1.frac, snap.v.ev1.exp};
    }
    return left;
}

}  // namespace

extern "C" int emu_pos_chains(int set_id, int mode, void *X, void *Y, int cnt, int chains, void *out) {
    const ModuliSet *s = get_set(set_id);
    DevConsts C;
    std::vector<int> pow2;
    if (!s || !compute_consts(*s, C, pow2)) return -1;
    C.pow2 = pow2.data();
    switch (C.n) {
        case 8: return chains_n<8>(C, mode, (char *)X, (char *)Y, cnt, chains, (char *)out);
        case 16: return chains_n<16>(C, mode, (char *)X, (char *)Y, cnt, chains, (char *)out);
    }
    return -1;
}
