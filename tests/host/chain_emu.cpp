// CPU emulation of the scalar chains on absolute bounds (k_chain_ops, k_gemm_chain_abs) beside the
// chains by sc_fma_step (k_gemm_chain). Built by tests/test_chain_cpu.py.
#include <vector>

#include "../../mpres-blas_amd/csrc/internal.hpp"
#include "../../mpres-blas_amd/csrc/kernels.hpp"

using namespace mph;

namespace {

template <class F>
void run(long long threads, unsigned y, F &&f) {
    for (long long g = 0; g < (threads + BLK - 1) / BLK * BLK; g++) {
        blockIdx = EmuIdx{(unsigned)(g / BLK), y, 0};
        threadIdx = EmuIdx{(unsigned)(g % BLK), 0, 0};
        f();
    }
}

template <int N>
int chain_n(const DevConsts &C, int ta, int tb, int m, int n, int k, char *A, int lda, char *B, int ldb, char *w1,
            char *w2) {
    const AoSRef<N> a{A}, b{B}, s1{w1}, s2{w2};
    std::vector<ChainOp> pa((size_t)m * k), pb((size_t)n * k);
    std::vector<int> ea((size_t)m * k), eb((size_t)n * k);
    const long long most = (long long)(m > n ? m : n) * k;
    for (unsigned side = 0; side < 2; side++)
        run(most, side, [&] {
            k_chain_ops<N, AoSRef<N>>(&C, ta, tb, m, n, k, a, lda, b, ldb, pa.data(), ea.data(), pb.data(), eb.data());
        });
    run((long long)m * n, 0, [&] { k_gemm_chain<N, 1, AoSRef<N>>(&C, ta, tb, m, n, k, a, lda, b, ldb, s1); });
    run((long long)m * n, 0, [&] {
        k_gemm_chain_abs<N, false, AoSRef<N>>(&C, ta, tb, m, n, k, a, lda, b, ldb, pa.data(), ea.data(), pb.data(),
                                              eb.data(), s2);
    });
    int unusual = 0;
    for (int e : ea) unusual += e == CA_BAD;
    return unusual;
}

}  // namespace

// returns the operands of op(A) outside the form's range
extern "C" int emu_chain_abs(int set_id, int ta, int tb, int m, int n, int k, void *A, int lda, void *B, int ldb,
                             void *w1, void *w2) {
    const ModuliSet *s = get_set(set_id);
    DevConsts C;
    std::vector<int> pow2;
    if (!s || !compute_consts(*s, C, pow2)) return -1;
    C.pow2 = pow2.data();
    switch (C.n) {
        case 16: return chain_n<16>(C, ta, tb, m, n, k, (char *)A, lda, (char *)B, ldb, (char *)w1, (char *)w2);
        case 32: return chain_n<32>(C, ta, tb, m, n, k, (char *)A, lda, (char *)B, ldb, (char *)w1, (char *)w2);
    }
    return -1;
}
