// CPU build of the element kernels with one lane per number over 16 and 32 moduli, whose numbers
// that need rounding are done again with the positional rounding, and of the integer routines
// behind them and behind division and square root. Built by tests/test_round_cpu.py.
#include <vector>

#include "../../mpres-blas_amd/csrc/internal.hpp"
#include "../../mpres-blas_amd/csrc/kernels.hpp"

using namespace mph;

namespace {

template <class F>
void run(long long threads, F &&f) {
    for (long long g = 0; g < (threads + BLK - 1) / BLK * BLK; g++) {
        blockIdx = EmuIdx{(unsigned)(g / BLK), 0, 0};
        threadIdx = EmuIdx{(unsigned)(g % BLK), 0, 0};
        f();
    }
}
template <int N>
int elem_n(const DevConsts &C, int op, int n, char *X, char *Y, const double *yd, char *R) {
    const AoSRef<N> x{X}, y{Y}, r{R};
    switch (op) {
        case 0: run(n, [&] { k_elem<N, 1, 0>(&C, n, x, y, yd, r); }); return 0;
        case 1: run(n, [&] { k_elem<N, 1, 1>(&C, n, x, y, yd, r); }); return 0;
        case 2: run(n, [&] { k_elem<N, 1, 2>(&C, n, x, y, yd, r); }); return 0;
        case 3: run(n, [&] { k_elem<N, 1, 3>(&C, n, x, y, yd, r); }); return 0;
        case 4: run(n, [&] { k_elem<N, 1, 4>(&C, n, x, y, yd, r); }); return 0;
        case 5: run(n, [&] { k_axpy_v2<N, 1>(&C, n, x, x, y, r); }); return 0;  // alpha = x[0]
        case 6: run(n, [&] { k_set_d<N, 1, false>(&C, yd, n, SoA{}, r); }); return 0;
    }
    return -1;
}

}  // namespace

extern "C" {
int emu_elem(int set_id, int op, int n, void *X, void *Y, const double *yd, void *R) {
    const ModuliSet *s = get_set(set_id);
    DevConsts C;
    std::vector<int> pow2;
    if (!s || !compute_consts(*s, C, pow2)) return -1;
    C.pow2 = pow2.data();
    return s->n == 16 ? elem_n<16>(C, op, n, (char *)X, (char *)Y, yd, (char *)R)
                      : elem_n<32>(C, op, n, (char *)X, (char *)Y, yd, (char *)R);
}
// a b mod m by the set's modulus i: by Barrett reduction (how = 0), or with the factor b's
// quotient (how = 1)
void emu_mulmod(int set_id, int how, int i, int count, const int *a, const int *b, int *r) {
    DevConsts C;
    std::vector<int> pow2;
    if (!compute_consts(*get_set(set_id), C, pow2)) return;
    const uint32_t m = (uint32_t)C.m[i];
    for (int k = 0; k < count; k++)
        r[k] = how ? mulmod_c((uint32_t)a[k], (uint32_t)b[k], (uint32_t)(((uint64_t)(uint32_t)b[k] << 32) / m), m)
                   : mulmod_i((uint32_t)a[k], (uint32_t)b[k], m, C.mu[i], C.mus);
}
constexpr int W = 16;
int emu_div(const uint32_t *a, const uint32_t *b, int q, uint32_t *o) {
    Big<W> x, y;
    for (int i = 0; i < W; i++) x.l[i] = a[i], y.l[i] = b[i];
    bool inexact;
    const Big<W> r = big_div_bits(x, y, q, inexact);
    for (int i = 0; i < W; i++) o[i] = r.l[i];
    return inexact;
}
int emu_isqrt(const uint32_t *a, uint32_t *o) {
    Big<W> x;
    for (int i = 0; i < W; i++) x.l[i] = a[i];
    bool inexact;
    const Big<W> r = big_isqrt(x, inexact);
    for (int i = 0; i < W; i++) o[i] = r.l[i];
    return inexact;
}
}
