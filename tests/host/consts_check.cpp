// compute_consts on moduli sets that the library does not ship. Built by tests/test_consts_bounds_cpu.py.
#include "../../mpres-blas_amd/csrc/internal.hpp"

extern "C" int check_set(int n, int log2m, const int *m) {
    mph::ModuliSet s{"test", n, log2m, {}};
    for (int i = 0; i < n && i < mph::MAXN; i++) s.m[i] = m[i];
    mph::DevConsts c;
    std::vector<int> pow2;
    return mph::compute_consts(s, c, pow2);
}
