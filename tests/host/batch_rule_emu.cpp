// The batch plan's choice of lanes on the CPU. Built by tests/test_batch_lanes_cpu.py.
#include "../../mpres-blas_amd/csrc/batch_plan.hpp"

extern "C" int emu_batch_one_lane(const mpres_batch_problem_t *probs, int count) {
    return mph::batch_one_lane(probs, count);
}
