// tlm_sigmoid on its own (tests/test_tlm_sim.py).  TEST INFRASTRUCTURE ONLY.
#include "tlm_kernels.h"

extern "C" void sigmoid_selftest_run(const float* x, int n, float* y) {
    for (int i = 0; i < n; ++i) y[i] = tlm_sigmoid(x[i]);
}
