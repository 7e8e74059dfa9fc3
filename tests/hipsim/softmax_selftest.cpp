// tlm_softmax_block on its own (tests/test_tlm_tiles.py): one column tile over blocks of 32 keys, in bf16.  TEST INFRASTRUCTURE ONLY.
#include "tlm_kernels.h"

// scores [blocks][32 keys][16 columns] -> p [blocks][32][16] as the value product gets them, m [blocks][16], l [16]
static void k_softmax(const float* scores, int blocks, float* p, float* mo, float* lo) {
    const int lane = threadIdx.x, bl = lane & 15, kq = lane >> 4;
    const TlmMask mask{0, 0, 1.f};
    float m = -1e30f, l = 0.f;
    f32x4 acc[1] = {{0.f, 0.f, 0.f, 0.f}};
    for (int b = 0; b < blocks; ++b) {
        f32x4 s0, s1;
        for (int r = 0; r < 4; ++r) {
            s0[r] = scores[(b * 32 + 4 * kq + r) * 16 + bl];
            s1[r] = scores[(b * 32 + 16 + 4 * kq + r) * 16 + bl];
        }
        u32x4 pf[1];
        tlm_softmax_block<TlmBf16, 1>(mask, s0, s1, b * 32 + 4 * kq, 1000, m, l, pf, acc);
        for (int r = 0; r < 8; ++r) p[(b * 32 + (r < 4 ? 0 : 16) + 4 * kq + (r & 3)) * 16 + bl] = mmi_bf16_to_f32((uint16_t)(pf[0][r / 2] >> (16 * (r & 1))));
        mo[b * 16 + bl] = m;
    }
    l += mmi_shfl_xor(l, 16);
    l += mmi_shfl_xor(l, 32);
    lo[bl] = l;
}

extern "C" void softmax_selftest_run(const float* scores, int blocks, float* p, float* m, float* l) {
    hipLaunchKernelGGL(k_softmax, dim3(1), dim3(64), 0, nullptr, scores, blocks, p, m, l);
}
