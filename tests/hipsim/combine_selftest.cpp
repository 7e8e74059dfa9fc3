// k_lm_attn_combine on its own (tests/test_lm_sim.py).  TEST INFRASTRUCTURE ONLY.
#include "lm_kernels.h"

// ml [B][H][NS][2], part [B][H][NS][Dh] -> out [B][H * Dh]
extern "C" void combine_selftest_run(float* ml, float* part, int B, int H, int Dh, int NS, float* out) {
    LmAttnArgs a;
    memset(&a, 0, sizeof(a));
    a.ml = ml; a.opart = part; a.B = B; a.H = H; a.Dh = Dh; a.NS = NS;
    a.T = 16; a.out_ksteps = (H * Dh + 31) / 32;
    std::vector<uint16_t> packed((size_t)mmi_cdiv(B, a.T) * a.out_ksteps * 64 * 8);
    a.out = packed.data();
    MMI_LAUNCH(k_lm_attn_combine, B * H, Dh < 64 ? 64 : Dh, 0, (hipStream_t)0, a);
    for (int b = 0; b < B; ++b)
        for (int k = 0; k < H * Dh; ++k) out[b * H * Dh + k] = mmi_bf16_to_f32(packed[mmi_xp_index(a.T, b, k, a.out_ksteps)]);
}
void mmi_note_launch(const char*) {}
