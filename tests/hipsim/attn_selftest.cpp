// k_lm_attn_wave on its own (tests/test_lm_sim.py): heads of 64 features, the ring over two workgroups that leave their partials in fp32.
// TEST INFRASTRUCTURE ONLY.
#include "lm_kernels.h"

// q [H][64], k and v [H][L][64] (bf16, or e4m3 bytes where kv8) -> ml [H][2][2], part [H][2][64]
extern "C" void attn_selftest_run(uint16_t* q, void* k, void* v, int H, int L, int kv8, float* ml, float* part) {
    LmAttnArgs a;
    memset(&a, 0, sizeof(a));
    const long off = L - 1;
    a.qrot = q; a.kc = (uint16_t*)k; a.vc = (uint16_t*)v; a.offsets = &off; a.opart = part; a.ml = ml;
    a.B = 1; a.H = H; a.Dh = 64; a.cap = L; a.context = L; a.NS = 2; a.solo_rows = -1;
    if (kv8) MMI_LAUNCH((k_lm_attn_wave<64, true>), dim3(H, 2), 256, 0, (hipStream_t)0, a);
    else MMI_LAUNCH((k_lm_attn_wave<64, false>), dim3(H, 2), 256, 0, (hipStream_t)0, a);
}
void mmi_note_launch(const char*) {}
