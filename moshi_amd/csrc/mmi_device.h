// Device-side primitives for the gfx950 (MI355X / CDNA4) build.  Every kernel in csrc/ is written
// against this small vocabulary: 64-lane wave shuffles, the four MFMA shapes we use, non-temporal
// 16-byte weight loads and the launch macro.  This file is the ONLY place the amdgcn builtins are
// named, so the kernels read as algorithms rather than intrinsic soup.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 mmi_bf16x8 __attribute__((ext_vector_type(8)));

#define MMI_WAVE 64
#define MMI_SHARED __shared__
#define MMI_DYN_SHARED(T, name)                                                   \
    extern __shared__ __attribute__((aligned(16))) unsigned char name##_raw_[];  \
    T* name = reinterpret_cast<T*>(name##_raw_)
// every launch is announced to the launch-list recorder (mmi_graph.h: which site of the step issued which kernel; a
// no-op unless a program is being recorded)
void mmi_note_launch(const char* kernel);
#define MMI_LAUNCH(kern, grid, block, shmem, stream, ...)                    \
    do {                                                                     \
        mmi_note_launch(#kern);                                              \
        hipLaunchKernelGGL(kern, grid, block, shmem, stream, __VA_ARGS__);   \
    } while (0)

// float -> bf16, round-to-nearest-even.  gfx950 has the conversion in hardware (v_cvt_pk_bf16_f32); host code (weight
// import helpers) takes the bit-level definition in mmi_common.h.
typedef __bf16 mmi_bf16x2 __attribute__((ext_vector_type(2)));
__host__ __device__ __forceinline__ uint16_t mmi_f32_to_bf16_bits(float f);
__host__ __device__ __forceinline__ uint16_t mmi_cvt_bf16(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_bit_cast(uint16_t, (__bf16)f);
#else
    return mmi_f32_to_bf16_bits(f);
#endif
}
__host__ __device__ __forceinline__ uint32_t mmi_cvt_pk_bf16(float lo, float hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, mmi_bf16x2));
#else
    return (uint32_t)mmi_f32_to_bf16_bits(lo) | ((uint32_t)mmi_f32_to_bf16_bits(hi) << 16);
#endif
}

__device__ __forceinline__ int mmi_lane() { return (int)(threadIdx.x & 63u); }

template <class T>
__device__ __forceinline__ T mmi_shfl_xor(T v, int mask) { return __shfl_xor(v, mask, 64); }
template <class T>
__device__ __forceinline__ T mmi_shfl(T v, int src) { return __shfl(v, src, 64); }

// Sum over groups of W consecutive lanes (W = 2, 4, 8, 16; a group never straddles a 16-lane row), every lane of the group
// receiving the total: DPP row operations - quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror, row_mirror - which are
// plain VALU operand modifiers.  __shfl_xor compiles to ds_bpermute_b32 + s_waitcnt lgkmcnt(0) per step: a dependent trip
// through the LDS crossbar each (the decode attention spent most of its issue slots waiting on four of them per key row).
template <int W>
__device__ __forceinline__ float mmi_group_sum(float x) {
    static_assert(W == 1 || W == 2 || W == 4 || W == 8 || W == 16, "group of 1..16 lanes inside a DPP row");
    if constexpr (W >= 2) x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true));
    if constexpr (W >= 4) x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true));
    if constexpr (W >= 8) x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xf, 0xf, true));
    if constexpr (W >= 16) x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xf, 0xf, true));
    return x;
}
// The same sum over rows of 16 lanes in the order of an exchange over distances 8, 4, 2, 1 (rotations by those distances inside the row: a lane
// and its partner hold what the exchange would give them), bit for bit what the shuffles give without their trips through LDS
__device__ __forceinline__ float mmi_row_sum(float x) {
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, true));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x124, 0xf, 0xf, true));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x122, 0xf, 0xf, true));
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x121, 0xf, 0xf, true));
    return x;
}
// sum over the whole wave in the order of an exchange over distances 32, 16, 8, 4, 2, 1, bit for bit; every lane gets it
__device__ __forceinline__ float mmi_wave_sum_down(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned a0 = a[0], a1 = a[1];
    const unsigned w = __builtin_bit_cast(unsigned, __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1));
    const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    const unsigned b0 = b[0], b1 = b[1];
    return mmi_row_sum(__builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1));
}
// maximum over the four lanes l, l ^ 16, l ^ 32, l ^ 48, every one of them gets it: two exchanges of rows between registers
// (v_permlane16_swap, v_permlane32_swap: a few cycles; the same steps through the LDS crossbar wait some 120 cycles each)
__device__ __forceinline__ float mmi_rows_max(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned a0 = a[0], a1 = a[1];                           // (a bit cast of a vector's element itself takes element 0)
    const unsigned w = __builtin_bit_cast(unsigned, fmaxf(__builtin_bit_cast(float, a0), __builtin_bit_cast(float, a1)));
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    const unsigned b0 = b[0], b1 = b[1];
    return fmaxf(__builtin_bit_cast(float, b0), __builtin_bit_cast(float, b1));
}
// the sum over the same four lanes
__device__ __forceinline__ float mmi_rows_sum(float x) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned a0 = a[0], a1 = a[1];
    const unsigned w = __builtin_bit_cast(unsigned, __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1));
    const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    const unsigned b0 = b[0], b1 = b[1];
    return __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
}
// maximum over the whole wave, every lane gets it
__device__ __forceinline__ float mmi_wave_max_f32(float x) {
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true)));
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x4E, 0xf, 0xf, true)));
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x141, 0xf, 0xf, true)));
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xf, 0xf, true)));
    return mmi_rows_max(x);
}
// x of lane K of every group of W lanes (W = 4, 8, 16), to the whole group
template <int W, int K>
__device__ __forceinline__ float mmi_group_bcast(float x) {
    static_assert((W == 4 || W == 8 || W == 16) && K < W, "group of 4, 8 or 16 lanes");
    if constexpr (W == 16) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x150 + K, 0xf, 0xf, true));
    else if constexpr (W == 4) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x55 * K, 0xf, 0xf, true));
    else return __shfl(x, (int)(threadIdx.x & 56u) + K, 64);
}
// a double of another lane of the row of 16 (a DPP control)
template <int CTRL>
__device__ __forceinline__ double mmi_dpp_f64(double x) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// sum over groups of 8 consecutive lanes, every lane of the group gets it
__device__ __forceinline__ double mmi_group8_sum_f64(double x) {
    x += mmi_dpp_f64<0xB1>(x);
    x += mmi_dpp_f64<0x4E>(x);
    return x + mmi_dpp_f64<0x141>(x);
}
// the smaller of two (value, index) pairs, the lower index where the values are equal
__device__ __forceinline__ void mmi_pair_min(double& d, int& i, double od, int oi) {
    const bool take = od < d || (od == d && oi < i);
    d = take ? od : d;
    i = take ? oi : i;
}
template <int CTRL>
__device__ __forceinline__ void mmi_pair_min_dpp(double& d, int& i) {
    const double od = mmi_dpp_f64<CTRL>(d);
    mmi_pair_min(d, i, od, __builtin_amdgcn_update_dpp(0, i, CTRL, 0xf, 0xf, true));
}
// smallest pair over the four lanes l, l ^ 16, l ^ 32, l ^ 48, every one of them gets it (mmi_rows_max)
__device__ __forceinline__ void mmi_pair_min_rows(double& d, int& i) {
    auto step = [&](auto swap) __attribute__((always_inline)) {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, d);
        const auto l = swap((unsigned)u), h = swap((unsigned)(u >> 32)), j = swap((unsigned)i);
        const unsigned l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1], j0 = j[0], j1 = j[1];
        d = __builtin_bit_cast(double, ((unsigned long long)h0 << 32) | l0);
        i = (int)j0;
        mmi_pair_min(d, i, __builtin_bit_cast(double, ((unsigned long long)h1 << 32) | l1), (int)j1);
    };
    step([](unsigned v) __attribute__((always_inline)) { return __builtin_amdgcn_permlane16_swap(v, v, false, false); });
    step([](unsigned v) __attribute__((always_inline)) { return __builtin_amdgcn_permlane32_swap(v, v, false, false); });
}
// ... over the whole wave; ... over the lanes l, l ^ 8, l ^ 16, ..., l ^ 56
__device__ __forceinline__ void mmi_wave_pair_min(double& d, int& i) {
    mmi_pair_min_dpp<0xB1>(d, i);
    mmi_pair_min_dpp<0x4E>(d, i);
    mmi_pair_min_dpp<0x141>(d, i);
    mmi_pair_min_dpp<0x140>(d, i);
    mmi_pair_min_rows(d, i);
}
__device__ __forceinline__ void mmi_group8_pair_min(double& d, int& i) {
    mmi_pair_min_dpp<0x128>(d, i);
    mmi_pair_min_rows(d, i);
}
// the upper 32 lanes of a change places with the lower 32 of b
__device__ __forceinline__ void mmi_swap32(float& a, float& b) {
    const auto v = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    const unsigned v0 = v[0], v1 = v[1];
    a = __builtin_bit_cast(float, v0);
    b = __builtin_bit_cast(float, v1);
}
// the odd rows of 16 lanes of a change places with the even rows of b
__device__ __forceinline__ void mmi_swap16(float& a, float& b) {
    const auto v = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    const unsigned v0 = v[0], v1 = v[1];
    a = __builtin_bit_cast(float, v0);
    b = __builtin_bit_cast(float, v1);
}
// over the lanes that share lane % LPR: inside a row of 16 (rotations; after a step by 8 a rotation by 4 reaches lane ^ 4's value, and so on), over the wave
template <int R>
__device__ __forceinline__ float mmi_row_ror(float x) { return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + R, 0xf, 0xf, true)); }
template <int LPR>
__device__ __forceinline__ float mmi_slots_row_sum(float x) {
    static_assert(LPR == 2 || LPR == 4 || LPR == 8 || LPR == 16, "a power of two inside a row");
    if constexpr (LPR <= 8) x += mmi_row_ror<8>(x);
    if constexpr (LPR <= 4) x += mmi_row_ror<4>(x);
    if constexpr (LPR <= 2) x += mmi_row_ror<2>(x);
    return x;
}
template <int LPR>
__device__ __forceinline__ float mmi_slots_sum(float x) { return mmi_rows_sum(mmi_slots_row_sum<LPR>(x)); }
template <int LPR>
__device__ __forceinline__ float mmi_slots_max(float x) {
    static_assert(LPR == 2 || LPR == 4 || LPR == 8 || LPR == 16, "a power of two inside a row");
    if constexpr (LPR <= 8) x = fmaxf(x, mmi_row_ror<8>(x));
    if constexpr (LPR <= 4) x = fmaxf(x, mmi_row_ror<4>(x));
    if constexpr (LPR <= 2) x = fmaxf(x, mmi_row_ror<2>(x));
    return mmi_rows_max(x);
}
// sum / maximum of an unsigned over the whole wave, every lane gets it: four DPP steps inside the rows of 16, two crossbar steps
// across the rows (a six-step __shfl_xor butterfly is six dependent trips through the LDS crossbar)
__device__ __forceinline__ unsigned mmi_wave_sum_u32(unsigned x) {
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, true);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, true);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xf, 0xf, true);
    x += (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x140, 0xf, 0xf, true);
    x += mmi_shfl_xor(x, 16);
    x += mmi_shfl_xor(x, 32);
    return x;
}
__device__ __forceinline__ unsigned mmi_wave_max_u32(unsigned x) {
    unsigned o;
    o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, true); x = o > x ? o : x;
    o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, true); x = o > x ? o : x;
    o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xf, 0xf, true); x = o > x ? o : x;
    o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x140, 0xf, 0xf, true); x = o > x ? o : x;
    o = mmi_shfl_xor(x, 16); x = o > x ? o : x;
    o = mmi_shfl_xor(x, 32); x = o > x ? o : x;
    return x;
}
__device__ __forceinline__ float mmi_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
// c + a.lo * b.lo + a.hi * b.hi on two packed bf16 pairs, fp32 accumulate (v_dot2c_f32_bf16): no unpacking of either operand
typedef __bf16 mmi_bf16x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float mmi_dot2_bf16(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(mmi_bf16x2v, a), __builtin_bit_cast(mmi_bf16x2v, b), c, false);
}

// D(32x32) += A(32x2) * B(2x32), exact fp32 fma chain.  lane l: a = A[l&31][l>>5], b = B[l>>5][l&31];
// d[r] = D[(r&3) + 8*(r>>2) + 4*(l>>5)][l&31].
__device__ __forceinline__ f32x16 mmi_mfma_f32_32x32x2(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// D(16x16) += A(16x4) * B(4x16).  lane l: a = A[l&15][l>>4], b = B[l>>4][l&15]; d[r] = D[4*(l>>4)+r][l&15].
__device__ __forceinline__ f32x4 mmi_mfma_f32_16x16x4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// D(32x32) += A(32x16) * B(16x32), bf16 in / fp32 acc.  lane l: a[e] = A[l&31][8*(l>>5)+e],
// b[e] = B[8*(l>>5)+e][l&31]; d as the 32x32 map above.
__device__ __forceinline__ f32x16 mmi_mfma_bf16_32x32x16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mmi_bf16x8, a),
                                                   __builtin_bit_cast(mmi_bf16x8, b), c, 0, 0, 0);
}
// D(16x16) += A(16x32) * B(32x16).  lane l: a[e] = A[l&15][8*(l>>4)+e], b[e] = B[8*(l>>4)+e][l&15];
// d[r] = D[4*(l>>4)+r][l&15].
__device__ __forceinline__ f32x4 mmi_mfma_bf16_16x16x32(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mmi_bf16x8, a),
                                                   __builtin_bit_cast(mmi_bf16x8, b), c, 0, 0, 0);
}

// One RoPE rotation (re, im) -> (re c - im s, re s + im c) in plain (un-packed) fp32 VALU instructions, each rounded once (no
// fma), pinned by inline asm so that the compiler cannot re-form them into packed math: the same six IEEE operations the C expression
// means under -ffp-contract=off.  Written as `re * c - im * sn` the compiler packed pairs of rotations into v_pk_mul_f32 / v_pk_add_f32 with
// op_sel swizzles, one of them in place, and on gfx950 that sequence inside k_gemm_xp<32, 2, ..> (64 sessions) returned, now and then, a
// stale last element for lanes 48-63 - q / k of 16 sessions wrong in one feature, a different one from run to run
// (profiles/r05_logs/c5_trace_*.txt).  Every epilogue that rotates takes this.
__device__ __forceinline__ void mmi_rope_rotate(float re, float im, float c, float sn, float& out_re, float& out_im) {
    float a, b, d, e;
    asm volatile("v_mul_f32 %0, %1, %2" : "=v"(a) : "v"(re), "v"(c));
    asm volatile("v_mul_f32 %0, %1, %2" : "=v"(b) : "v"(im), "v"(sn));
    asm volatile("v_mul_f32 %0, %1, %2" : "=v"(d) : "v"(re), "v"(sn));
    asm volatile("v_mul_f32 %0, %1, %2" : "=v"(e) : "v"(im), "v"(c));
    asm volatile("v_sub_f32 %0, %1, %2" : "=v"(out_re) : "v"(a), "v"(b));
    asm volatile("v_add_f32 %0, %1, %2" : "=v"(out_im) : "v"(d), "v"(e));
}

// ---- fp8 (OCP e4m3fn on gfx950: 4 exponent bits, bias 7, 3 mantissa bits, max 448, no infinity) -----------------------
// four fp32 -> four fp8 bytes (byte i = value i), round-to-nearest-even, clamped to +-448 first so that the result does not
// depend on the conversion's overflow mode
__device__ __forceinline__ uint32_t mmi_cvt_fp8x4(float a, float b, float c, float d) {
    a = __builtin_amdgcn_fmed3f(a, -448.f, 448.f);
    b = __builtin_amdgcn_fmed3f(b, -448.f, 448.f);
    c = __builtin_amdgcn_fmed3f(c, -448.f, 448.f);
    d = __builtin_amdgcn_fmed3f(d, -448.f, 448.f);
    int r = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    r = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, r, true);
    return (uint32_t)r;
}
// four fp8 bytes -> four fp32 (exact)
__device__ __forceinline__ void mmi_fp8x4_to_f32(uint32_t w, float* o) {
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    o[0] = lo[0]; o[1] = lo[1]; o[2] = hi[0]; o[3] = hi[1];
}
// four fp8 bytes -> four bf16 (exact: e4m3 has 3 mantissa bits)
__device__ __forceinline__ u32x2 mmi_fp8x4_to_bf16(uint32_t w) {
    return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false)),
                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true))};
}
// D(32x32) += A(32x16) * B(16x32), fp8 in / fp32 acc.  Same element map as the bf16 32x32x16 form with one byte per
// element: lane l: a[e] = A[l&31][8*(l>>5)+e], b[e] = B[8*(l>>5)+e][l&31] (8 bytes per operand per lane).
__device__ __forceinline__ f32x16 mmi_mfma_fp8_32x32x16(u32x2 a, u32x2 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), c, 0, 0, 0);
}
// D(16x16) += A(16x32) * B(32x16): lane l: a[e] = A[l&15][8*(l>>4)+e], b[e] = B[8*(l>>4)+e][l&15].
__device__ __forceinline__ f32x4 mmi_mfma_fp8_16x16x32(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), c, 0, 0, 0);
}

// ---- int8 x int8 on the matrix core (the reference's bitsandbytes int8 matmul, utils/quantize.py:24-40) ----
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
// D(32x32) += A(32x32) * B(32x32), int8 in / int32 acc (v_mfma_i32_32x32x32_i8): 16 bytes per operand per lane.  Both operands
// are packed with the SAME (lane, byte) -> k map (k_pack_w_i8: lane (i, kq), byte e <-> k = 32 kp + 16 (e >> 3) + 8 kq + (e & 7)),
// and the sum over k does not depend on the order the hardware walks it in.  d as the 32x32 map of the bf16 form.
__device__ __forceinline__ i32x16 mmi_mfma_i8_32x32x32(u32x4 a, u32x4 b, i32x16 c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}
// D(16x16) += A(16x64) * B(64x16) (v_mfma_i32_16x16x64_i8); d[r] = D[4*(l>>4)+r][l&15].
__device__ __forceinline__ i32x4 mmi_mfma_i8_16x16x64(u32x4 a, u32x4 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a), __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}
// the low bytes of four words -> one word (byte i = low byte of argument i): two v_perm_b32 + one
__device__ __forceinline__ uint32_t mmi_pack_low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    const uint32_t ab = __builtin_amdgcn_perm(b, a, 0x0c0c0400u);      // bytes: [a.0, b.0, 0, 0]  (selector bytes 0-3 index the second operand, 4-7 the first, 0x0c = zero)
    const uint32_t cd = __builtin_amdgcn_perm(d, c, 0x04000c0cu);      // bytes: [0, 0, c.0, d.0]
    return ab | cd;
}
// round-half-even to the nearest integer (v_rndne_f32), the rounding of bitsandbytes' int8_vectorwise_quant
__device__ __forceinline__ float mmi_rint(float x) { return __builtin_rintf(x); }

// "Last arriver finishes" inside one launch (k_lm_attn_wave's ring split): a workgroup publishes its partial result with plain
// stores, then ONE lane releases at agent scope (L2 write-back), drains, and bumps the arrival counter; the workgroup that sees
// the final count acquires at agent scope (invalidates its CU's L1) and reads the others' partials with plain loads - the
// producer / consumer form that is valid across XCDs.  Call from ONE thread, between two __syncthreads().
__device__ __forceinline__ unsigned mmi_arrive_release(unsigned* counter) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (the compiler may drop the fence's own wait: keep one it cannot see through)
    return __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void mmi_acquire_agent() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent"); }
__device__ __forceinline__ void mmi_store_relaxed_agent(unsigned* p, unsigned v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The instruction scheduler moves nothing across this point: keeps a batch of loads issued ahead of the products that consume the batch
// before it (left alone it sinks each load to its use when registers are short, and the loads then wait for one another)
__device__ __forceinline__ void mmi_sched_barrier() { __builtin_amdgcn_sched_barrier(0); }
// x is computed here and unknown from here on.  Without it the compiler moves arithmetic whose result is only used much later down to that
// use, across barriers, and keeps all the operands it read from LDS until then; and it computes the addresses of all a kernel's phases, where
// they follow from one lane index, at the kernel's start, and keeps those
template <class T>
__device__ __forceinline__ void mmi_here(T& x) { asm volatile("" : "+v"(x)); }
// a value that is the same in every lane (a wave index, what was loaded through one), told to the compiler: it stays in scalar registers,
// and loads addressed by it are scalar loads - they do not queue behind the vector loads in flight
__device__ __forceinline__ int mmi_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
// a load from memory that nothing writes while the kernel runs: by a uniform address a scalar load, also where the compiler cannot rule out that
// one of the kernel's stores meets it
__device__ __forceinline__ int mmi_load_const(const int* p) { return *(const __attribute__((address_space(4))) int*)p; }
// true in every lane when any lane's flag is set
__device__ __forceinline__ bool mmi_any(bool v) { return __any(v) != 0; }

// 16 bytes per lane from global memory into LDS without a register in between: lane l's land at lds[at + l] (lds, at: the same in every
// lane).  Nothing waits for them but mmi_wait_loads (the compiler does not know of them), which counts this wave's loads in the order of
// their issue, and behind it a barrier for the other waves' ones.  First form: base (uniform) + offset per lane in bytes.
// (m0 is named as overwritten so that no value of the compiler's own stays in it; it notes that the register is a reserved one)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ unsigned mmi_lds_addr(const void* p) { return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)p; }
__device__ __forceinline__ void mmi_load_lds(const void* base, unsigned off, u32x4* lds, int at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(mmi_lds_addr(lds) + 16u * (unsigned)at), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void mmi_load_lds(const u32x4* from, u32x4* lds, int at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(mmi_lds_addr(lds) + 16u * (unsigned)at), "v"(from) : "memory", "m0");
}
#pragma clang diagnostic pop
// until at most N of this wave's loads are in flight
template <int N>
__device__ __forceinline__ void mmi_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// the workgroup's waves meet; unlike __syncthreads it does not wait for loads in flight (LDS reads and writes of this wave are done)
__device__ __forceinline__ void mmi_meet() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// streamed-once weights: non-temporal so they do not evict the activations / KV the other kernels reuse
__device__ __forceinline__ u32x4 mmi_load_nt(const u32x4* p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ f32x4 mmi_load_nt(const f32x4* p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ void mmi_store_nt(f32x4* p, f32x4 v) { __builtin_nontemporal_store(v, p); }

__device__ __forceinline__ float mmi_rsqrtf(float x) { return 1.0f / sqrtf(x); }  // IEEE, matches torch.rsqrt closely
// natural log on the hardware's v_log_f32 (log2, ~1 ulp) - for the sampler's own noise only (nothing the reference's arithmetic
// fixes): the library logf is ~25 dependent instructions on a one-wave-per-SIMD kernel that runs at ~9 cycles per instruction
// base-2 exponential and logarithm in hardware (v_exp_f32, v_log_f32: ~1 ulp, denormals flushed)
__device__ __forceinline__ float mmi_fast_exp2f(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float mmi_fast_log2f(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float mmi_fast_rcpf(float x) { return __builtin_amdgcn_rcpf(x); }      // ~1 ulp
__device__ __forceinline__ float mmi_fast_logf(float x) { return __logf(x); }
__device__ __forceinline__ unsigned mmi_atomic_add(unsigned* p, unsigned v) { return atomicAdd(p, v); }

// Cross-stream hand-off flags (duplex.hip): a monotonic counter in device memory, published with release semantics by a
// one-thread kernel at the end of a producer stream's work and polled by a one-wave kernel at the head of the consumer's.
// Why not hipStreamWaitEvent: a wait that stays PENDING makes the command processor poll the producer queue's signal, which
// slows every dependent launch of the producer (1.60 -> 2.77 ms for a chain of 1000 tiny kernels on this stack; a resident
// polling wave costs 1.71 ms - scripts/stream_probe.hip test 1e, profiles/r03_logs/stream_probe.txt).
// constant-rate device clock (100 MHz on gfx950): the pipeline's diagnostic stamps
__device__ __forceinline__ long mmi_wall_clock() { return (long)wall_clock64(); }
__device__ __forceinline__ void mmi_flag_publish(long* flag, long v) {
    __threadfence();
    __hip_atomic_store(flag, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}
// The poll is a RELAXED agent-scope load (it bypasses the non-coherent cache levels by itself); the acquire fence - on gfx950 an
// invalidation of the polling XCD's L2, which would evict the working set of every kernel running there once per iteration -
// comes once, after the flag was seen.
__device__ __forceinline__ void mmi_flag_wait(const long* flag, long v) {
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < v) __builtin_amdgcn_s_sleep(96);
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
}
