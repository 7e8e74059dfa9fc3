// Mimi codec kernels for gfx950 (fp32, like the reference: loaders.get_mimi never casts, loaders.py:353).
//
// Data layout in HBM
//   activations   [B][C][H + T] fp32, time contiguous ("conv layout", same as the reference's [B,C,T]).
//                 The first H columns of a buffer are the causal history of its consumer conv
//                 (the reference's `previous` ring state, conv.py:161-169,245-274); the producer writes
//                 its T new columns behind them and k_commit_history shifts the last H columns to the
//                 front once the frame is done (only for rows whose exec mask is set).
//   conv weights  packed at load into MFMA A-fragment order for v_mfma_f32_32x32x2_f32:
//                 P[mt][q][lane][e] = W[mt*32 + (lane&31)][(q*4+e)*2 + (lane>>5)]  (zero padded),
//                 so that a wave's 16-byte-per-lane load is one contiguous 1 KiB read feeding 4 MFMAs.
//   codebooks     E[level][bins][D] fp32 + ||e||^2 in fp64.
//   KV ring       [layer][2][B][H][cap][D] fp32 (transformer.py:196-288).
//
// Every conv / linear of the codec (SEANet convs, the GEMM half of the transposed convs, the 1x1
// RVQ projections, the transformer's linears) is the implicit GEMM
//   out[co][n=(b,t)] = sum_{kd=(ci,k)} W[co][kd] * act(in[b][ci][t*S + k])
// on the fp32 MFMA (an exact fma chain, so results track the fp32 reference to rounding order); see k_conv_wide /
// k_gemm_f32 below.  Activations that feed k_gemm_f32 are additionally kept as a packed B operand:
//   Bp[nt][q][lane][e] = act(in)[kd = (q*4+e)*2 + (lane>>5)][n = nt*32 + (lane&31)]
#pragma once
#include "mmi_common.h"

// ------------------------------------------------------------------------------------------------
// weight packing
// ------------------------------------------------------------------------------------------------
// P[mt][q][lane][e] = W[m*sm + kd*sk], m = mt*32 + (lane&31), kd = (q*4+e)*2 + (lane>>5)
__global__ void k_pack_a_f32(const float* __restrict__ W, float* __restrict__ P, int M, int Kd, long sm, long sk,
                             int Mt, int Q) {
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long total = (long)Mt * Q * 256;
    if (idx >= total) return;
    int e = (int)(idx & 3);
    int lane = (int)((idx >> 2) & 63);
    long rest = idx >> 8;
    int q = (int)(rest % Q);
    int mt = (int)(rest / Q);
    int m = mt * 32 + (lane & 31);
    int kd = (q * 4 + e) * 2 + (lane >> 5);
    float v = 0.f;
    if (m < M && kd < Kd) v = W[(long)m * sm + (long)kd * sk];
    P[idx] = v;
}

// dst[r*dld + c] = src[r*sld + c]  (row-block copy used to concatenate weight matrices / stage I/O)
__global__ void k_copy2d_f32(const float* __restrict__ src, long sld, float* __restrict__ dst, long dld, int rows,
                             int cols) {
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)rows * cols) return;
    int r = (int)(idx / cols), c = (int)(idx % cols);
    dst[(long)r * dld + c] = src[(long)r * sld + c];
}

// codebook = embedding_sum / clamp(cluster_usage, eps)[:, None]   (core_vq.py:178-186); e2 = ||e||^2 (fp64)
__global__ void k_codebook_prepare(const float* __restrict__ esum, const float* __restrict__ usage,
                                   float* __restrict__ E, double* __restrict__ e2, int bins, int D, float eps) {
    int c = blockIdx.x;
    if (c >= bins) return;
    float u = usage[c];
    u = u < eps ? eps : u;
    MMI_SHARED double red[64];
    double acc = 0.0;
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        float v = esum[(long)c * D + d] / u;
        E[(long)c * D + d] = v;
        acc += (double)v * (double)v;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int i = 0; i < (int)blockDim.x; ++i) s += red[i];
        e2[c] = s;
    }
}

// ------------------------------------------------------------------------------------------------
// implicit-GEMM conv / linear
// ------------------------------------------------------------------------------------------------
// out[co][n=(b,t)] = sum_{kd=(ci,k)} W[co][kd] * act(in[b][ci][t*S + k]), fp32 MFMA 32x32x2 (exact fma chain).
//   k_conv_wide  (N = B*T_out > 128 columns: SEANet layers at audio rate).  A wave owns 32 columns x MTB m-tiles x a
//                K-slice; lane (j, h) gathers exactly the B-operand elements its own MFMA lane consumes
//                (column j, reduction index kd = 2q+h), applies ELU once, and reuses them for the MTB m-tiles.
//                The input offsets (ci*x_ld + k) of the next quad are a few additions away (ConvWalk).
//   k_conv_cols  the same sums, bit for bit, in groups of frames: a wave takes all slices of a reduction in turn.
//   k_gemm_f32   (N <= 128: the 12.5/25 Hz layers - last strided convs, resampling, RVQ projections; weights
//                dominate).  Same shape as the LM's weight-streaming GEMM: one m-tile per workgroup, K split over
//                waves (+ workgroups), activations pre-packed into B-fragment order by k_pack_b_f32 (im2col + ELU +
//                replicate padding) or by the producing kernel.
//   k_conv_few   the same sums, bit for bit, for few streams (operands from the input as it lies) and for small products of a packed
//                operand: 16 x 16 tiles.
// The transformers' linears have kernels of their own (k_mimi_lin, k_mimi_lin_rows).
// n / d for 0 <= n < 2^20 and 1 <= d < 2^20 (column and tap indices) as one multiply-high and a shift: an integer division costs
// ~30 instructions, and the small kernels here are instruction bound.  magic = ceil(2^(32 + shift) / d), 0 means d == 1; exact while
// n d < 2^(32 + shift), hence the 8 more bits (which still fit the magic number) from d = 2^11 on.
MMI_HD unsigned mmi_div_shift(int d) { return d < (1 << 11) ? 0u : 8u; }
MMI_HD unsigned mmi_div_magic(int d, unsigned shift = 0u) { return d <= 1 ? 0u : (unsigned)(((0x100000000ull << shift) + (unsigned)d - 1) / (unsigned)d); }
MMI_HD int mmi_fast_div(int n, unsigned magic, unsigned shift = 0u) {
    return magic == 0u ? n : (int)((unsigned)(((unsigned long long)(unsigned)n * magic) >> 32) >> shift);
}
enum { MMI_GOUT_NATURAL = 0, MMI_GOUT_PARTIAL = 1 };

struct ConvGemmArgs {
    const float* x;       // input [B][Cin][x_ld]; position p of a row = history (p < H) then the T new columns
    long x_bstride;       // Cin * x_ld
    int x_ld;
    int x_off;            // first column this conv reads (H_buffer - (K - S)); normally 0
    int H;                // history columns in front of the new data (for replicate-first)
    const float* wpk;     // packed weights
    const float* bias;    // [Cout] or null
    float* out;           // [B][Cout][out_ld], written at column out_off + t
    int out_ld, out_off;
    const float* res;     // residual [B][Cout][res_ld] read at res_off + t, or null
    int res_ld, res_off;
    const uint8_t* first; // replicate-pad flags [B] or null (conv.py:253-259)
    const uint8_t* exec;  // exec mask [B] (only read with `first`)
    int B, Cin, Cout, K, S, T_out;
    unsigned T_magic, K_magic;   // mmi_div_magic(T_out), mmi_div_magic(K)
    int Mt, Q;            // M tiles of 32, packed k-quads (Kdim_pad / 8)
    int Ntot;             // B * T_out
    int elu_in;           // apply ELU(alpha=1) to every loaded input (seanet.py:63,205,222)
    // ELU hoisted out of the consumers: every SEANet conv but the first reads ELU(x) (seanet.py:63,205,222), and an audio-rate
    // conv reads each input K * (Cout / 32) times, so the PRODUCER applies it once per element: elu_out = 1 stores ELU(result)
    // instead of the result (buffers whose only readers are such convs), out2 != null additionally stores ELU(result) there
    // (same geometry as `out`; block inputs, which the residual connection also needs raw).  Same function on the same values
    // as applying it at the consumer's load - bit-identical.
    int elu_out;
    float* out2;
    // --- filled in by the engine's planner
    const float* bp;      // k_gemm_f32: packed activations [ceil(N/32)][Q][64][4]
    int x_packed;         // the producer already wrote `bp` (no k_pack_b_f32 launch)
    int out_mode;         // MMI_GOUT_*
    float* outp;          // packed B operand of the consumer, also stored: [ceil(N/32)][outQ][64][4], or with outJ the transformers'
    int outQ, outJ;       //   fragments of 16 columns (mmi_lin_index)
    float* partial;       // GOUT_PARTIAL: [gridDim.y][Mt*32][Npad] raw sums, finished by k_conv_finish
    int Npad;
    // groups of frames: T_magic = mmi_div_magic(T_out, T_shift), 0 where T_out < 2^11; quads per workgroup of a split reduction (Q: not split)
    unsigned T_shift;
    int q_blk;
};

__device__ __forceinline__ float mmi_elu(float v) { return v > 0.f ? v : expm1f(v); }
__device__ __forceinline__ float mmi_gelu_erf(float v) { return 0.5f * v * (1.0f + erff(v * 0.70710678118654752440f)); }

// index of element (kd, n) in a packed B operand with Q k-quads
__device__ __forceinline__ long mmi_bp_index(int kd, int n, int Q) {
    return ((((long)(n >> 5) * Q + (kd >> 3)) * 64) + (kd & 1) * 32 + (n & 31)) * 4 + ((kd & 7) >> 1);
}

// element (k, n) of a transformer linear's operand, fragments of 16 columns x 16 reduction indices (J of them): lane (k & 3, n) of
// fragment k / 16 holds k = 4 e + its own quarter at element e, so that four v_mfma_f32_16x16x4_f32 walk them in rising order
MMI_HD long mmi_lin_index(int k, int n, int J) {
    return ((((long)(n >> 4) * J + (k >> 4)) * 64) + (k & 3) * 16 + (n & 15)) * 4 + ((k >> 2) & 3);
}

// bias / residual, then the store to [B][Cout][out_ld] - shared by the epilogues.
// NV results of one thread are finished together: all bias / scale / residual loads are issued first (under branches
// that are uniform for the launch), so that the epilogue costs one memory round trip instead of NV of them.
template <int NV>
__device__ __forceinline__ void mmi_conv_ask_n(const ConvGemmArgs& a, const int (&co)[NV], const int (&b)[NV], const int (&t)[NV],
                                               const bool (&ok)[NV], long (&row)[NV], float (&bia)[NV], float (&rsv)[NV]) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int cc = ok[i] ? co[i] : 0;
        row[i] = (long)(ok[i] ? b[i] : 0) * a.Cout + cc;
        bia[i] = 0.f; rsv[i] = 0.f;
    }
    if (a.bias) {
#pragma unroll
        for (int i = 0; i < NV; ++i) bia[i] = a.bias[ok[i] ? co[i] : 0];
    }
    if (a.res) {
#pragma unroll
        for (int i = 0; i < NV; ++i) rsv[i] = a.res[row[i] * a.res_ld + a.res_off + (ok[i] ? t[i] : 0)];
    }
}
template <int NV>
__device__ __forceinline__ void mmi_conv_put_n(const ConvGemmArgs& a, const int (&co)[NV], const int (&b)[NV], const int (&t)[NV],
                                               const bool (&ok)[NV], const long (&row)[NV], const float (&bia)[NV], const float (&rsv)[NV], float (&v)[NV]) {
    // launch-uniform flags are tested once per group of NV values, not per value: these kernels are instruction bound, and a
    // per-value maze of scalar branches (with the erf and expm1 bodies in line) was a third of a residual block's time
    if (a.bias) {
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] += bia[i];
    }
    if (a.res) {
#pragma unroll
        for (int i = 0; i < NV; ++i) v[i] = rsv[i] + v[i];
    }
    long at[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) at[i] = row[i] * a.out_ld + a.out_off + (ok[i] ? t[i] : 0);
    if (a.out2) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (ok[i]) { a.out[at[i]] = v[i]; a.out2[at[i]] = mmi_elu(v[i]); }
    } else if (a.elu_out) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            v[i] = mmi_elu(v[i]);
            if (ok[i]) a.out[at[i]] = v[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (ok[i]) a.out[at[i]] = v[i];
    }
    // also stored as the packed operand of the consumer (what `out` holds: the ELU'd value where that is what is stored): the encoder's
    // last conv for its transformer, the decoder's first conv for the first transposed-conv GEMM, the latent for the RVQ input projection -
    // no launch that packs in between
    if (a.outp && a.out_mode == MMI_GOUT_NATURAL) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (ok[i]) a.outp[a.outJ ? mmi_lin_index(co[i], b[i] * a.T_out + t[i], a.outJ) : mmi_bp_index(co[i], b[i] * a.T_out + t[i], a.outQ)] = v[i];
    }
}

template <int NV>
__device__ __forceinline__ void mmi_conv_store_n(const ConvGemmArgs& a, const int (&co)[NV], const int (&b)[NV], const int (&t)[NV],
                                                 const bool (&ok)[NV], float (&v)[NV]) {
    float bia[NV], rsv[NV];
    long row[NV];
    mmi_conv_ask_n<NV>(a, co, b, t, ok, row, bia, rsv);
    mmi_conv_put_n<NV>(a, co, b, t, ok, row, bia, rsv, v);
}

// The input's places (bytes from a.x on) of the four values of a quad that a lane of the 32 x 32 form takes, kd = 8 q + 2 e + kh for column
// (b, t): the next quad's are a few additions away, where a table of offsets is one more load in front of the gathers (and a launch per conv
// that fills it whenever a stream starts).  Reduction indices past the last one read some valid place: they meet zero weights.
struct ConvWalk {
    unsigned off[4], top, step, carry;
    int tap[4], tap_step;
    __device__ __forceinline__ void begin(const ConvGemmArgs& a, int b, int t, int q, int kh) {
        const unsigned base = 4u * (unsigned)(b * (int)a.x_bstride + a.x_off + t * a.S);
        const int c8 = mmi_fast_div(8, a.K_magic);
        tap_step = 8 - c8 * a.K;
        step = 4u * (unsigned)(c8 * a.x_ld + tap_step);
        carry = 4u * (unsigned)(a.x_ld - a.K);
        top = base + 4u * (unsigned)((a.Cin - 1) * a.x_ld + a.K - 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int kd = q * 8 + 2 * e + kh, ci = mmi_fast_div(kd, a.K_magic);
            tap[e] = kd - ci * a.K;
            off[e] = base + 4u * (unsigned)(ci * a.x_ld + tap[e]);
        }
    }
    __device__ __forceinline__ float at(const ConvGemmArgs& a, int e) const {
        return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.x) + min(off[e], top));
    }
    __device__ __forceinline__ void advance(const ConvGemmArgs& a, bool on = true) {      // (selected, not branched around: the loads stay in one block)
        const int ts = on ? tap_step : 0;
        const unsigned st = on ? step : 0u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            tap[e] += ts;
            off[e] += st;
            const bool over = tap[e] >= a.K;
            tap[e] -= over ? a.K : 0;
            off[e] += over ? carry : 0u;
        }
    }
};

// GROUP: several frames of a stream at once - more columns per stream (T_shift), and the reduction also split over gridDim.z workgroups
// where the frame program splits it (k_conv_finish adds their sums), cut as k_gemm_f32 cuts it
template <int MTB, int W, int U, bool ELU_IN, bool GROUP>
__global__ __launch_bounds__(W * 64) void k_conv_wide(ConvGemmArgs a) {
    const unsigned tsh = GROUP ? a.T_shift : 0u;
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const int jl = lane & 31, kh = lane >> 5;
    const int n = (int)blockIdx.x * 32 + jl;
    const int mt0 = (int)blockIdx.y * MTB;
    const bool nvalid = n < a.Ntot;
    const int nn = nvalid ? n : 0;
    const int b = mmi_fast_div(nn, a.T_magic, tsh), t = nn - b * a.T_out;
    const int qb0 = GROUP ? min(a.Q, (int)blockIdx.z * a.q_blk) : 0, qb1 = GROUP ? min(a.Q, qb0 + a.q_blk) : a.Q;
    const int qper = (qb1 - qb0 + W - 1) / W;
    const int q0 = min(qb1, qb0 + wave * qper), q1 = min(qb1, q0 + qper);

    f32x16 acc[MTB];
#pragma unroll
    for (int m = 0; m < MTB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = 0.f;
    const f32x4* wp[MTB];
#pragma unroll
    for (int m = 0; m < MTB; ++m) wp[m] = reinterpret_cast<const f32x4*>(a.wpk) + (long)min(mt0 + m, a.Mt - 1) * a.Q * 64 + lane;
    ConvWalk in;
    in.begin(a, b, t, q0, kh);

    // groups of U k-quads, double buffered: the gathers / weight fragments of group g+1 are in flight while group g
    // runs on the matrix core.  Loads past the slice are clamped to its last quad and their MFMAs skipped.
    f32x4 avA[U][MTB], avB[U][MTB];
    float bvA[U][4], bvB[U][4];
#define MMI_W_LOAD(AV, BV, qb)                                                                      \
    _Pragma("unroll") for (int u = 0; u < U; ++u) {                                                 \
        const int qq = min((qb) + u, q1 - 1);                                                       \
        /* plain unconditional gathers (a conditional load would be serialised behind s_waitcnt vmcnt(0)); columns past Ntot  \
           are computed and discarded */                                                            \
        _Pragma("unroll") for (int e = 0; e < 4; ++e) BV[u][e] = in.at(a, e);                       \
        in.advance(a);                                                                              \
        _Pragma("unroll") for (int m = 0; m < MTB; ++m) AV[u][m] = wp[m][(long)qq * 64];           \
    }
#define MMI_W_MMA(AV, BV, qb)                                                                       \
    _Pragma("unroll") for (int u = 0; u < U; ++u) {                                                 \
        if ((qb) + u < q1) {                                                                        \
            _Pragma("unroll") for (int e = 0; e < 4; ++e) {                                         \
                const float v = (ELU_IN && a.elu_in) ? mmi_elu(BV[u][e]) : BV[u][e];                \
                _Pragma("unroll") for (int m = 0; m < MTB; ++m) acc[m] = mmi_mfma_f32_32x32x2(AV[u][m][e], v, acc[m]); \
            }                                                                                       \
        }                                                                                           \
    }
    const int G = (q1 - q0 + U - 1) / U;
    if (G > 0) {
        MMI_W_LOAD(avA, bvA, q0);
        int g = 0;
        for (; g + 2 < G; g += 2) {
            MMI_W_LOAD(avB, bvB, q0 + (g + 1) * U);
            MMI_W_MMA(avA, bvA, q0 + g * U);
            MMI_W_LOAD(avA, bvA, q0 + (g + 2) * U);
            MMI_W_MMA(avB, bvB, q0 + (g + 1) * U);
        }
        if (G - g == 2) {
            MMI_W_LOAD(avB, bvB, q0 + (g + 1) * U);
            MMI_W_MMA(avA, bvA, q0 + g * U);
            MMI_W_MMA(avB, bvB, q0 + (g + 1) * U);
        } else {
            MMI_W_MMA(avA, bvA, q0 + g * U);
        }
    }
#undef MMI_W_LOAD
#undef MMI_W_MMA

    if (W > 1) {   // split-K reduction across the waves, fixed order
        MMI_DYN_SHARED(float, red);
        const int NE = MTB * 16 * 64;
#pragma unroll
        for (int m = 0; m < MTB; ++m)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[wave * NE + (m * 16 + r) * 64 + lane] = acc[m][r];
        __syncthreads();
        constexpr int NVT = MTB * 16 / W;                      // results per thread (W divides 16)
        constexpr int NV = NVT < 8 ? NVT : 8;                  // finished 8 at a time (register budget)
#pragma unroll 1
        for (int i0 = 0; i0 < NVT; i0 += NV) {
            int co[NV], bb[NV], tt[NV];
            bool ok[NV];
            float v[NV];
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int e = (int)threadIdx.x + (i0 + i) * W * 64;
                const int le = e & 63, r = (e >> 6) & 15, m = e >> 10;
                const int nn2 = (int)blockIdx.x * 32 + (le & 31);
                co[i] = (mt0 + m) * 32 + (r & 3) + 8 * (r >> 2) + 4 * (le >> 5);
                ok[i] = nn2 < a.Ntot && co[i] < a.Cout;
                const int n3 = ok[i] ? nn2 : 0;
                bb[i] = mmi_fast_div(n3, a.T_magic, tsh);
                tt[i] = n3 - bb[i] * a.T_out;
                float s = 0.f;
                for (int w = 0; w < W; ++w) s += red[w * NE + e];
                v[i] = s;
                if (GROUP && a.out_mode == MMI_GOUT_PARTIAL && (mt0 + m) < a.Mt) a.partial[((long)blockIdx.z * a.Mt * 32 + co[i]) * a.Npad + nn2] = s;
            }
            if (GROUP && a.out_mode == MMI_GOUT_PARTIAL) continue;
            mmi_conv_store_n<NV>(a, co, bb, tt, ok, v);
        }
        return;
    }
#pragma unroll
    for (int m = 0; m < MTB; ++m) {
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += 8) {
            int co[8], bb[8], tt[8];
            bool ok[8];
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int r = r0 + i;
                co[i] = (mt0 + m) * 32 + (r & 3) + 8 * (r >> 2) + 4 * kh;
                ok[i] = nvalid && co[i] < a.Cout;
                bb[i] = b; tt[i] = t;
                v[i] = acc[m][r];
            }
            mmi_conv_store_n<8>(a, co, bb, tt, ok, v);
        }
    }
}

// k_conv_wide's sums by waves of their own: a wave owns 32 columns x MTB m-tiles and takes the `pieces` of its reduction - what k_conv_wide's waves
// would split it into - one after the other, each from zero, and adds them up in the same order: the same bits without the exchange through LDS.
// Four waves of a workgroup own neighbouring column tiles and read the same weights.  grid (ceil(column tiles / 4), ceil(Mt / MTB), ks).
// Bound by the matrix core where a wave's reduction is long; what it loses are the gathers
// (one load per value and wave, met by MTB m-tiles).
// A file's 129 frames: 64 -> 128, K 8 on 61920 columns 151 -> 98 us (83 TFLOP/s), 128 -> 256, K 10 on 12384 144 -> 117, 512 -> 3072 on 2064 103 -> 87,
// 256 -> 1280 on 12384 143 -> 99, 128 -> 512 on 61920 144 -> 112; stores bound the convs of few products (32 -> 64 on 247680: 59 -> 43).
template <int MTB, int U>
__global__ __launch_bounds__(256, 2) void k_conv_cols(ConvGemmArgs a, int pieces) {
    const int wave = mmi_uniform((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63, jl = lane & 31, kh = lane >> 5;
    const int nt = (int)blockIdx.x * 4 + wave, n = nt * 32 + jl, mt0 = (int)blockIdx.y * MTB;
    if (nt * 32 >= a.Ntot) return;
    const bool nvalid = n < a.Ntot;
    const int nn = nvalid ? n : 0, b = mmi_fast_div(nn, a.T_magic, a.T_shift), t = nn - b * a.T_out;
    const int q0 = min(a.Q, (int)blockIdx.z * a.q_blk), q1 = min(a.Q, q0 + a.q_blk), qper = max((q1 - q0 + pieces - 1) / pieces, 1);
    const f32x4* wp[MTB];
#pragma unroll
    for (int m = 0; m < MTB; ++m) wp[m] = reinterpret_cast<const f32x4*>(a.wpk) + (long)min(mt0 + m, a.Mt - 1) * a.Q * 64 + lane;
    ConvWalk in;
    in.begin(a, b, t, q0, kh);
    f32x16 acc[MTB], sum[MTB];
#pragma unroll
    for (int m = 0; m < MTB; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[m][r] = sum[m][r] = 0.f;
    f32x4 avA[U][MTB], avB[U][MTB], bvA[U], bvB[U];
    struct At { int q, end; };                               // a group of U quads: its first one, the end of its piece (where the group ends too)
    auto after = [&](const At& at) __attribute__((always_inline)) {
        At n = {at.q + U, at.end};
        if (n.q >= at.end) { n.q = at.end; n.end = min(q1, at.end + qper); }
        return n;
    };
    // no load is conditional, so that the wait in front of a product covers the older group only
    auto load = [&](f32x4 (&av)[U][MTB], f32x4 (&bv)[U], const At& at) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int qq = min(at.q + u, q1 - 1);
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[u][e] = in.at(a, e);
            in.advance(a, at.q + u < at.end);
#pragma unroll
            for (int m = 0; m < MTB; ++m) av[u][m] = wp[m][(long)qq * 64];
        }
    };
    auto mma = [&](f32x4 (&av)[U][MTB], f32x4 (&bv)[U], const At& at) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool on = at.q + u < at.end;               // (quads past the piece's end meet zeros: a branch around them would cost a wait for all loads)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = on ? bv[u][e] : 0.f;
#pragma unroll
                for (int m = 0; m < MTB; ++m) acc[m] = mmi_mfma_f32_32x32x2(av[u][m][e], v, acc[m]);
            }
        }
        if (pieces > 1 && at.q + U >= at.end)
#pragma unroll
            for (int m = 0; m < MTB; ++m)
#pragma unroll
                for (int r = 0; r < 16; ++r) { sum[m][r] += acc[m][r]; acc[m][r] = 0.f; }
    };
    if (q0 < q1) {
        At cur = {q0, min(q1, q0 + qper)};
        load(avA, bvA, cur);
        At next = after(cur);
        while (next.q < q1) {                                // (one way out, at the end of a pair: a break between its halves costs a wait for all loads)
            load(avB, bvB, next);
            mmi_sched_barrier();
            mma(avA, bvA, cur);
            cur = after(next);
            load(avA, bvA, cur);
            mmi_sched_barrier();
            mma(avB, bvB, next);
            next = after(cur);
        }
        if (cur.q < q1) mma(avA, bvA, cur);
    }
#pragma unroll
    for (int m = 0; m < MTB; ++m) {
        if (mt0 + m >= a.Mt) break;
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += 8) {
            int co[8], bb[8], tt[8];
            bool ok[8];
            float v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int r = r0 + i;
                co[i] = (mt0 + m) * 32 + (r & 3) + 8 * (r >> 2) + 4 * kh;
                ok[i] = nvalid && co[i] < a.Cout;
                bb[i] = b; tt[i] = t;
                v[i] = pieces > 1 ? sum[m][r] : acc[m][r];
                if (a.out_mode == MMI_GOUT_PARTIAL) a.partial[((long)blockIdx.z * a.Mt * 32 + co[i]) * a.Npad + n] = v[i];
            }
            if (a.out_mode != MMI_GOUT_PARTIAL) mmi_conv_store_n<8>(a, co, bb, tt, ok, v);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// SEANet residual block in ONE launch (seanet.py:31-77 SEANetResnetBlock, true_skip):
//     y = x + conv1x1(ELU(convK(ELU(x))))        convK: C -> C/2 (K = residual_kernel_size, dilation 1), conv1x1: C/2 -> C
// at audio rate (N = B*T > 128 columns).  As two k_conv_wide launches the block writes the hidden tensor to HBM and reads it
// back, and pays two launches for ~1 GFLOP; here a workgroup owns 32 columns and MT1 = ceil((C/2) / 32) waves:
//   stage 0  the tile's input window (Cin x (32 + K - 1) floats of ONE session: T % 32 == 0) is staged in LDS with coalesced row
//            loads that are all in flight at once - one memory round trip for the whole tile, where the gather loop of
//            k_conv_wide pays one per group of k-quads (measured: ~4 us per group at one wave per SIMD)
//   stage 1  wave w computes hidden m-tile w over the whole reduction, B operand from LDS (ds_read at table offsets): acc1
//   hand-off h = ELU(acc1 + b1) stays in the accumulator layout: lane (j, hh) holds hidden rows 32w + 8(r>>2) + 4hh + (r&3),
//            r = 0..15, of its own column j.  The second conv's reduction index is free to be ANY order, so its weights are packed
//            (k_pack_a_f32_hperm) such that MFMA k-slot (qq, hh) of the 32x32x2 B operand IS hidden row 32(qq/16) + 8((qq%16)>>2)
//            + 4hh + (qq&3): the B operand of stage 2 is the lane's own registers.  MT1 > 1: the waves swap their tiles through
//            a per-lane LDS mailbox [MT1][4][64] x 16 bytes (conflict free, one barrier).
//   stage 2  wave w computes output m-tiles w, w + MT1, ... : 16 * MT1 MFMAs each, weights streamed from L2, then the usual
//            epilogue (bias, residual x, ELU'd store / twin).
// a1 / a2 are the ConvGemmArgs the two launches would get (a2.wpk replaced by the permuted packing).
struct ResBlockArgs {
    ConvGemmArgs a1, a2;
};

// P[mt][q][lane][e] = W[m][kperm], m = mt*32 + (lane&31), k-slot qq = q*4+e, hh = lane>>5, kperm as above (K = 1 convs only)
__global__ void k_pack_a_f32_hperm(const float* __restrict__ W, float* __restrict__ P, int M, int Kd, int Mt, int Q) {
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long total = (long)Mt * Q * 256;
    if (idx >= total) return;
    int e = (int)(idx & 3);
    int lane = (int)((idx >> 2) & 63);
    long rest = idx >> 8;
    int q = (int)(rest % Q);
    int mt = (int)(rest / Q);
    int m = mt * 32 + (lane & 31);
    int qq = q * 4 + e, hh = lane >> 5;
    int kd = 32 * (qq >> 4) + 8 * ((qq & 15) >> 2) + 4 * hh + (qq & 3);
    float v = 0.f;
    if (m < M && kd < Kd) v = W[(long)m * Kd + kd];
    P[idx] = v;
}

template <int MT1, int U, bool GROUP>
__global__ __launch_bounds__(MT1 * 64) void k_resblock(ResBlockArgs ra) {
    const ConvGemmArgs& a = ra.a1;
    const ConvGemmArgs& c = ra.a2;
    constexpr int NTH = MT1 * 64;
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int jl = lane & 31, kh = lane >> 5;
    // the tile's 32 columns belong to ONE session (T_out % 32 == 0, checked by the engine): b, t0 are uniform
    const int n0 = (int)blockIdx.x * 32;
    const int b = mmi_fast_div(n0, a.T_magic, GROUP ? a.T_shift : 0u), t0 = n0 - b * a.T_out;
    const int LD = 32 + a.K - 1;                 // input columns the tile's windows cover (stride 1)
    MMI_DYN_SHARED(float, smem);                 // Xs[Cin][LD] | offs[Q][2][4] | mailbox[MT1][4][64][4]
    float* Xs = smem;
    int* offs = reinterpret_cast<int*>(smem + ((a.Cin * LD + 3) & ~3));
    float* hs = reinterpret_cast<float*>(offs + a.Q * 8);

    // ---- stage 0: the input window -> LDS in ONE memory round trip: wave w stages channels w, w + MT1, ..., one row of LD
    // consecutive floats per load instruction (coalesced; Cin <= 64 * MT1), all requested before the first one is used
    constexpr int NR = 64;
    float xr[NR];
    {
        const float* xw = a.x + (long)b * a.x_bstride + a.x_off + t0;
        const int jj = lane < LD ? lane : LD - 1;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int ci = min(wave + i * MT1, a.Cin - 1);
            xr[i] = xw[(long)ci * a.x_ld + jj];
        }
    }
    // meanwhile: the weight fragments of this wave's first output tile, the hidden tile's bias, the first stage-1 fragments
    constexpr int Q2 = 4 * MT1;
    f32x4 w2v[Q2], w2n[Q2];
    {
        const f32x4* w2 = reinterpret_cast<const f32x4*>(c.wpk) + (long)min(wave, c.Mt - 1) * c.Q * 64 + lane;
#pragma unroll
        for (int q = 0; q < Q2; ++q) w2v[q] = w2[(long)min(q, c.Q - 1) * 64];
    }
    float b1v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = wave * 32 + 8 * (r >> 2) + 4 * kh + (r & 3);
        b1v[r] = a.bias ? a.bias[min(row, a.Cout - 1)] : 0.f;
        if (row >= a.Cout) b1v[r] = 0.f;
    }
    const f32x4* wp = reinterpret_cast<const f32x4*>(a.wpk) + (long)min(wave, a.Mt - 1) * a.Q * 64 + lane;
    const int q1 = a.Q;
    f32x4 avA[U], avB[U];
#define MMI_R_LOAD(AV, qb)                                                                          \
    _Pragma("unroll") for (int u = 0; u < U; ++u) AV[u] = wp[(long)min((qb) + u, q1 - 1) * 64];
    MMI_R_LOAD(avA, 0);
    // reduction index -> LDS offset of its window start: kd = (q*4+e)*2 + hh -> (ci, k) -> ci * LD + k; 0 past Cin*K (zero weights)
    for (int i = tid; i < a.Q * 8; i += NTH) {
        const int e = i & 3, hh = (i >> 2) & 1, q = i >> 3;
        const int kd = (q * 4 + e) * 2 + hh;
        const int ci = mmi_fast_div(kd, a.K_magic), k = kd - ci * a.K;
        offs[i] = kd < a.Cin * a.K ? ci * LD + k : 0;
    }
    if (lane < LD) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int ci = wave + i * MT1;
            if (ci < a.Cin) Xs[ci * LD + lane] = a.elu_in ? mmi_elu(xr[i]) : xr[i];
        }
    }
    __syncthreads();

    // ---- stage 1: hidden m-tile `wave` = W1[32 rows][Cin*K] . Xs windows; weights one group of U quads ahead, B operand from LDS
    f32x16 acc1;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc1[r] = 0.f;
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    const i32x4* ko = reinterpret_cast<const i32x4*>(offs) + kh;
    const float* xl = Xs + jl;
#define MMI_R_MMA(AV, qb)                                                                           \
    _Pragma("unroll") for (int u = 0; u < U; ++u) {                                                 \
        if ((qb) + u < q1) {                                                                        \
            const i32x4 o = ko[((qb) + u) * 2];                                                     \
            _Pragma("unroll") for (int e = 0; e < 4; ++e) acc1 = mmi_mfma_f32_32x32x2(AV[u][e], xl[o[e]], acc1); \
        }                                                                                           \
    }
    {
        const int G = (q1 + U - 1) / U;
        int g = 0;
        for (; g + 2 < G; g += 2) {
            MMI_R_LOAD(avB, (g + 1) * U);
            MMI_R_MMA(avA, g * U);
            MMI_R_LOAD(avA, (g + 2) * U);
            MMI_R_MMA(avB, (g + 1) * U);
        }
        if (G - g == 2) {
            MMI_R_LOAD(avB, (g + 1) * U);
            MMI_R_MMA(avA, g * U);
            MMI_R_MMA(avB, (g + 1) * U);
        } else {
            MMI_R_MMA(avA, g * U);
        }
    }
#undef MMI_R_LOAD
#undef MMI_R_MMA
    // ---- hand-off: h = ELU(acc1 + b1) in the accumulator layout (rows past Cout1 have zero weights on both sides)
    f32x4 hb[MT1][4];
    {
        float h[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) h[r] = mmi_elu(acc1[r] + b1v[r]);
        if constexpr (MT1 == 1) {
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4) hb[0][c4] = f32x4{h[4 * c4], h[4 * c4 + 1], h[4 * c4 + 2], h[4 * c4 + 3]};
        } else {
#pragma unroll
            for (int c4 = 0; c4 < 4; ++c4)
                *reinterpret_cast<f32x4*>(hs + ((wave * 4 + c4) * 64 + lane) * 4) = f32x4{h[4 * c4], h[4 * c4 + 1], h[4 * c4 + 2], h[4 * c4 + 3]};
            __syncthreads();
#pragma unroll
            for (int m = 0; m < MT1; ++m)
#pragma unroll
                for (int c4 = 0; c4 < 4; ++c4) hb[m][c4] = *reinterpret_cast<const f32x4*>(hs + ((m * 4 + c4) * 64 + lane) * 4);
        }
    }
    // ---- stage 2: output m-tiles wave, wave + MT1, ...; the epilogue is this block's own (bias, + x, ELU'd store and / or twin),
    // with none of the generic epilogue's per-value branches on launch-uniform flags: these kernels are instruction bound
    const int t = t0 + jl;
    const float* resb = c.res + (long)b * c.Cout * c.res_ld + c.res_off + t;
    float* outb = c.out + (long)b * c.Cout * c.out_ld + c.out_off + t;
    float* out2b = c.out2 ? c.out2 + (long)b * c.Cout * c.out_ld + c.out_off + t : nullptr;
    for (int mt2 = wave; mt2 < c.Mt; mt2 += MT1) {
        {   // the next tile's fragments are requested before this tile's MFMAs and epilogue
            const f32x4* w2 = reinterpret_cast<const f32x4*>(c.wpk) + (long)min(mt2 + MT1, c.Mt - 1) * c.Q * 64 + lane;
#pragma unroll
            for (int q = 0; q < Q2; ++q) w2n[q] = w2[(long)min(q, c.Q - 1) * 64];
        }
        // this tile's bias and residual values travel under the MFMAs (rows clamped into the tensor, masked at the store)
        const int row0 = mt2 * 32 + 4 * kh;
        float b2v[16], rv[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = min(row0 + (r & 3) + 8 * (r >> 2), c.Cout - 1);
            b2v[r] = c.bias ? c.bias[row] : 0.f;
            rv[r] = resb[(long)row * c.res_ld];
        }
        f32x16 acc2;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc2[r] = 0.f;
#pragma unroll
        for (int q = 0; q < Q2; ++q) {
            if (q < c.Q) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int qq = q * 4 + e;                 // k-slot: hidden tile qq / 16, accumulator register qq % 16
                    acc2 = mmi_mfma_f32_32x32x2(w2v[q][e], hb[qq >> 4][(qq & 15) >> 2][qq & 3], acc2);
                }
            }
        }
        {
            const bool full = mt2 * 32 + 32 <= c.Cout;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = row0 + (r & 3) + 8 * (r >> 2);
                if (!full && row >= c.Cout) continue;
                const float x = rv[r] + (acc2[r] + b2v[r]);             // x_orig + (conv + bias)  (seanet.py:76-77)
                const long at = (long)row * c.out_ld;
                if (out2b) { outb[at] = x; out2b[at] = mmi_elu(x); }
                else outb[at] = c.elu_out ? mmi_elu(x) : x;
            }
        }
#pragma unroll
        for (int q = 0; q < Q2; ++q) w2v[q] = w2n[q];
    }
}

// natural [B][Cin][x_ld] -> packed B operand: im2col (K, S), ELU, replicate padding of the first frame.
// One thread per (n-subtile, k-quad, lane): 4 elements kd = (q*4+e)*2 + (lane>>5), column n = nt*32 + (lane&31).
__global__ void k_pack_b_f32(ConvGemmArgs a, float* __restrict__ bp) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int ntn = (a.Ntot + 31) / 32;
    if (idx >= (long)ntn * a.Q * 64) return;
    const int lane = (int)(idx & 63);
    const int q = (int)((idx >> 6) % a.Q);
    const int nt = (int)((idx >> 6) / a.Q);
    const int n = nt * 32 + (lane & 31), kh = lane >> 5;
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    {   // columns past Ntot / reduction indices past Cin*K read a clamped (valid) element: they meet zero weights or are
        // discarded, and unconditional loads are not serialised by the compiler
        const int nc = n < a.Ntot ? n : 0;
        const int b = mmi_fast_div(nc, a.T_magic), t = nc - b * a.T_out;
        const float* xb = a.x + (long)b * a.x_bstride + a.x_off + t * a.S;
        const bool rep = a.first != nullptr && a.first[b] != 0 && a.exec[b] != 0;
        const int hist = a.H - a.x_off;  // columns (relative to x_off) that belong to the history
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int kd = (q * 4 + e) * 2 + kh;
            const int ci0 = mmi_fast_div(kd, a.K_magic), k = kd - ci0 * a.K;
            const int ci = ci0 < a.Cin ? ci0 : a.Cin - 1;
            int p = k;
            if (rep && (t * a.S + p) < hist) p = hist - t * a.S;  // replicate x[..., :1]
            float v = xb[(long)ci * a.x_ld + p];
            if (a.elu_in) v = mmi_elu(v);
            o[e] = v;
        }
    }
    reinterpret_cast<f32x4*>(bp)[idx] = o;
}

// split-K reduction over the workgroup's waves (fixed order) + the epilogue of k_gemm_f32
template <int NSUB, int WAVES>
__device__ __forceinline__ void mmi_gemm_f32_finish(const ConvGemmArgs& a, f32x16 (&acc)[NSUB], int mt, int s0, int wave, int lane) {
    constexpr int NE = NSUB * 16 * 64;
    MMI_SHARED float red[WAVES * NE];
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave * NE + (s * 16 + r) * 64 + lane] = acc[s][r];
    __syncthreads();
    constexpr int NV = NE / (WAVES * 64);
    int co[NV], nn[NV];
    float v[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int e = (int)threadIdx.x + i * WAVES * 64;
        const int le = e & 63, r = (e >> 6) & 15, s = e >> 10;
        nn[i] = (s0 + s) * 32 + (le & 31);
        co[i] = mt * 32 + (r & 3) + 8 * (r >> 2) + 4 * (le >> 5);
        float x = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) x += red[w * NE + e];
        v[i] = x;
    }
    if (a.out_mode == MMI_GOUT_PARTIAL) {
#pragma unroll
        for (int i = 0; i < NV; ++i) a.partial[((long)blockIdx.y * a.Mt * 32 + co[i]) * a.Npad + nn[i]] = v[i];   // padded rows / columns included
        return;
    }
    int bb[NV], tt[NV];
    bool ok[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        ok[i] = nn[i] < a.Ntot && co[i] < a.Cout;
        const int n3 = ok[i] ? nn[i] : 0;
        bb[i] = mmi_fast_div(n3, a.T_magic);
        tt[i] = n3 - bb[i] * a.T_out;
    }
    mmi_conv_store_n<NV>(a, co, bb, tt, ok, v);
}

// grid (Mt, ksplit, n-subtile groups); a workgroup covers NSUB n-subtiles of 32 columns starting at blockIdx.z*NSUB; its
// WAVES waves split the workgroup's k-quads.  The fp32 MFMA takes 64 cycles, so these GEMMs are matrix-core-latency
// bound unless they are spread over many waves: small weight matrices give each n-subtile its own workgroup.
template <int NSUB, int WAVES, int U>
__global__ __launch_bounds__(WAVES * 64) void k_gemm_f32(ConvGemmArgs a) {
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const int mt = blockIdx.x;
    const int qb_per = (a.Q + (int)gridDim.y - 1) / (int)gridDim.y;
    const int qb0 = min(a.Q, (int)blockIdx.y * qb_per), qb1 = min(a.Q, qb0 + qb_per);
    const int qper = (qb1 - qb0 + WAVES - 1) / WAVES;
    const int q0 = min(qb1, qb0 + wave * qper);
    const int nq = min(qb1, q0 + qper) - q0;
    const int ntn = (a.Ntot + 31) / 32;
    const int s0 = (int)blockIdx.z * NSUB;

    f32x16 acc[NSUB];
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[s][r] = 0.f;
    const f32x4* wp = reinterpret_cast<const f32x4*>(a.wpk) + ((long)mt * a.Q + q0) * 64 + lane;
    const f32x4* bp[NSUB];
#pragma unroll
    for (int s = 0; s < NSUB; ++s) bp[s] = reinterpret_cast<const f32x4*>(a.bp) + ((long)min(s0 + s, ntn - 1) * a.Q + q0) * 64 + lane;

    f32x4 wA[U], bA[U][NSUB], wB[U], bB[U][NSUB];
#define MMI_F_LOAD(W_, B_, base)                                                              \
    _Pragma("unroll") for (int u = 0; u < U; ++u) {                                           \
        W_[u] = mmi_load_nt(wp + ((base) + u) * 64);                                          \
        _Pragma("unroll") for (int s = 0; s < NSUB; ++s) B_[u][s] = bp[s][((base) + u) * 64]; \
    }
#define MMI_F_MMA(W_, B_)                                                                     \
    _Pragma("unroll") for (int u = 0; u < U; ++u)                                             \
        _Pragma("unroll") for (int e = 0; e < 4; ++e)                                         \
            _Pragma("unroll") for (int s = 0; s < NSUB; ++s) acc[s] = mmi_mfma_f32_32x32x2(W_[u][e], B_[u][s][e], acc[s]);
    const int nfull = nq / U;
    if (nfull > 0) {
        MMI_F_LOAD(wA, bA, 0);
        int g = 0;
        for (; g + 2 < nfull; g += 2) {
            MMI_F_LOAD(wB, bB, (g + 1) * U);
            MMI_F_MMA(wA, bA);
            MMI_F_LOAD(wA, bA, (g + 2) * U);
            MMI_F_MMA(wB, bB);
        }
        if (nfull - g == 2) {
            MMI_F_LOAD(wB, bB, (g + 1) * U);
            MMI_F_MMA(wA, bA);
            MMI_F_MMA(wB, bB);
        } else {
            MMI_F_MMA(wA, bA);
        }
    }
    for (int q = nfull * U; q < nq; ++q) {
        wA[0] = mmi_load_nt(wp + q * 64);
#pragma unroll
        for (int s = 0; s < NSUB; ++s) bA[0][s] = bp[s][q * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int s = 0; s < NSUB; ++s) acc[s] = mmi_mfma_f32_32x32x2(wA[0][e], bA[0][s][e], acc[s]);
    }
#undef MMI_F_LOAD
#undef MMI_F_MMA

    mmi_gemm_f32_finish<NSUB, WAVES>(a, acc, mt, s0, wave, lane);
}

// A conv of few columns on v_mfma_f32_16x16x4_f32: grid (ceil(Cout/16), ceil(Ntot/16), ks), one 16 x 16 tile per workgroup.  The reduction is cut as
// k_gemm_f32 cuts it - into gridDim.z pieces of a.q_blk quads, each of them over the workgroup's waves - and added up in the same order, so the
// results are the same bits (k_conv_finish adds the gridDim.z sums).  Operands come from the conv's input as it lies (PACKED: from `bp`).
// Weights and `bp` hold quads of 8 reduction indices for 32 rows: the lanes of the upper half take the next quad, an exchange of register halves
// (mmi_swap32) turns two quads into the four operands of the 16 x 16 form, in rising order.
// Bound by latency, like k_mimi_lin: the launch that packed the input (4.5 us) is gone, 32 x 32 tiles left 8 - 32 CUs at work.  One stream:
// 256 -> 128, K 3 on 96 columns 4.4 + 6.8 -> 5.6 us; 512 -> 256, K 3 on 16 columns 4.5 + 10.7 -> 7.6; 512 -> 1024, K 16 on 2 columns
// 4.6 + 11.3 -> 13.1.  All pieces of a split reduction in one workgroup, without the launch that adds them, measured slower (1024 -> 512, K 3 on
// 2 columns: 12.0 against 4.9 + 4.8 - one CU streams 20 - 50 KB of weights per us).
template <bool PACKED, bool FIRST>
__global__ __launch_bounds__(512) void k_conv_few(ConvGemmArgs a) {
    constexpr int U = 5;                                     // pairs of quads per group; two groups are in flight
    MMI_SHARED float red[8 * 256];
    const int tid = (int)threadIdx.x, wave = mmi_uniform(tid >> 6), lane = tid & 63, nw = (int)blockDim.x >> 6;
    const int r16 = lane & 15, quarter = lane >> 4, kh = quarter & 1, hi = quarter >> 1;
    const int m0 = (int)blockIdx.x * 16, n0 = (int)blockIdx.y * 16;

    // what this thread stores: element tid of the tile in the accumulators' order
    int co[1] = {m0 + 4 * ((tid >> 4) & 3) + ((tid >> 6) & 3)}, bb[1], tt[1];
    const int no = n0 + (tid & 15);
    bool ok[1] = {tid < 256 && no < a.Ntot && co[0] < a.Cout};
    bb[0] = mmi_fast_div(ok[0] ? no : 0, a.T_magic);
    tt[0] = (ok[0] ? no : 0) - bb[0] * a.T_out;
    long row[1];
    float bia[1], rsv[1];
    mmi_conv_ask_n<1>(a, co, bb, tt, ok, row, bia, rsv);

    const int qb0 = min(a.Q, (int)blockIdx.z * a.q_blk), qb1 = min(a.Q, qb0 + a.q_blk), qper = (qb1 - qb0 + nw - 1) / nw;
    const int qa = min(qb1, qb0 + wave * qper), qz = min(qb1, qa + qper), last = max(qz - 1, 0);
    const f32x4* wp = reinterpret_cast<const f32x4*>(a.wpk) + (long)(m0 >> 5) * a.Q * 64 + kh * 32 + (m0 & 16) + r16;
    const f32x4* bp = nullptr;
    // the input's places of the four values of a pair of quads (bytes from a.x on), and their taps: 16 indices further is a few additions
    unsigned off[4], top = 0, step = 0, carry = 0;
    int tap[4], tap_step = 0, tap_min = 0;
    if constexpr (PACKED) {
        const int ntn = (a.Ntot + 31) / 32;
        bp = reinterpret_cast<const f32x4*>(a.bp) + (long)min(n0 >> 5, ntn - 1) * a.Q * 64 + kh * 32 + (n0 & 16) + r16;
    } else {
        const int nc = n0 + r16 < a.Ntot ? n0 + r16 : 0;     // (columns past the last one are computed and dropped)
        const int b = mmi_fast_div(nc, a.T_magic), t = nc - b * a.T_out;
        const unsigned base = 4u * (unsigned)(b * (int)a.x_bstride + a.x_off + t * a.S);
        if (FIRST && a.first[b] != 0 && a.exec[b] != 0) tap_min = a.H - a.x_off - t * a.S;      // replicate x[..., :1]
        const int c16 = mmi_fast_div(16, a.K_magic);
        tap_step = 16 - c16 * a.K;
        step = 4u * (unsigned)(c16 * a.x_ld + tap_step);
        carry = 4u * (unsigned)(a.x_ld - a.K);
        top = base + 4u * (unsigned)((a.Cin - 1) * a.x_ld + a.K - 1);        // (reduction indices past the last one meet zero weights or no product)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int kd = (qa + (e >> 1)) * 8 + 4 * (e & 1) + quarter, ci = mmi_fast_div(kd, a.K_magic);
            tap[e] = kd - ci * a.K;
            off[e] = base + 4u * (unsigned)(ci * a.x_ld + tap[e]);
        }
    }
    auto load = [&](f32x4 (&w)[U], f32x4 (&x)[U], int q) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            w[u] = mmi_load_nt(wp + (long)min(q + 2 * u + hi, last) * 64);
            if constexpr (PACKED) x[u] = bp[(long)min(q + 2 * u + hi, last) * 64];
            else
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    unsigned o = off[e];
                    if (FIRST) o += 4u * (unsigned)max(tap_min - tap[e], 0);
                    x[u][e] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.x) + min(o, top));
                    tap[e] += tap_step;
                    off[e] += step;
                    const bool over = tap[e] >= a.K;
                    tap[e] -= over ? a.K : 0;
                    off[e] += over ? carry : 0u;
                }
        }
    };
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto quads = [](f32x4& v) __attribute__((always_inline)) {     // element e of quads (q, q + 1) -> steps 0, 1 of q, steps 0, 1 of q + 1
        float e0 = v[0], e1 = v[1], e2 = v[2], e3 = v[3];
        mmi_swap32(e0, e1);
        mmi_swap32(e2, e3);
        v = f32x4{e0, e2, e1, e3};
    };
    auto mma = [&](f32x4 (&w)[U], f32x4 (&x)[U], int q) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            quads(w[u]);
            if constexpr (PACKED) quads(x[u]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (q + 2 * u + (e >> 1) < qz) acc = mmi_mfma_f32_16x16x4(w[u][e], x[u][e], acc);
        }
    };
    if (qa < qz) {
        f32x4 wA[U], xA[U], wB[U], xB[U];
        load(wA, xA, qa);
        for (int q = qa; q < qz; q += 4 * U) {
            if (q + 2 * U < qz) load(wB, xB, q + 2 * U);
            mma(wA, xA, q);
            if (q + 4 * U < qz) load(wA, xA, q + 4 * U);
            if (q + 2 * U < qz) mma(wB, xB, q + 2 * U);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave * 256 + r * 64 + lane] = acc[r];
    __syncthreads();
    if (tid >= 256) return;
    float v[1] = {0.f};
    for (int w = 0; w < nw; ++w) v[0] += red[w * 256 + tid];
    if (a.out_mode == MMI_GOUT_PARTIAL) a.partial[((long)blockIdx.z * a.Mt * 32 + co[0]) * a.Npad + no] = v[0];       // padded rows / columns included
    else mmi_conv_put_n<1>(a, co, bb, tt, ok, row, bia, rsv, v);
}

// ------------------------------------------------------------------------------------------------
// linears of the Mimi transformers
// ------------------------------------------------------------------------------------------------
// W[m][k] (m < M, k < K) -> P[ceil(M/16)][J][lane][e], element (row, k) where mmi_lin_index has (k, column); zero padded
__global__ void k_pack_lin(const float* __restrict__ W, float* __restrict__ P, int M, int K, int Mt, int J) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)Mt * J * 256) return;
    const int e = (int)(idx & 3), lane = (int)((idx >> 2) & 63);
    const long f = idx >> 8;
    const int j = (int)(f % J), m = (int)(f / J) * 16 + (lane & 15), k = 16 * j + 4 * e + (lane >> 4);
    P[idx] = m < M && k < K ? W[(long)m * K + k] : 0.f;
}
// LayerNorm weight / bias [C] in the operand's element order: out[(j * 4 + quarter) * 4 + e] = v[16 j + 4 e + quarter]; C % 16 == 0
__global__ void k_pack_ln(const float* __restrict__ v, float* __restrict__ out, int C) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < C) out[i] = v[16 * (i >> 4) + 4 * (i & 3) + ((i >> 2) & 3)];
}

enum { MIMI_LIN_ROWS = 0, MIMI_LIN_GELU = 1, MIMI_LIN_RESID = 2 };
struct MimiLinArgs {
    const float* w;              // [Mt][J] fragments (k_pack_lin)
    const float* x;              // [ceil(N/16)][J] fragments (mmi_lin_index)
    int M, N, J;                 // rows, columns n = b * T + t, 16-deep pieces of the reduction
    int share;                   // k_mimi_lin, FM = 1: 2^share workgroups share a row tile
    const float *ln_w, *ln_b;    // LayerNorm over the 16 J values of a column in front (k_pack_ln)
    float ln_eps;
    int mode;                    // ROWS: out = W x;  GELU: outp = gelu(W x);  RESID: outp += scale * W x (the residual stream), and out too where it is set
    float* outp;
    int outJ;
    const float* scale;
    float* out;                  // [B][M][out_ld] from column out_off on
    int out_ld, out_off, T;
    unsigned T_magic, T_shift;
};

// out[m][n] = sum_k W[m][k] x[k][n] on v_mfma_f32_16x16x4_f32 (an exact fma chain), LayerNorm of the columns in front where LN.
// grid (ceil(Mt/FM), ceil(N/(16 FN))); a workgroup owns 16 FM rows x 16 FN columns; its 8 waves cut the reduction into 8 pieces, their sums are
// added in rising order.  What a workgroup covers changes no bit (a piece and its order are the reduction's alone), so one stream, many
// streams and groups of frames agree.
// Measured, 1 stream (N = 2): norm + linear 8.2 -> 5.0 us, K = 512 5.9 -> 4.7, K = 2048 9.3 (with a second launch that added its sums) -> 6.6; 32 streams
// (N = 64): norm + linear 8.4 -> 6.3, K = 2048 9.6 -> 6.9; a file's 258 columns: K = 512 7.9 -> 6.2, K = 2048 19.2 -> 13.0 (norm + linear: k_mimi_lin_rows).
// Fragments pass in a ring that asks for none past the slice, 8 of them for long reductions (a double buffer of 4 asked for 4 twice): one stream 690.9 -> 680.9
// us a frame, 32 streams 1178 -> 1169.
// Bound by latency: one column tile has M / 16 workgroups of 16 KB - 64 KB of weights and a few hundred cycles of matrix work each.  Hence
// 16-wide tiles (a live stream has two columns: a 32-wide tile keeps the matrix core busy four times as long, 1.7 us at K = 512, on half the
// CUs), every operand of the epilogue requested ahead of the sums, the norm's whole slice in registers (U fragments per wave), and
// no reduction split over workgroups (K = 2048 needed a second launch to add the sums).
template <int FM, int FN, int U, bool LN, bool NT>
__global__ __launch_bounds__(512) void k_mimi_lin(MimiLinArgs a) {
    auto weight = [](const f32x4* p) __attribute__((always_inline)) { return NT ? mmi_load_nt(p) : *p; };
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63;
    // a row tile shared by 2^share workgroups: 16 >> share rows each; lanes of the others' rows repeat its own (their sums are dropped)
    const int share = FM == 1 ? a.share : 0, mine = 16 >> share, r0 = ((int)blockIdx.x & ((1 << share) - 1)) * mine;
    const int m0 = ((int)blockIdx.x >> share) * FM, n0 = (int)blockIdx.y * FN, wl = (lane & 48) + r0 + (lane & (mine - 1));
    const int Mt = (a.M + 15) >> 4, Nt = (a.N + 15) >> 4;
    const int per = (a.J + 7) >> 3;                          // LN: <= U (the planner checks)
    const int j0 = min(a.J, wave * per), nj = min(a.J, j0 + per) - j0;
    const int jl = min(j0, a.J - 1), last = nj > 0 ? nj - 1 : 0;
    const f32x4* wp[FM];
    const f32x4* xp[FN];
#pragma unroll
    for (int m = 0; m < FM; ++m) wp[m] = reinterpret_cast<const f32x4*>(a.w) + ((long)min(m0 + m, Mt - 1) * a.J + jl) * 64 + wl;
#pragma unroll
    for (int n = 0; n < FN; ++n)                             // (a column past the last one reads the last one: nobody need have stored it)
        xp[n] = reinterpret_cast<const f32x4*>(a.x) + ((long)min(n0 + n, Nt - 1) * a.J + jl) * 64 + (lane & 48) + min(lane & 15, max(a.N - (n0 + n) * 16, 1) - 1);

    f32x4 acc[FM][FN];
#pragma unroll
    for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

    // results of this thread: element idx & 255 of tile idx >> 8, idx = tid + 512 i.  In operand order (GELU, RESID) that is the tile's place in
    // outp; in the accumulators' order (ROWS) 16 columns of a row lie side by side.
    constexpr int NV = (FM * FN + 1) / 2;
    int rm[NV], rn[NV];
    float scl[NV], res[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int idx = tid + 512 * i, f = idx >> 8, q = idx & 255;
        const int row = a.mode == MIMI_LIN_ROWS ? 4 * ((q >> 4) & 3) + (q >> 6) : 4 * (q & 3) + (q >> 6);
        rm[i] = (m0 + f / FN) * 16 + row;
        rn[i] = (n0 + f % FN) * 16 + (a.mode == MIMI_LIN_ROWS ? q & 15 : (q >> 2) & 15);
        if (idx >= FM * FN * 256 || rm[i] >= a.M || (unsigned)(row - r0) >= (unsigned)mine) rn[i] = a.N;          // nothing to store
        scl[i] = 0.f; res[i] = 0.f;
    }
    if (a.mode == MIMI_LIN_RESID) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const bool ok = rn[i] < a.N;
            scl[i] = a.scale[ok ? rm[i] : 0];
            res[i] = a.outp[ok ? mmi_lin_index(rm[i], rn[i], a.outJ) : 0];
        }
    }

    if constexpr (LN) {
        MMI_SHARED float stat[2][8][FN * 16];
        const f32x4* gp = reinterpret_cast<const f32x4*>(a.ln_w) + (long)jl * 4 + (lane >> 4);
        const f32x4* hp = reinterpret_cast<const f32x4*>(a.ln_b) + (long)jl * 4 + (lane >> 4);
        f32x4 wv[U][FM], xv[U][FN], gv[U], bv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {                        // unconditional loads from clamped (valid) places, masked afterwards
            const int uu = min(u, last);
#pragma unroll
            for (int n = 0; n < FN; ++n) xv[u][n] = xp[n][uu * 64];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int uu = min(u, last);
#pragma unroll
            for (int m = 0; m < FM; ++m) wv[u][m] = weight(wp[m] + uu * 64);
            gv[u] = gp[uu * 4];
            bv[u] = hp[uu * 4];
        }
        auto column_sum = [&](int which, float (&s)[FN]) __attribute__((always_inline)) {      // over the lanes that hold a column, then over the waves
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                s[n] = mmi_rows_sum(s[n]);
                if (lane < 16) stat[which][wave][n * 16 + lane] = s[n];
            }
            __syncthreads();
#pragma unroll
            for (int n = 0; n < FN; ++n) {
                float t = 0.f;
#pragma unroll
                for (int w = 0; w < 8; ++w) t += stat[which][w][n * 16 + (lane & 15)];
                s[n] = t;
            }
        };
        float mean[FN], rstd[FN];
#pragma unroll
        for (int n = 0; n < FN; ++n) mean[n] = rstd[n] = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < nj)
#pragma unroll
                for (int n = 0; n < FN; ++n) mean[n] += (xv[u][n][0] + xv[u][n][1]) + (xv[u][n][2] + xv[u][n][3]);
        column_sum(0, mean);
#pragma unroll
        for (int n = 0; n < FN; ++n) mean[n] /= (float)(a.J * 16);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < nj)
#pragma unroll
                for (int n = 0; n < FN; ++n)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float d = xv[u][n][e] - mean[n];
                        rstd[n] += d * d;
                    }
        column_sum(1, rstd);
#pragma unroll
        for (int n = 0; n < FN; ++n) rstd[n] = mmi_rsqrtf(rstd[n] / (float)(a.J * 16) + a.ln_eps);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < nj)
#pragma unroll
                for (int n = 0; n < FN; ++n)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float y = (xv[u][n][e] - mean[n]) * rstd[n] * gv[u][e] + bv[u][e];
#pragma unroll
                        for (int m = 0; m < FM; ++m) acc[m][n] = mmi_mfma_f32_16x16x4(wv[u][m][e], y, acc[m][n]);
                    }
    } else {
        // U fragments of weights and operand on their way in a ring: each is asked for again as soon as its products are done, none past the slice
        f32x4 w[U][FM], x[U][FN];
        auto load = [&](int u, int at) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < FM; ++m) w[u][m] = weight(wp[m] + (long)at * 64);
#pragma unroll
            for (int n = 0; n < FN; ++n) x[u][n] = xp[n][(long)at * 64];
        };
        auto mma = [&](int u, bool on) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < FN; ++n) {
                    const float v = on ? x[u][n][e] : 0.f;       // (past the slice: zeros, not a branch - see k_conv_cols)
#pragma unroll
                    for (int m = 0; m < FM; ++m) acc[m][n] = mmi_mfma_f32_16x16x4(w[u][m][e], v, acc[m][n]);
                }
        };
#pragma unroll
        for (int u = 0; u < U; ++u) load(u, min(u, last));
        mmi_sched_barrier();
        int at = 0;
#pragma unroll 1
        for (; at + U < nj; at += U)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                mma(u, true);
                load(u, min(at + U + u, last));
                mmi_sched_barrier();
            }
#pragma unroll
        for (int u = 0; u < U; ++u) mma(u, at + u < nj);
    }

    MMI_SHARED float red[8 * FM * FN * 256];
#pragma unroll
    for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((wave * FM + m) * FN + n) * 256 + r * 64 + lane] = acc[m][n][r];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int idx = tid + 512 * i, q = idx & 255;
        if (rn[i] >= a.N) continue;
        const int at = (idx & ~255) + (a.mode == MIMI_LIN_ROWS ? q : (q >> 6) * 64 + (q & 3) * 16 + ((q >> 2) & 15));
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) v += red[w * FM * FN * 256 + at];
        if (a.mode == MIMI_LIN_GELU) v = mmi_gelu_erf(v);
        if (a.mode == MIMI_LIN_RESID) v = res[i] + scl[i] * v;
        if (a.mode != MIMI_LIN_ROWS) a.outp[mmi_lin_index(rm[i], rn[i], a.outJ)] = v;
        if (a.out) {
            const int b = mmi_fast_div(rn[i], a.T_magic, a.T_shift), t = rn[i] - b * a.T;
            a.out[((long)b * a.M + rm[i]) * a.out_ld + a.out_off + t] = v;
        }
    }
}

// norm + linear of many columns: a workgroup of 8 to 12 waves owns 16 rows per wave x 16 columns, grid (row tiles / waves, ceil(N/16)).  Wave w < 8
// normalises piece w of the reduction, as k_mimi_lin's does, and leaves it in LDS; then a wave takes the eight pieces one after the other, each from zero, added in
// rising order: k_mimi_lin's bits.  With 16 rows per workgroup every column was normalised by 96 - 128 of them - 570 vector instructions around 32
// products per wave: a file's 258 columns 512 -> 1536 15.5 -> 11.5 us, 512 -> 2048 20.1 -> 15.6.  J <= 60.
template <int KJ>
__global__ __launch_bounds__(768) void k_mimi_lin_rows(MimiLinArgs a) {
    constexpr int U = 8;
    MMI_DYN_SHARED(f32x4, y);                                // [J][64]
    MMI_SHARED float stat[2][8][16];
    const int tid = (int)threadIdx.x, wave = mmi_uniform(tid >> 6), lane = tid & 63;
    const int rt = (int)blockIdx.x * ((int)blockDim.x >> 6) + wave, n0 = (int)blockIdx.y * 16, Mt = (a.M + 15) >> 4;
    const int per = (a.J + 7) >> 3, j0 = min(a.J, wave * per), nj = min(a.J, j0 + per) - j0;      // <= KJ (the planner checks)
    const int jl = min(j0, a.J - 1), last = nj > 0 ? nj - 1 : 0;
    const f32x4* xp = reinterpret_cast<const f32x4*>(a.x) + ((long)blockIdx.y * a.J + jl) * 64 + (lane & 48) + min(lane & 15, a.N - n0 - 1);
    const f32x4* gp = reinterpret_cast<const f32x4*>(a.ln_w) + (long)jl * 4 + (lane >> 4);
    const f32x4* hp = reinterpret_cast<const f32x4*>(a.ln_b) + (long)jl * 4 + (lane >> 4);
    const f32x4* wp = reinterpret_cast<const f32x4*>(a.w) + (long)min(rt, Mt - 1) * a.J * 64 + lane;
    f32x4 xv[KJ], gv[KJ], bv[KJ], wA[U], wB[U];
    auto load = [&](f32x4 (&w)[U], int j) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = wp[(long)min(j + u, a.J - 1) * 64];
    };
#pragma unroll
    for (int u = 0; u < KJ; ++u) xv[u] = xp[min(u, last) * 64];
#pragma unroll
    for (int u = 0; u < KJ; ++u) { gv[u] = gp[min(u, last) * 4]; bv[u] = hp[min(u, last) * 4]; }
    load(wA, 0);
    mmi_sched_barrier();
    auto column_sum = [&](int which, float s) __attribute__((always_inline)) {
        s += mmi_shfl_xor(s, 16);
        s += mmi_shfl_xor(s, 32);
        if (lane < 16 && wave < 8) stat[which][wave][lane] = s;
        __syncthreads();
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) t += stat[which][w][lane & 15];
        return t;
    };
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < KJ; ++u)
        if (u < nj) s += (xv[u][0] + xv[u][1]) + (xv[u][2] + xv[u][3]);
    const float mean = column_sum(0, s) / (float)(a.J * 16);
    s = 0.f;
#pragma unroll
    for (int u = 0; u < KJ; ++u)
        if (u < nj)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = xv[u][e] - mean;
                s += d * d;
            }
    const float rstd = mmi_rsqrtf(column_sum(1, s) / (float)(a.J * 16) + a.ln_eps);
#pragma unroll
    for (int u = 0; u < KJ; ++u)
        if (u < nj) {
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (xv[u][e] - mean) * rstd * gv[u][e] + bv[u][e];
            y[(j0 + u) * 64 + lane] = v;
        }
    __syncthreads();
    if (rt >= Mt) return;

    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, sum = acc;
    int end = per;
    auto mma = [&](f32x4 (&w)[U], int j) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (j + u == end) { sum += acc; acc = f32x4{0.f, 0.f, 0.f, 0.f}; end += per; }
            f32x4 v = y[min(j + u, a.J - 1) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = mmi_mfma_f32_16x16x4(w[u][e], j + u < a.J ? v[e] : 0.f, acc);
        }
    };
    int j = 0;
    while (j + U < a.J) {                                    // pairs of groups, one way out (k_conv_cols)
        load(wB, j + U);
        mmi_sched_barrier();
        mma(wA, j);
        load(wA, j + 2 * U);
        mmi_sched_barrier();
        mma(wB, j + U);
        j += 2 * U;
    }
    if (j < a.J) mma(wA, j);
    sum += acc;
    const int n = n0 + (lane & 15);
    if (n >= a.N) return;
    const int b = mmi_fast_div(n, a.T_magic, a.T_shift), t = n - b * a.T;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = rt * 16 + 4 * (lane >> 4) + r;
        if (m >= a.M) continue;
        if (a.mode == MIMI_LIN_GELU) a.outp[mmi_lin_index(m, n, a.outJ)] = mmi_gelu_erf(sum[r]);
        else a.out[((long)b * a.M + m) * a.out_ld + a.out_off + t] = sum[r];
    }
}

// sum of the split-K partials + epilogue -> [B][Cout][out_ld]
__global__ void k_conv_finish(ConvGemmArgs a, int ksplit) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)a.Cout * a.Ntot) return;
    const int n = (int)(idx % a.Ntot), co = (int)(idx / a.Ntot);
    float pv[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) pv[s] = a.partial[((long)min(s, ksplit - 1) * a.Mt * 32 + co) * a.Npad + n];   // ksplit <= 8, all in flight
    float x = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) x += s < ksplit ? pv[s] : 0.f;
    const int bq = mmi_fast_div(n, a.T_magic, a.T_shift);
    int co1[1] = {co}, b1[1] = {bq}, t1[1] = {n - bq * a.T_out};
    bool ok1[1] = {true};
    float v1[1] = {x};
    mmi_conv_store_n<1>(a, co1, b1, t1, ok1, v1);
}

// ------------------------------------------------------------------------------------------------
// transposed conv: overlap-add of the GEMM result with the streaming `partial` (conv.py:340-362)
// tmp [B][Cout*K][tmp_ld >= T_in] holds tmp[b][co*K + k][t] = sum_ci Wtr[ci][co][k] * elu(x[b][ci][t]); K == 2*S.
// ------------------------------------------------------------------------------------------------
// out2: the ELU'd twin of `out` (same geometry) read by the next conv, or null (see ConvGemmArgs::out2)
__global__ void k_convtr_combine(const float* __restrict__ tmp, const float* __restrict__ bias,
                                 float* __restrict__ partial, const uint8_t* __restrict__ exec, float* __restrict__ out,
                                 int out_ld, int out_off, int B, int Cout, int K, int S, int T_in, float* __restrict__ out2,
                                 int tmp_ld, int T_frame) {
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int Tout = T_in * S;
    if (idx >= (long)B * Cout * Tout) return;
    int p = (int)(idx % Tout);
    long row = idx / Tout;  // b*Cout + co
    int co = (int)(row % Cout);
    int b = (int)(row / Cout);
    int t = p / S, r = p - t * S;
    const float* trow = tmp + row * (long)K * tmp_ld;  // [K][T_in], row stride tmp_ld
    float v = trow[(long)r * tmp_ld + t];
    if (T_frame == T_in) {
        if (t > 0) v += trow[(long)(r + S) * tmp_ld + (t - 1)];
        if (bias) v += bias[co];
    } else {                                      // what a frame takes over from the one before it is added last, as when it is kept as `partial`
        const bool inside = t % T_frame != 0;
        const float before = t > 0 ? trow[(long)(r + S) * tmp_ld + (t - 1)] : 0.f;
        if (inside) v += before;
        if (bias) v += bias[co];
        if (!inside && t > 0) v += before;
    }
    if (t == 0) {
        // y[..., :PT] += partial; then the thread that consumed partial[b][co][r] also refreshes it
        long pi = row * (long)(K - S) + r;
        v += partial[pi];
        if (exec[b]) partial[pi] = trow[(long)(r + S) * tmp_ld + (T_in - 1)];  // tail, bias excluded (conv.py:354-360)
    }
    out[row * (long)out_ld + out_off + p] = v;
    if (out2) out2[row * (long)out_ld + out_off + p] = mmi_elu(v);
}

// depthwise (groups == C) transposed conv, K == 2*S, no bias: ConvTrUpsample1d (resample.py:68-119)
__global__ void k_upsample_dw(const float* __restrict__ x, int x_ld, int x_off, const float* __restrict__ w,
                              float* __restrict__ partial, const uint8_t* __restrict__ exec, float* __restrict__ out,
                              int out_ld, int out_off, int B, int C, int K, int S, int T_in, float* __restrict__ outp, int outJ) {
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int Tout = T_in * S;
    if (idx >= (long)B * C * Tout) return;
    int p = (int)(idx % Tout);
    long row = idx / Tout;
    int c = (int)(row % C);
    int b = (int)(row / C);
    int t = p / S, r = p - t * S;
    const float* xr = x + row * (long)x_ld + x_off;
    float v = w[c * K + r] * xr[t];
    if (t > 0) v += w[c * K + r + S] * xr[t - 1];
    if (t == 0) {
        long pi = row * (long)(K - S) + r;
        v += partial[pi];
        if (exec[b]) partial[pi] = w[c * K + r + S] * xr[T_in - 1];
    }
    out[row * (long)out_ld + out_off + p] = v;
    outp[mmi_lin_index(c, b * Tout + p, outJ)] = v;        // the transformer's residual stream
}

// ------------------------------------------------------------------------------------------------
// end-of-frame state commit: history shift, transformer offsets, replicate flags
// ------------------------------------------------------------------------------------------------
struct HistDesc {
    float* p;       // buffer [B][C][ld]
    int C, ld, H, T;
    int row_begin;  // prefix of B*C rows over the descriptor table
};

__global__ void k_commit_history(const HistDesc* __restrict__ descs, int ndesc, int total_rows,
                                 const uint8_t* __restrict__ exec) {
    int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid >= total_rows) return;
    int d = 0;
    while (d + 1 < ndesc && descs[d + 1].row_begin <= gid) ++d;
    HistDesc h = descs[d];
    int row = gid - h.row_begin;
    int b = row / h.C;
    if (!exec[b]) return;
    float* r = h.p + (long)row * h.ld;
    for (int p = 0; p < h.H; ++p) r[p] = r[p + h.T];  // ascending: source p+T is always ahead of the write
}

// Both commits of a step in ONE launch, with the descriptor table passed by value (kernel arguments: scalar loads) instead of
// searched through global memory by every thread: threads [0, total_rows) shift the histories, the next B advance the counters.
#define MMI_HIST_MAX 16
struct HistTable {
    HistDesc d[MMI_HIST_MAX];
    int n;
};
__global__ void k_commit_all(HistTable tab, int total_rows, const uint8_t* __restrict__ exec, long* __restrict__ counters,
                             int n_counters, int inc, uint8_t* __restrict__ first, int B) {
    int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid >= total_rows) {
        gid -= total_rows;
        if (gid >= B || !exec[gid]) return;
        for (int i = 0; i < n_counters; ++i) counters[(long)i * B + gid] += inc;
        if (first) first[gid] = 0;
        return;
    }
    int d = 0;
#pragma unroll
    for (int i = 1; i < MMI_HIST_MAX; ++i)
        if (i < tab.n && tab.d[i].row_begin <= gid) d = i;
    const HistDesc h = tab.d[d];
    int row = gid - h.row_begin;
    int b = row / h.C;
    if (!exec[b]) return;
    // eight at a time, all of them read before one is written (source p + T is always ahead of the write; one by one each waited for the last: 6.0 us for
    // a stream, here 5.3)
    float* r = h.p + (long)row * h.ld;
    for (int p0 = 0; p0 < h.H; p0 += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = r[min(p0 + i, h.H - 1) + h.T];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (p0 + i < h.H) r[p0 + i] = v[i];
    }
}

// the histories of one set of buffers -> the same ones of another
__global__ void k_move_history(HistTable from, HistTable to, int total_rows) {
    const int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid >= total_rows) return;
    int d = 0;
#pragma unroll
    for (int i = 1; i < MMI_HIST_MAX; ++i)
        if (i < from.n && from.d[i].row_begin <= gid) d = i;
    const HistDesc f = from.d[d], t = to.d[d];
    const long row = gid - f.row_begin;
    for (int p0 = 0; p0 < f.H; p0 += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = f.p[row * f.ld + min(p0 + i, f.H - 1)];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (p0 + i < f.H) t.p[row * t.ld + p0 + i] = v[i];
    }
}

// offsets[i][b] += inc where exec; first[b] = 0 where exec
__global__ void k_commit_counters(long* __restrict__ counters, int n_counters, int inc, uint8_t* __restrict__ first,
                                  const uint8_t* __restrict__ exec, int B) {
    int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid >= B) return;
    if (!exec[gid]) return;
    for (int i = 0; i < n_counters; ++i) counters[(long)i * B + gid] += inc;
    if (first) first[gid] = 0;
}

__global__ void k_reset_history(const HistDesc* __restrict__ descs, int ndesc, int total_rows,
                                const uint8_t* __restrict__ mask) {
    int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid >= total_rows) return;
    int d = 0;
    while (d + 1 < ndesc && descs[d + 1].row_begin <= gid) ++d;
    HistDesc h = descs[d];
    int row = gid - h.row_begin;
    int b = row / h.C;
    if (mask && !mask[b]) return;
    float* r = h.p + (long)row * h.ld;
    for (int p = 0; p < h.H; ++p) r[p] = 0.f;
}

// A reset in one launch: the histories of both directions, the overlap-adds' partial rows, then a stream's offsets and flags, where mask
// (null: everywhere)
#define MMI_PARTIALS_MAX 12
struct ResetTable {
    HistTable hist[2];
    int rows[2];
    float* part[MMI_PARTIALS_MAX];
    long part_end[MMI_PARTIALS_MAX], part_row[MMI_PARTIALS_MAX];      // running ends in elements, elements per stream
    int n_part, B;
    long* counters; uint8_t *first, *exec;
};
__global__ void k_reset_all(ResetTable t, const uint8_t* __restrict__ mask) {
    long at = (long)blockIdx.x * blockDim.x + threadIdx.x;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        if (at >= 0 && at < t.rows[side]) {
            int d = 0;
#pragma unroll
            for (int i = 1; i < MMI_HIST_MAX; ++i)
                if (i < t.hist[side].n && t.hist[side].d[i].row_begin <= at) d = i;
            const HistDesc h = t.hist[side].d[d];
            const int row = (int)at - h.row_begin;
            if (mask && !mask[row / h.C]) return;
            for (int p = 0; p < h.H; ++p) h.p[(long)row * h.ld + p] = 0.f;
            return;
        }
        at -= t.rows[side];
    }
    long begin = 0;
    for (int i = 0; i < t.n_part; ++i) {
        if (at >= begin && at < t.part_end[i]) {
            if (!mask || mask[(at - begin) / t.part_row[i]]) t.part[i][at - begin] = 0.f;
            return;
        }
        begin = t.part_end[i];
    }
    const int b = (int)(at - begin);
    if (b < 0 || b >= t.B || (mask && !mask[b])) return;
    t.counters[b] = t.counters[t.B + b] = 0;
    t.first[b] = t.exec[b] = 1;
}

// generic masked fill of per-row state: buf[b][0..n) = 0 where mask
__global__ void k_reset_rows_f32(float* __restrict__ buf, long n_per_row, int B, const uint8_t* __restrict__ mask) {
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)B * n_per_row) return;
    int b = (int)(idx / n_per_row);
    if (mask && !mask[b]) return;
    buf[idx] = 0.f;
}

// counters -> 0, first -> 1, exec -> 1 for the reset rows (streaming.py:43-44, conv.py:166-169, transformer.py:329-334)
__global__ void k_reset_counters(long* __restrict__ counters, int n_counters, uint8_t* __restrict__ first,
                                 uint8_t* __restrict__ exec, int B, const uint8_t* __restrict__ mask) {
    int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid >= B) return;
    if (mask && !mask[gid]) return;
    for (int i = 0; i < n_counters; ++i) counters[(long)i * B + gid] = 0;
    if (first) first[gid] = 1;
    exec[gid] = 1;
}

__global__ void k_set_mask(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src, int B) {
    int gid = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (gid < B) dst[gid] = src[gid] ? 1 : 0;
}

// ------------------------------------------------------------------------------------------------
// Mimi transformer pieces ([B][C][T] layout)
// ------------------------------------------------------------------------------------------------
// RoPE (rope.py:11-82, interleaved) on q,k + ring-KV write (transformer.py:236-253) + masked attention over the
// valid part of the ring (transformer.py:574-585).  One block per (b, head); T queries (T <= 8).
//   qkv  [B][3*H*D][T]  rows: q = h*D + d, k = H*D + h*D + d, v = 2*H*D + h*D + d   (transformer.py:557-559)
//   kc/vc [B][H][cap][D];  offsets[b] = tokens seen so far (== RingKVCache.end_offset == MHA offset)
struct MimiAttnArgs {
    const float* qkv;
    float* kc;
    float* vc;
    const long* offsets;
    float* outp;   // operand of out_proj (mmi_lin_index: feature h*D+d, column b*T+t)
    int outJ;
    int B, H, D, T, cap, context;
    float max_period;
};

// Several frames at once: T = all of the call's positions.  A frame's positions enter the ring together, so a query sees the positions of
// (last - cap, own], `last` being its frame's last one.  Those of this call are read from its own rows and reach the ring after all layers
// (k_mimi_group_ring): the ring cannot hold what the call's oldest and its newest query see at the same time.
struct MimiGroupRows {
    int T, qkv_ld;
    float *q, *kn, *vn;        // [B][H][T][D]
};

// 256 threads; D/4 lanes share a ring row (one 16-byte load each), so a wave instruction reads 64/(D/4) consecutive
// rows.  Only the min(offset + T, cap) valid slots are visited (the reference masks all `cap`).  Head dim D and the
// steps per frame T are compile-time so that the query slices live in registers and every loop unrolls.
// Dynamic LDS: qs[T][D] | sc[T][cap] | red[(256/(D/4)) * T * D].
template <int D, int T>
__global__ __launch_bounds__(256) void k_mimi_attn(MimiAttnArgs a) {
    constexpr int LPR = D / 4;             // lanes per row
    constexpr int RPB = 256 / LPR;         // rows per block pass
    const int b = blockIdx.x / a.H, h = blockIdx.x % a.H;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cap = a.cap;
    MMI_DYN_SHARED(float, sm);
    float* qs = sm;               // [T][D] roped queries
    float* sc = qs + T * D;       // [T][cap] scores / probabilities
    float* red = sc + ((T * cap + 3) & ~3);   // [RPB][T][D] partial outputs (16-byte aligned: written as f32x4)
    const long off = a.offsets[b];
    const int HD = a.H * D;
    const float* qrow = a.qkv + (long)b * 3 * HD * T;
    float* kcb = a.kc + ((long)b * a.H + h) * cap * D;
    float* vcb = a.vc + ((long)b * a.H + h) * cap * D;

    // phase 1: rope(q), rope(k) -> ring, v -> ring (written unconditionally, transformer.py:243-250)
    for (int i = tid; i < T * (D / 2); i += 256) {
        const int t = i / (D / 2), j = i % (D / 2);
        const float freq = expf((float)j * (-logf(a.max_period) * 2.0f / (float)D));
        const float ts = (float)(off + t);
        const float ang = freq * ts;
        const float c = cosf(ang), s = sinf(ang);
        const float qr = qrow[(long)(h * D + 2 * j) * T + t], qi = qrow[(long)(h * D + 2 * j + 1) * T + t];
        const float kr = qrow[(long)(HD + h * D + 2 * j) * T + t], ki = qrow[(long)(HD + h * D + 2 * j + 1) * T + t];
        float q_re, q_im, k_re, k_im;          // (plain VALU rotations: see mmi_rope_rotate)
        mmi_rope_rotate(qr, qi, c, s, q_re, q_im);
        mmi_rope_rotate(kr, ki, c, s, k_re, k_im);
        qs[t * D + 2 * j] = q_re;
        qs[t * D + 2 * j + 1] = q_im;
        const int slot = (int)((off + t) % cap);
        kcb[(long)slot * D + 2 * j] = k_re;
        kcb[(long)slot * D + 2 * j + 1] = k_im;
    }
    for (int i = tid; i < T * D; i += 256) {
        const int t = i / D, d = i % D;
        const int slot = (int)((off + t) % cap);
        vcb[(long)slot * D + d] = qrow[(long)(2 * HD + h * D + d) * T + t];
    }
    __syncthreads();

    // phase 2: scores over the valid slots.  positions of ring slots after this call's write (transformer.py:258-286)
    const long last = off + T - 1;
    const int end_index = (int)(last % cap);
    const long end_new = off + T;
    const int L = (int)(end_new < (long)cap ? end_new : (long)cap);
    const float scale = 1.0f / sqrtf((float)D);
    const int seg = tid % LPR, rsub = tid / LPR;
    f32x4 qv[T];
#pragma unroll
    for (int t = 0; t < T; ++t) qv[t] = *reinterpret_cast<const f32x4*>(qs + t * D + seg * 4);
    constexpr int NP = 8;                             // ring rows in flight per thread (unconditional, clamped loads)
    for (int s0 = 0; s0 < L; s0 += NP * RPB) {        // block-uniform trip count
        f32x4 kk[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) kk[i] = *reinterpret_cast<const f32x4*>(kcb + (long)min(s0 + i * RPB + rsub, L - 1) * D + seg * 4);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int slot = s0 + i * RPB + rsub;
            const int delta = slot - end_index;
            const long pos = delta <= 0 ? last + delta : last + delta - cap;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                float dv = (qv[t][0] * kk[i][0] + qv[t][1] * kk[i][1]) + (qv[t][2] * kk[i][2] + qv[t][3] * kk[i][3]);
                if constexpr (LPR == 16) dv = mmi_row_sum(dv);
                else
#pragma unroll
                    for (int m = LPR / 2; m >= 1; m >>= 1) dv += mmi_shfl_xor(dv, m);
                if (seg == 0 && slot < L) {
                    const long dq = (off + t) - pos;
                    const bool ok = pos >= 0 && dq >= 0 && dq < a.context;
                    sc[t * cap + slot] = ok ? dv * scale : -INFINITY;
                }
            }
        }
    }
    __syncthreads();

    // phase 3: softmax per query over [0, L): wave t owns query t (T <= 4 waves), so the reductions are wave shuffles
    if (wave < T) {
        const int t = wave;
        float m = -INFINITY;
        for (int slot = lane; slot < L; slot += 64) m = fmaxf(m, sc[t * cap + slot]);
#pragma unroll
        for (int x = 32; x >= 1; x >>= 1) m = fmaxf(m, mmi_shfl_xor(m, x));
        float sum = 0.f;
        for (int slot = lane; slot < L; slot += 64) {
            const float e = expf(sc[t * cap + slot] - m);
            sc[t * cap + slot] = e;
            sum += e;
        }
#pragma unroll
        for (int x = 32; x >= 1; x >>= 1) sum += mmi_shfl_xor(sum, x);
        const float inv = 1.0f / sum;
        for (int slot = lane; slot < L; slot += 64) sc[t * cap + slot] *= inv;
    }
    __syncthreads();

    // phase 4: out[t][d] = sum_slot p[t][slot] * V[slot][d]
    float acc[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] = 0.f;
    for (int s0 = 0; s0 < L; s0 += NP * RPB) {
        f32x4 vv[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) vv[i] = *reinterpret_cast<const f32x4*>(vcb + (long)min(s0 + i * RPB + rsub, L - 1) * D + seg * 4);
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const int slot = s0 + i * RPB + rsub;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const float pr = slot < L ? sc[t * cap + slot] : 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[t][e] += pr * vv[i][e];
            }
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
        *reinterpret_cast<f32x4*>(red + (rsub * T + t) * D + seg * 4) = f32x4{acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
    __syncthreads();
    for (int i = tid; i < T * D; i += 256) {
        const int t = i / D, d = i % D;
        float s = 0.f;
#pragma unroll 8
        for (int r = 0; r < RPB; ++r) s += red[(r * T + t) * D + d];
        a.outp[mmi_lin_index(h * D + d, b * T + t, a.outJ)] = s;
    }
}

// Same operation in ONE memory round trip, for rings of at most 8 * (512 / (D/4)) slots (Mimi: 250 slots of 64 floats):
// every thread first issues its 8 key and 8 value row segments (unconditional, clamped loads: 128 KiB per workgroup in
// flight), ropes the new tokens while they travel, and then keeps scores, exponentials and the weighted value sum in
// registers.  The slots written by this call are taken from LDS instead of the ring (the ring loads were issued before the write).
// GROUP: one workgroup per (b, head) and frame (blockIdx.y) of a MimiGroupRows call; the same sums in the same order as frame by frame.
// Bound by the instructions of its eight waves (one workgroup per head: 8 CUs of a live stream).  Hence a score lives in ONE lane of the
// D/4 that share its row - lane j % (D/4) keeps row pass i of query t, j = 8 t + i - so that mask and exponential are formed once and not D/4
// times; its weight goes back to the others as a DPP broadcast.  The waves agree on the maximum before the exponentials: nothing is rescaled
// behind them.  One stream 8.6 -> 6.0, 32 streams 10.3 -> 7.5, a file's 129 frames 23.3 -> 11.7 us.
// (Requesting the whole ring before the offset that says how much of it is valid measured slower, 9.0 -> 10.1 us at 50 of 250 rows.)
template <int D, int T, bool GROUP = false>
__global__ __launch_bounds__(512) void k_mimi_attn_1pass(MimiAttnArgs a, MimiGroupRows g) {
    constexpr int LPR = D / 4;                   // lanes per ring row
    constexpr int RPB = 512 / LPR;               // rows per block pass
    constexpr int IT = 8;                        // passes: cap <= IT * RPB
    constexpr int NS = (T * IT + LPR - 1) / LPR; // scores per lane
    constexpr int WAVES = 8;
    const int b = blockIdx.x / a.H, h = blockIdx.x % a.H;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cap = a.cap;
    MMI_SHARED __attribute__((aligned(16))) float qs[T * D];
    MMI_SHARED __attribute__((aligned(16))) float kn[T * D];
    MMI_SHARED __attribute__((aligned(16))) float vn[T * D];
    MMI_SHARED __attribute__((aligned(16))) float red[WAVES * T * D];
    MMI_SHARED float mw[WAVES * T];
    MMI_SHARED float sw[WAVES * T];
    const long off0 = a.offsets[b], off = off0 + (GROUP ? (long)blockIdx.y * T : 0);
    const int HD = a.H * D;
    const float* qrow = a.qkv + (long)b * 3 * HD * T;
    float* kcb = a.kc + ((long)b * a.H + h) * cap * D;
    float* vcb = a.vc + ((long)b * a.H + h) * cap * D;
    const int seg = tid % LPR, rsub = tid / LPR;
    f32x4 kk[IT], vv[IT], qv[T];
    const long last = off + T - 1;
    // slot of the first new token (a 64-bit remainder is some 200 dependent instructions)
    const int slot0 = off < (1L << 31) ? (int)((unsigned)off % (unsigned)cap) : (int)(off % cap);
    auto new_slot = [&](int t) __attribute__((always_inline)) {
        const int x = slot0 + t;
        return x < cap ? x : (T <= cap || x < 2 * cap ? x - cap : x % cap);
    };
    const int end_index = new_slot(T - 1);
    const long end_new = off + T;
    const int L = (int)(end_new < (long)cap ? end_new : (long)cap);
    // rows past the valid ones repeat one that this stream has written since it began: their weight is 0, and 0 x NaN is NaN
    const int rows = GROUP ? L : (off < (long)cap ? max((int)off, 1) : cap);
    if constexpr (GROUP) {
#pragma unroll
        for (int t = 0; t < T; ++t) qv[t] = *reinterpret_cast<const f32x4*>(g.q + ((long)blockIdx.x * g.T + (long)blockIdx.y * T + t) * D + seg * 4);
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int slot = min(i * RPB + rsub, rows - 1);
        const long r = (long)slot * D + seg * 4;
        if constexpr (GROUP) {
            const long pos = slot <= end_index ? last + slot - end_index : last + slot - end_index - cap, n = pos - off0;
            const long w = (((long)blockIdx.x * g.T) + (n > 0 ? n : 0)) * D + seg * 4;
            kk[i] = *reinterpret_cast<const f32x4*>(n >= 0 ? g.kn + w : kcb + r);
            vv[i] = *reinterpret_cast<const f32x4*>(n >= 0 ? g.vn + w : vcb + r);
        } else {
            kk[i] = *reinterpret_cast<const f32x4*>(kcb + r);
            vv[i] = *reinterpret_cast<const f32x4*>(vcb + r);
        }
    }

    int newslot[T];
#pragma unroll
    for (int t = 0; t < T; ++t) newslot[t] = new_slot(t);
    if constexpr (!GROUP) {
        if (off == 0)                              // (there is no such row yet)
#pragma unroll
            for (int i = 0; i < IT; ++i) vv[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        // rope(q), rope(k) -> LDS and ring, v -> LDS and ring (written unconditionally, transformer.py:243-250)
        if (tid < T * (D / 2)) {
            const int t = tid / (D / 2), j = tid % (D / 2);
            const float freq = expf((float)j * (-logf(a.max_period) * 2.0f / (float)D));
            const float ang = freq * (float)(off + t);
            const float c = cosf(ang), s = sinf(ang);
            const float qr = qrow[(long)(h * D + 2 * j) * T + t], qi = qrow[(long)(h * D + 2 * j + 1) * T + t];
            const float kr = qrow[(long)(HD + h * D + 2 * j) * T + t], ki = qrow[(long)(HD + h * D + 2 * j + 1) * T + t];
            mmi_rope_rotate(qr, qi, c, s, qs[t * D + 2 * j], qs[t * D + 2 * j + 1]);      // (plain VALU rotations: see mmi_rope_rotate)
            mmi_rope_rotate(kr, ki, c, s, kn[t * D + 2 * j], kn[t * D + 2 * j + 1]);
        } else if (tid >= 512 - T * D) {
            const int i = tid - (512 - T * D), t = i / D, d = i % D;
            vn[i] = qrow[(long)(2 * HD + h * D + d) * T + t];
        }
        __syncthreads();
        if (tid < T * D) {
            const int t = tid / D, d = tid % D;
            const long slot = new_slot(t);
            kcb[slot * D + d] = kn[tid];
            vcb[slot * D + d] = vn[tid];
        }
#pragma unroll
        for (int t = 0; t < T; ++t) qv[t] = *reinterpret_cast<const f32x4*>(qs + t * D + seg * 4);
#pragma unroll
        for (int i = 0; i < IT; ++i)
#pragma unroll
            for (int t = 0; t < T; ++t)
                if (i * RPB + rsub == newslot[t]) {        // a later token of this call overwrites an earlier one when T > cap never happens (T <= 2 <= cap)
                    kk[i] = *reinterpret_cast<const f32x4*>(kn + t * D + seg * 4);
                    vv[i] = *reinterpret_cast<const f32x4*>(vn + t * D + seg * 4);
                }
    }

    float s[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) s[n] = 0.f;
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
        for (int t = 0; t < T; ++t) {
            float dv = mmi_fma(qv[t][3], kk[i][3], mmi_fma(qv[t][2], kk[i][2], mmi_fma(qv[t][1], kk[i][1], qv[t][0] * kk[i][0])));
            if constexpr (LPR == 16) dv = mmi_row_sum(dv);
            else dv = mmi_group_sum<LPR>(dv);
            const int j = t * IT + i;
            s[j / LPR] = seg == j % LPR ? dv : s[j / LPR];
        }
    // position held by a slot (transformer.py:258-286): last + delta, or a ring length before that; a query sees its own and `context` - 1 before it
    const float scale = 1.0f / sqrtf((float)D);
    int query[NS];
    float mx[T], sum[T];
#pragma unroll
    for (int t = 0; t < T; ++t) { mx[t] = -INFINITY; sum[t] = 0.f; }
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        const int j = n * LPR + seg, slot = (j & (IT - 1)) * RPB + rsub, delta = slot - end_index;
        query[n] = j / IT;
        const int dq = query[n] - (T - 1) - (delta <= 0 ? delta : delta - cap);
        const bool ok = j < T * IT && slot < L && dq >= 0 && dq < a.context;
        s[n] = ok ? s[n] * scale : -INFINITY;
#pragma unroll
        for (int t = 0; t < T; ++t) mx[t] = fmaxf(mx[t], query[n] == t ? s[n] : -INFINITY);
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        mx[t] = mmi_wave_max_f32(mx[t]);
        if (lane == 0) mw[wave * T + t] = mx[t];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mx[t] = fmaxf(mx[t], mw[w * T + t]);
#pragma unroll
    for (int n = 0; n < NS; ++n) {
        float m = mx[0];
#pragma unroll
        for (int t = 1; t < T; ++t) m = query[n] == t ? mx[t] : m;
        s[n] = expf(s[n] - m);
#pragma unroll
        for (int t = 0; t < T; ++t) sum[t] += query[n] == t ? s[n] : 0.f;
    }
    float acc[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] = 0.f;
    mmi_static_for<T * IT>([&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value, t = j / IT, i = j % IT;
        const float p = mmi_group_bcast<LPR, j % LPR>(s[j / LPR]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] = mmi_fma(p, vv[i][e], acc[t][e]);
    });
#pragma unroll
    for (int t = 0; t < T; ++t) {
        sum[t] = mmi_rows_sum(mmi_group_sum<16>(sum[t]));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = LPR; m < 16; m <<= 1) acc[t][e] += mmi_shfl_xor(acc[t][e], m);
            acc[t][e] = mmi_rows_sum(acc[t][e]);
        }
        if (lane < LPR) *reinterpret_cast<f32x4*>(red + (wave * T + t) * D + seg * 4) = f32x4{acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
        if (lane == 0) sw[wave * T + t] = sum[t];
    }
    __syncthreads();
    if (tid < T * D) {
        const int t = tid / D, d = tid % D;
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            num += red[(w * T + t) * D + d];
            den += sw[w * T + t];
        }
        a.outp[mmi_lin_index(h * D + d, GROUP ? b * g.T + (int)blockIdx.y * T + t : b * T + t, a.outJ)] = num / den;
    }
}

// Rows of a call that brings several frames of a stream at once (MimiGroupRows): qkv [B][3 H D][ld] -> rotated queries, rotated keys and
// values row by row [b][h][T][D], through LDS so that both sides move whole lines.
#define MIMI_ROPE_T 8         // positions per workgroup: one rotation per thread at 64 dimensions
template <int D>
__global__ __launch_bounds__(256) void k_mimi_group_rope(MimiAttnArgs a, MimiGroupRows g) {
    const int b = (int)blockIdx.x / a.H, h = (int)blockIdx.x % a.H, t0 = (int)blockIdx.y * MIMI_ROPE_T, tid = (int)threadIdx.x;
    const int HD = a.H * D;
    MMI_SHARED float tile[3 * D * (MIMI_ROPE_T + 1)];                     // [q | k | v][d][t]
    for (int i = tid; i < 3 * D * MIMI_ROPE_T; i += 256) {
        const int t = i % MIMI_ROPE_T, d = i / MIMI_ROPE_T % D, w = i / MIMI_ROPE_T / D;
        tile[(w * D + d) * (MIMI_ROPE_T + 1) + t] = a.qkv[((long)b * 3 * HD + w * HD + h * D + d) * g.qkv_ld + min(t0 + t, g.T - 1)];
    }
    __syncthreads();
    const long off = a.offsets[b], row0 = (long)blockIdx.x * g.T + t0;
    for (int i = tid; i < MIMI_ROPE_T * (D / 2); i += 256) {
        const int j = i % (D / 2), t = i / (D / 2);
        if (t0 + t >= g.T) continue;
        const float freq = expf((float)j * (-logf(a.max_period) * 2.0f / (float)D));
        const float ang = freq * (float)(off + t0 + t);
        const float c = cosf(ang), s = sinf(ang);
        float q0, q1, k0, k1;
        mmi_rope_rotate(tile[(2 * j) * (MIMI_ROPE_T + 1) + t], tile[(2 * j + 1) * (MIMI_ROPE_T + 1) + t], c, s, q0, q1);
        mmi_rope_rotate(tile[(D + 2 * j) * (MIMI_ROPE_T + 1) + t], tile[(D + 2 * j + 1) * (MIMI_ROPE_T + 1) + t], c, s, k0, k1);
        const long at = (row0 + t) * D + 2 * j;
        g.q[at] = q0; g.q[at + 1] = q1;
        g.kn[at] = k0; g.kn[at + 1] = k1;
        g.vn[at] = tile[(2 * D + 2 * j) * (MIMI_ROPE_T + 1) + t]; g.vn[at + 1] = tile[(2 * D + 2 * j + 1) * (MIMI_ROPE_T + 1) + t];
    }
}

// kvn [layer][k | v][B][H][T][D] -> kv [layer][k | v][B][H][cap][D], four values per thread
__global__ void k_mimi_group_ring(const float* __restrict__ kvn, float* __restrict__ kv, const long* __restrict__ offsets, int L, int B, int H, int T,
                                  int cap, int D) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int n = T < cap ? T : cap, D4 = D / 4;
    if (idx >= (long)L * 2 * B * H * n * D4) return;
    const int d = (int)(idx % D4), t = T - n + (int)(idx / D4 % n);
    const long row = idx / D4 / n;                         // (layer, k | v, b, h)
    const int b = (int)(row / H % B);
    reinterpret_cast<f32x4*>(kv)[(row * cap + (offsets[b] + t) % cap) * D4 + d] = reinterpret_cast<const f32x4*>(kvn)[(row * T + t) * D4 + d];
}

// ------------------------------------------------------------------------------------------------
// residual vector quantiser (core_vq.py:270-287,507-528; vq.py:126-151,269-287)
// ------------------------------------------------------------------------------------------------
// Distances are evaluated in fp64 (||e||^2 - 2 x.e; the ||x||^2 term is constant per row), i.e. the exact
// nearest centroid of the fp32 inputs, lowest index on ties - the answer the reference's fp32 cdist
// agrees with except at ~1e-7-relative near-ties.
#define MMI_RVQ_CHUNK 32
// One level of one half of the split quantiser.  A launch carries two of them (grid.z picks): the semantic quantiser's only level and the
// acoustic quantiser's first level work on different halves of the projected latent and do not depend on each other
// (vq.py:269-287 SplitResidualVectorQuantizer.encode).
struct RvqLevel {
    const float* x;        // residual rows [Bn][x_rstride] in front of the previous level
    float* x_next;         // ... and behind it, for the next level (another buffer)
    const float* E;        // codebook [bins][D]
    const double* e2;      // ||e||^2
    double* best_d;        // [Bn][nchunk] nearest code of each chunk
    int* best_i;
    const float* prev_E;   // the previous level, null in front of a half's first one
    const double* prev_d;
    const int* prev_i;
    int prev_level;        // column of `codes`
};

// the winning code of a row: a strided scan of the chunk winners by one wave (lowest index on ties)
__device__ __forceinline__ int mmi_rvq_winner(const double* __restrict__ best_d, const int* __restrict__ best_i, int nchunk, int lane) {
    double bd = INFINITY;
    int bi = 0x7fffffff;
    for (int ch = lane; ch < nchunk; ch += 64) mmi_pair_min(bd, bi, best_d[ch], best_i[ch]);
    mmi_wave_pair_min(bd, bi);
    return bi == 0x7fffffff ? 0 : bi;              // no distance is a number (a NaN or infinite latent): where an argmin over NaNs ends
}

// grid (chunks of 32 codes, groups of `group` <= 8 rows, levels); 256 threads, D % 4 == 0.  Every workgroup picks the previous level's winners of its rows
// and takes their centroids off (the first chunk's workgroup stores codes and residuals), then thread (code c, part p) forms the products of its
// part of a code - the quads p, p + 8, ... - with all of its rows.
// Bound by its chain of dependent loads (winners, centroid).  The selection was a launch of its own behind every level (one stream: 9.5 + 4.4 us a
// level, now 5.0); thread (code, row) with the whole dot product left 7 of 8 threads idle at one row and read every code from LDS once per row
// (32 rows: 11.9 + 4.5 us, now 8.0; 129 rows: 22.6 + 4.7, now 16.4, with the rows' LDS reads in front).
template <int NR>
__device__ __forceinline__ void mmi_rvq_products(double (&acc)[8], const f32x4 (&ev)[8], const double* xs, int D, int q0, int p) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = q0 + p + 8 * i;
        if (4 * q >= D) break;
        const double e0 = ev[i][0], e1 = ev[i][1], e2 = ev[i][2], e3 = ev[i][3];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const double* x = xs + r * D + 4 * q;
            acc[r] = fma(e3, x[3], fma(e2, x[2], fma(e1, x[1], fma(e0, x[0], acc[r]))));
        }
    }
}
__global__ __launch_bounds__(256) void k_rvq_level(RvqLevel l0, RvqLevel l1, int x_rstride, int Bn, int group, int D, int bins, int nchunk,
                                                   int* __restrict__ codes, int codes_rstride) {
    const RvqLevel& L = blockIdx.z == 0 ? l0 : l1;
    MMI_DYN_SHARED(double, xs);              // [8][D]
    MMI_SHARED int win[8];
    MMI_SHARED double wd[4 * 8];
    MMI_SHARED int wi[4 * 8];
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int chunk = blockIdx.x, c0 = chunk * MMI_RVQ_CHUNK, rg0 = (int)blockIdx.y * group, nr = min(group, Bn - rg0);
    const int D4 = D >> 2, c = tid >> 3, p = tid & 7;
    const int code = min(c0 + c, bins - 1);
    const f32x4* Ec = reinterpret_cast<const f32x4*>(L.E + (long)code * D);
    f32x4 ev[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) ev[i] = Ec[min(p + 8 * i, D4 - 1)];
    const double en = L.e2[code];
    const int xr = tid >> 5, j0 = tid & 31;
    const f32x4* xp = reinterpret_cast<const f32x4*>(L.x + (long)(rg0 + min(xr, nr - 1)) * x_rstride);
    const f32x4 xa = xp[min(j0, D4 - 1)], xb = xp[min(j0 + 32, D4 - 1)];
    if (L.prev_E) {
        for (int r = wave; r < nr; r += 4) {
            const int best = mmi_rvq_winner(L.prev_d + (long)(rg0 + r) * nchunk, L.prev_i + (long)(rg0 + r) * nchunk, nchunk, lane);
            if (lane == 0) {
                win[r] = best;
                if (chunk == 0) codes[(long)(rg0 + r) * codes_rstride + L.prev_level] = best;
            }
        }
        __syncthreads();
    }
    if (xr < nr) {
        const f32x4* pe = L.prev_E ? reinterpret_cast<const f32x4*>(L.prev_E + (long)win[xr] * D) : nullptr;
        f32x4* xn = reinterpret_cast<f32x4*>(L.x_next + (long)(rg0 + xr) * x_rstride);
        for (int j = j0; j < D4; j += 32) {
            f32x4 v = j == j0 ? xa : (j == j0 + 32 ? xb : xp[j]);
            if (pe) {
                const f32x4 e = pe[j];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] -= e[k];
                if (chunk == 0) xn[j] = v;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) xs[xr * D + 4 * j + k] = (double)v[k];
        }
    }
    __syncthreads();
    double acc[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) acc[r] = 0.0;
    for (int q0 = 0;;) {                     // 256 dimensions at a time
        if (nr == 1) mmi_rvq_products<1>(acc, ev, xs, D, q0, p);
        else if (nr == 2) mmi_rvq_products<2>(acc, ev, xs, D, q0, p);
        else if (nr <= 4) mmi_rvq_products<4>(acc, ev, xs, D, q0, p);
        else mmi_rvq_products<8>(acc, ev, xs, D, q0, p);
        if ((q0 += 64) >= D4) break;
#pragma unroll
        for (int i = 0; i < 8; ++i) ev[i] = Ec[min(q0 + p + 8 * i, D4 - 1)];
    }
    double dot = 0.0;                        // lane (c, p): row p
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const double t = mmi_group8_sum_f64(acc[r]);
        dot = r == p ? t : dot;
    }
    double dist = en - 2.0 * dot;
    int idx = c0 + c;
    if (idx >= bins || p >= nr || dist != dist) { dist = INFINITY; idx = 0x7fffffff; }
    mmi_group8_pair_min(dist, idx);
    if (lane < 8) { wd[wave * 8 + lane] = dist; wi[wave * 8 + lane] = idx; }
    __syncthreads();
    if (tid < nr) {
        dist = wd[tid]; idx = wi[tid];
#pragma unroll
        for (int w = 1; w < 4; ++w) mmi_pair_min(dist, idx, wd[w * 8 + tid], wi[w * 8 + tid]);
        L.best_d[(long)(rg0 + tid) * nchunk + chunk] = dist;
        L.best_i[(long)(rg0 + tid) * nchunk + chunk] = idx;
    }
}

// the codes of the halves' last levels: prev_* of l0 (and l1), one wave per row
__global__ __launch_bounds__(256) void k_rvq_last(RvqLevel l0, RvqLevel l1, int Bn, int nchunk, int* __restrict__ codes, int codes_rstride) {
    const RvqLevel& L = blockIdx.y == 0 ? l0 : l1;
    const int r = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6), lane = (int)threadIdx.x & 63;
    if (r >= Bn) return;
    const int best = mmi_rvq_winner(L.prev_d + (long)r * nchunk, L.prev_i + (long)r * nchunk, nchunk, lane);
    if (lane == 0) codes[(long)r * codes_rstride + L.prev_level] = best;
}

// decode: q[b][0:D] = E_0[c_0]; q[b][D:2D] = ((0 + E_1[c_1]) + E_2[c_2]) + ...   (core_vq.py:521-528)
// n_codes_dev (optional): the number of codebooks of THIS call, read from device memory so that the captured decoder program
// serves `decode` calls with any K <= n_q (the split RVQ decodes however many codebooks it is given, vq.py:281-287)
__global__ void k_rvq_gather(const int* __restrict__ codes, int codes_rstride, int n_codes,
                             const float* __restrict__ Eall, int bins, int D, int n_sem, float* __restrict__ q, int Bn,
                             const int* __restrict__ n_codes_dev, float* __restrict__ qp, int qpQ) {
    int idx = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (idx >= Bn * D) return;
    int r = idx / D, d = idx % D;
    float first = 0.f, rest = 0.f;
    // eight codes, then their eight entries are asked for at once, whatever their number turns out to be (a row holds codes_rstride codes, as many as
    // there are codebooks): one after the other, 8 of them took 5.5 - 7 us, here 3.7
    if (n_codes_dev) n_codes = *n_codes_dev;
    constexpr int N = 8;
    for (int k0 = 0; k0 < codes_rstride; k0 += N) {
        int c[N];
        float e[N];
#pragma unroll
        for (int i = 0; i < N; ++i) c[i] = codes[(long)r * codes_rstride + min(k0 + i, codes_rstride - 1)];
#pragma unroll
        for (int i = 0; i < N; ++i) e[i] = Eall[((long)min(k0 + i, codes_rstride - 1) * bins + max(0, min(c[i], bins - 1))) * D + d];      // the reference crashes on OOB codes (vq.py:144-146); we clamp
#pragma unroll
        for (int i = 0; i < N; ++i) {
            if (k0 + i >= n_codes) continue;
            if (k0 + i < n_sem) first += e[i]; else rest += e[i];
        }
        if (k0 + N >= n_codes) break;
    }
    q[(long)r * 2 * D + d] = first;
    q[(long)r * 2 * D + D + d] = rest;
    if (qp) {   // also as the packed B operand of the output projection (column = row r): no k_pack_b_f32 launch in between
        qp[mmi_bp_index(d, r, qpQ)] = first;
        qp[mmi_bp_index(D + d, r, qpQ)] = rest;
    }
}

// int64 <-> int32 code tensors at the ABI boundary: [B][K][F] i64 <-> [B * G][K] i32 of the G frames from f on
__global__ void k_codes_out(const int* __restrict__ src, int src_rstride, long* __restrict__ dst, int B, int K, int F,
                            int f, int G) {
    int idx = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (idx >= B * G * K) return;
    int r = idx / K, k = idx % K, b = r / G;
    dst[((long)b * K + k) * F + f + r - b * G] = (long)src[(long)r * src_rstride + k];
}
// src: i64 [B][K][F] with `src_bstride` elements between batch rows (K * F when dense; larger for a column slice of a wider
// tensor such as LMGen's [B][1 + dep_q][1] step output read from its second column on)
__global__ void k_codes_in(const long* __restrict__ src, long src_bstride, int* __restrict__ dst, int dst_rstride, int B, int K,
                           int F, int f, int G) {
    int idx = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (idx >= B * G * K) return;
    int r = idx / K, k = idx % K, b = r / G;
    dst[(long)r * dst_rstride + k] = (int)src[(long)b * src_bstride + (long)k * F + f + r - b * G];
}
