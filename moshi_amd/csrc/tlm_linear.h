// Mixers of the token language models that carry a matrix per head and sequence, S [dim][vdim] fp32:
//
//   lightning      S <- d S + k v^T                                                  o = S^T q      d: a constant per head
//   channel delta  S <- g * S (per row); u = b (v - S^T k); S <- S + k u^T           o = S^T q      g: per head, row and token
//
// Everything in this file is fp32 (v_mfma_f32_16x16x4_f32, an exact fma chain), in the bf16 format too.  Sequences that bring at most
// TLM_SMALL tokens in a step go through k_tlm_state_step, token by token with S in registers.  Prompt portions are cut into chunks of 64
// tokens: what does not depend on S is computed for all chunks in parallel, then k_tlm_chunk_scan walks a sequence's chunks with S in the
// registers of four waves per 16 columns.  With G_t the product of the decays from the chunk's first token to t (per row of S):
//
//   u_t + b_t sum_(s<t) (k_t G_t/G_s k_s) u_s = b_t (v_t - S_0^T (G_t k_t))          a unit lower triangular system, (I + A) U = B
//   o_t = S_0^T (G_t q_t) + sum_(s<=t) (q_t G_t/G_s k_s) u_s                         P
//   S_end = G_end S_0 + sum_s (G_end/G_s k_s) u_s^T
//
// so W = (I + A)^-1 diag(b) (G K) and U0 = (I + A)^-1 diag(b) V turn the system into U = U0 - W S_0.  Decay ratios are never formed by a
// division or from logarithms: inside 8 tokens they are running products, across them (product to the end of s's 8) x (whole 8s between)
// x (product from the start of t's 8), so that they lose nothing however strong the decay is, and underflow to the zero they stand for.
#pragma once
#include "tlm_kernels.h"

constexpr int TLM_CHUNK = 64;
constexpr int TLM_SMALL = 4;             // up to here a sequence's tokens are stepped one by one
constexpr int TLM_PST = 68;              // row stride of a 64-column panel in LDS: rows stay 16-byte aligned, columns spread over the banks

struct TlmUnit { int row0, n, slot, par, fresh, chunk0, n_chunks, pad; };      // one sequence of the step; fresh: position 0, the state is zero

// Heads are padded to 16 in both sizes; every per-head section of a buffer has the padded stride.
struct TlmLinArgs {
    const float* in; int in_ld;          // the input projection: columns q0 .. (kv_heads), k0 .. (kv_heads), v0 .. (heads), b0 .. (delta: one per head)
    int q0, k0, v0, b0;
    int heads, kv_heads, dim, vdim, dim_p, vdim_p;
    float q_scale, eps;
    const float* conv_w; float* conv_state; int conv_c, taps;      // delta: [taps][channels]; [slot][2][taps - 1][channels], read one copy and write the other
    const float* decay;                  // delta: projection [row][heads][dim_p] (tlm_decay); lightning: powers 0 .. TLM_CHUNK of every head's constant
    const float* decay_c;                // delta: [2][heads][dim_p] summand, factor
    const float* gate; int gate_ld;      // the normalised output's factor, before its sigmoid
    const float* nw;                     // its weight (delta: per head column, lightning: per column)
    float* state;                        // [slot][heads][dim_p][vdim_p]
    const TlmUnit* small; const TlmUnit* unit; const TlmSeg* chunk;
    float* qkv;                          // delta: convolved and normalised [row][conv_c], same columns as `in`
    // per (chunk, head), in fragments of 16 x 16 (a lane's four elements together, so that the walk's loads are contiguous): w and qg
    // [64][dim_p], kt [dim_p][64], p [64][64] by tlm_tile; u0 [64][vdim_p] in the layout of the matrix core's sums; gend [dim_p]
    float *w, *qg, *kt, *u0, *p, *gend;
    float* o;                            // [row][heads][vdim_p] before the norm
    void* out; int out_ks;               // packed operand of the output projection
};

// decay of channel d of a head: exp(-factor softplus(z)), z = projection + summand, as 2^(-factor log2(1 + e^z)).  With u = e^z rounded
// and w = 1 + u rounded, log2(w) u / (w - 1) is log2(1 + u) to the last bits however small u is.
__device__ __forceinline__ float tlm_decay(float z, float factor) {
    constexpr float LOG2E = 1.44269504088896340736f;
    const float u = mmi_fast_exp2f(fminf(z, 30.f) * LOG2E), w = 1.0f + u;
    float l = w > 1.0f ? mmi_fast_log2f(w) * u / (w - 1.0f) : u * LOG2E;
    if (z > 20.f) l = z * LOG2E;
    return mmi_fast_exp2f(-factor * l);
}
__device__ __forceinline__ float tlm_decay(const TlmLinArgs& a, long row, int h, int d) {
    const int c = h * a.dim_p + d;
    return tlm_decay(a.decay[row * a.heads * a.dim_p + c] + a.decay_c[c], a.decay_c[a.heads * a.dim_p + c]);
}
__device__ __forceinline__ float tlm_silu(float x) { return x * tlm_sigmoid(x); }

// element (row, k) of an operand with `ks` 16-wide blocks per 16 rows
MMI_HD long tlm_tile(int row, int k, int ks) { return (((long)(row >> 4) * ks + (k >> 4)) * 64 + ((k & 15) >> 2) * 16 + (row & 15)) * 4 + (k & 3); }

// four floats of a buffer whose start is the same in every lane: its address stays in scalar registers, a lane adds 32 bits
template <class T = f32x4, class F>
__device__ __forceinline__ auto& tlm_quad(F* base, int at) {
    using C = std::conditional_t<std::is_const_v<F>, const char, char>;
    using E = std::conditional_t<std::is_const_v<F>, const T, T>;
    return *reinterpret_cast<E*>(reinterpret_cast<C*>(base) + 4u * (unsigned)at);
}

// channel c of the convolution at token t of a sequence whose rows start at row0 of the projection; four taps are requested at a time (a tap before
// the sequence's start reads some valid address and counts as zero).  `now`: where the taps - 1 inputs that the next step's first token needs
// stay, or null
__device__ __forceinline__ float tlm_conv(const TlmLinArgs& a, const float* old, int fresh, int row0, int t, int c, float* now) {
    float s = 0.f;
    for (int j0 = 0; j0 < a.taps; j0 += 4) {
        float x[4], w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int tap = min(j0 + j, a.taps - 1), at = t - (a.taps - 1) + tap;
            x[j] = *(at >= 0 || fresh ? a.in + (long)(row0 + max(at, 0)) * a.in_ld + c : old + (long)(a.taps - 1 + at) * a.conv_c + c);
            w[j] = a.conv_w[(long)tap * a.conv_c + c];
            if (j0 + j >= a.taps || (at < 0 && fresh)) x[j] = 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) s += w[j] * x[j];
        if (now)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j0 + j >= 1 && j0 + j < a.taps) now[(long)(j0 + j - 1) * a.conv_c + c] = x[j];
    }
    return s;
}

// ------------------------------------------------------------------------------------------------
// few tokens: one workgroup per (sequence, head), S in registers (thread: 4 columns of every parts-th row)
// ------------------------------------------------------------------------------------------------
inline int tlm_step_groups(int vdim_p) {                  // column groups of 4, a power of two
    int g = 4;
    while (4 * g < vdim_p) g *= 2;
    return g;
}
// sh: q, k, g [parts * RT] (zeros from dim_p on), v [vdim_p], red [2][parts][vdim_p]
template <class Tr, bool DELTA, int RT>
__device__ __forceinline__ void tlm_state_step(const TlmLinArgs& a, float* sh, int cgp, int seq, int h) {
    const int tid = (int)threadIdx.x, nthr = (int)blockDim.x, lane = tid & 63;
    const int parts = nthr / cgp, cg = tid & (cgp - 1), part = tid / cgp, col = 4 * cg;
    const TlmUnit un = a.small[seq];
    const int rep = a.heads / a.kv_heads, kh = h / rep, D = a.dim_p, V = a.vdim_p;
    float *q = sh, *k = q + parts * RT, *g = k + parts * RT, *v = g + parts * RT, *red = v + V;
    for (int i = D + tid; i < parts * RT; i += nthr) q[i] = k[i] = g[i] = 0.f;
    const bool mine = col < V;
    float* S = a.state + ((long)un.slot * a.heads + h) * D * V;
    f32x4 s[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) s[i] = mmi_load_nt(reinterpret_cast<const f32x4*>(S + (long)min(part + parts * i, D - 1) * V + min(col, V - 4)));
#pragma unroll
    for (int i = 0; i < RT; ++i)
        if (un.fresh || !mine || part + parts * i >= D) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* old = nullptr;
    float* now = nullptr;
    if constexpr (DELTA) {
        old = a.conv_state + ((long)un.slot * 2 + un.par) * (a.taps - 1) * a.conv_c;
        now = a.conv_state + ((long)un.slot * 2 + (un.par ^ 1)) * (a.taps - 1) * a.conv_c;
    }
    for (int t = 0; t < un.n; ++t) {
        const long row = un.row0 + t;
        const float* in = a.in + row * a.in_ld;
        // everything the token needs is requested before anything is used: q, k, v and (delta) the decays, one value per thread and round
        f32x4 gt = {0.f, 0.f, 0.f, 0.f}, nw = gt;
        float beta = 0.f;
        if constexpr (DELTA) {
            beta = in[a.b0 + h];
            gt = *reinterpret_cast<const f32x4*>(a.gate + row * a.gate_ld + h * V + min(col, V - 4));
            nw = *reinterpret_cast<const f32x4*>(a.nw + min(col, V - 4));
        }
#pragma unroll 1
        for (int i = tid; i < (DELTA ? 3 : 2) * D + V; i += nthr) {
            if (DELTA && i >= 2 * D + V) {
                g[i - 2 * D - V] = tlm_decay(a, row, h, i - 2 * D - V);
                continue;
            }
            const int c = i < D ? a.q0 + kh * D + i : (i < 2 * D ? a.k0 + kh * D + i - D : a.v0 + h * V + i - 2 * D);
            float x;
            if constexpr (DELTA) x = tlm_silu(tlm_conv(a, old, un.fresh, un.row0, t, c, t + 1 == un.n && (i >= 2 * D || h % rep == 0) ? now : nullptr));      // (the heads of a group share query and key channels)
            else x = in[c];
            if (i < D) q[i] = x;
            else if (i < 2 * D) k[i - D] = x;
            else v[i - 2 * D] = x;
        }
        __syncthreads();
        float qq = 0.f, kk = 0.f, kq = 0.f;                // every wave sums for itself
#pragma unroll 1
        for (int i = lane; i < D; i += 64) {
            qq = mmi_fma(q[i], q[i], qq);
            kk = mmi_fma(k[i], k[i], kk);
            kq = mmi_fma(k[i], q[i], kq);
        }
        kq = tlm_wave_sum(kq);
        float iq = 1.f, ik = 1.f, dec = 1.f;
        if constexpr (DELTA) {
            iq = a.q_scale / sqrtf(tlm_wave_sum(qq) + 1e-6f);
            ik = 1.0f / sqrtf(tlm_wave_sum(kk) + 1e-6f);
            kq *= iq * ik;
            beta = tlm_sigmoid(beta);
        } else {
            dec = a.decay[h * (TLM_CHUNK + 1) + 1];
        }
        f32x4 ak = {0.f, 0.f, 0.f, 0.f}, aq = ak;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int d = part + parts * i;
            s[i] *= DELTA ? g[d] : dec;
            if constexpr (DELTA) ak += (k[d] * ik) * s[i];
            aq += (q[d] * iq) * s[i];
        }
        if (mine) {
            *reinterpret_cast<f32x4*>(red + (long)part * V + col) = aq;
            if constexpr (DELTA) *reinterpret_cast<f32x4*>(red + (long)(parts + part) * V + col) = ak;
        }
        __syncthreads();
        f32x4 u = {0.f, 0.f, 0.f, 0.f}, o = u;
        if (mine) {
#pragma unroll 4
            for (int p = 0; p < parts; ++p) {
                o += *reinterpret_cast<const f32x4*>(red + (long)p * V + col);
                if constexpr (DELTA) u += *reinterpret_cast<const f32x4*>(red + (long)(parts + p) * V + col);
            }
            const f32x4 vv = *reinterpret_cast<const f32x4*>(v + col);
            u = DELTA ? beta * (vv - u) : vv;
            o += kq * u;
        }
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const int d = part + parts * i;
            s[i] += (k[d] * ik) * u;
        }
        if constexpr (DELTA) {
            float ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
            for (int x = 1; x < cgp; x *= 2) ss += mmi_shfl_xor(ss, x);      // (the groups of one row part are neighbours in a wave)
            const float inv = 1.0f / sqrtf(ss / (float)a.vdim + a.eps);
            if (part == 0 && mine) {
#pragma unroll
                for (int e = 0; e < 4; ++e) gt[e] = tlm_sigmoid(gt[e]);
                Tr::store4((typename Tr::elem*)a.out + tlm_index<Tr>(row, h * V + col, a.out_ks), o * inv * nw * gt);
            }
        } else if (part == 0 && mine) {
            *reinterpret_cast<f32x4*>(a.o + (row * a.heads + h) * V + col) = o;
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const int d = part + parts * i;
        if (mine && d < D) mmi_store_nt(reinterpret_cast<f32x4*>(S + (long)d * V + col), s[i]);
    }
}
template <class Tr, bool DELTA, int RT, int MAXB>
__global__ __launch_bounds__(MAXB, MAXB == 512 && !DELTA ? 5 : 4) void k_tlm_state_step(TlmLinArgs a, int cgp) {
    MMI_DYN_SHARED(float, sh);
    tlm_state_step<Tr, DELTA, RT>(a, sh, cgp, (int)blockIdx.x, (int)blockIdx.y);
}

// ------------------------------------------------------------------------------------------------
// chunks: convolutions and unit norms (delta).  grid: chunks, 2 kv_heads + heads, shares of a chunk; a lane takes 4 channels of 4 tokens in a row, which share
// seven inputs per four taps; a power of two of lanes stand side by side.  Bound by its bytes with many chunks, by two trips to memory with few,
// so a workgroup goes round once.  In a prompt's step, heads of 128 x 128, with a token per lane and now: 1773 tokens of 32 heads (174 MB) 54.0 and 42.6 us,
// 639 of 16 15.8 and 12.9
// ------------------------------------------------------------------------------------------------
inline __global__ __launch_bounds__(256, 4) void k_tlm_conv(TlmLinArgs a, int kgroups, int vgroups) {
    const int y = (int)blockIdx.y;
    const TlmSeg ck = a.chunk[blockIdx.x];
    const int kind = y < a.kv_heads ? 0 : (y < 2 * a.kv_heads ? 1 : 2);
    const int width = kind == 2 ? a.vdim_p : a.dim_p, groups = kind == 2 ? vgroups : kgroups;
    const int c0 = kind == 0 ? a.q0 + y * a.dim_p : (kind == 1 ? a.k0 + (y - a.kv_heads) * a.dim_p : a.v0 + (y - 2 * a.kv_heads) * a.vdim_p);
    const int back = a.taps - 1, s0 = ck.index * TLM_CHUNK;
    const float* old = a.conv_state + ((long)ck.slot * 2 + ck.par) * back * a.conv_c + c0;
    float* now = a.conv_state + ((long)ck.slot * 2 + (ck.par ^ 1)) * back * a.conv_c + c0;
    const float *in = a.in + (long)(ck.row0 - s0) * a.in_ld + c0, *cw = a.conv_w + c0;       // in: the sequence's first row of this step
    const int c = 4 * ((int)threadIdx.x & (groups - 1)), cc = min(c, width - 4), step = 4 * (256 / groups);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int t0 = (int)blockIdx.z * step; t0 < ck.n; t0 += (int)gridDim.z * step) {      // (every lane of a wave goes round as often)
        const int t = t0 + 4 * ((int)threadIdx.x / groups);
        f32x4 x[4] = {zero, zero, zero, zero};
        for (int j0 = 0; j0 < a.taps; j0 += 4) {           // (inputs past the chunk or the taps: a valid address, not used)
            f32x4 v[7], w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = *reinterpret_cast<const f32x4*>(cw + (long)min(j0 + j, back) * a.conv_c + cc);
#pragma unroll
            for (int m = 0; m < 7; ++m) {
                const int at = s0 + min(t + j0 + m - back, ck.n - 1);
                v[m] = *reinterpret_cast<const f32x4*>(at >= 0 || ck.fresh ? in + (long)max(at, 0) * a.in_ld + cc : old + (long)(back + at) * a.conv_c + cc);
                if (at < 0 && ck.fresh) v[m] = zero;
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (j0 + j <= back) x[r] += w[j] * v[r + j];
            if (ck.last && t < ck.n && t + 4 >= ck.n && c < width)      // the inputs that the next step's first tokens need
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (t + r + 1 == ck.n)
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (j0 + j >= 1 && j0 + j <= back) *reinterpret_cast<f32x4*>(now + (long)(j0 + j - 1) * a.conv_c + c) = v[r + j];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bool in_place = t + r < ck.n && c < width;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[r][e] = in_place ? x[r][e] * tlm_sigmoid(x[r][e]) : 0.f;
            if (kind != 2) {
                float ss = x[r][0] * x[r][0] + x[r][1] * x[r][1] + x[r][2] * x[r][2] + x[r][3] * x[r][3];
                for (int m = 1; m < groups; m *= 2) ss += mmi_shfl_xor(ss, m);
                x[r] *= (kind == 0 ? a.q_scale : 1.0f) / sqrtf(ss + 1e-6f);
            }
            if (in_place) *reinterpret_cast<f32x4*>(a.qkv + (long)(ck.row0 + t + r) * a.conv_c + c0 + c) = x[r];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// chunks, lightning: P, the decayed queries, the decayed transposed keys.  grid: chunks x heads, in eight waves: wave w has
// token block w % 4 of P and every other column block
// ------------------------------------------------------------------------------------------------
inline size_t tlm_chunk_lightning_smem() { return (size_t)(2 * TLM_CHUNK * TLM_PST + TLM_CHUNK + 1) * sizeof(float); }
__device__ __forceinline__ void tlm_chunk_lightning(const TlmLinArgs& a, float* sh, int chunk, int h) {
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = mmi_uniform(tid >> 6), bl = lane & 15, kq = lane >> 4;
    const int tb = wave & 3, j0 = wave >> 2;
    const TlmSeg ck = a.chunk[chunk];
    const int D = a.dim_p;
    const long id = (long)chunk * a.heads + h;
    float *Q = sh, *K = Q + TLM_CHUNK * TLM_PST, *pw = K + TLM_CHUNK * TLM_PST;      // [64][TLM_PST] twice, [65]
    for (int i = tid; i <= TLM_CHUNK; i += 512) pw[i] = a.decay[h * (TLM_CHUNK + 1) + i];
    const float* qp = a.in + (long)ck.row0 * a.in_ld + a.q0 + h * D;
    const float* kp = a.in + (long)ck.row0 * a.in_ld + a.k0 + h * D;
    float *Qg = a.qg + id * TLM_CHUNK * D, *Kt = a.kt + id * TLM_CHUNK * D, *P = a.p + id * (TLM_CHUNK * TLM_CHUNK);
    f32x4 acc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < D; c0 += 64) {                   // panels of 64 channels (a multiple of 16 in the last one)
        const int cn = min(64, D - c0);
        f32x4 qv[2], kv[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {                      // (rows and columns past the end: a valid address, as zeros)
            const int t = (tid >> 4) + 32 * i, c = min(4 * (tid & 15), cn - 4);
            qv[i] = *reinterpret_cast<const f32x4*>(qp + (long)min(t, ck.n - 1) * a.in_ld + c0 + c);
            kv[i] = *reinterpret_cast<const f32x4*>(kp + (long)min(t, ck.n - 1) * a.in_ld + c0 + c);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = (tid >> 4) + 32 * i, c = 4 * (tid & 15);
            if (t >= ck.n || c >= cn) qv[i] = kv[i] = f32x4{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<f32x4*>(Q + t * TLM_PST + c) = qv[i];
            *reinterpret_cast<f32x4*>(K + t * TLM_PST + c) = kv[i];
            if (c < cn) *reinterpret_cast<f32x4*>(Qg + tlm_tile(t, c0 + c, D / 16)) = qv[i] * pw[t + 1];
        }
        __syncthreads();
        for (int c = 4 * kq; c < cn; c += 16) {
            const u32x4 q = *reinterpret_cast<const u32x4*>(Q + (16 * tb + bl) * TLM_PST + c);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (2 * j + j0 <= tb) acc[j] = TlmF32::mfma(q, *reinterpret_cast<const u32x4*>(K + (16 * (2 * j + j0) + bl) * TLM_PST + c), acc[j]);
        }
        for (int i = wave; i < cn / 4; i += 8) {           // transposed fragments: 16 channels x 16 tokens
            const int c = 16 * (i >> 2) + bl, t = 16 * (i & 3) + 4 * kq;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = t + e < ck.n ? K[(t + e) * TLM_PST + c] * pw[ck.n - 1 - t - e] : 0.f;
            *reinterpret_cast<f32x4*>(Kt + tlm_tile(c0 + c, t, 4)) = v;
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
        if (2 * j + j0 <= tb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = 16 * tb + 4 * kq + r, s = 16 * (2 * j + j0) + bl;
                P[tlm_tile(t, s, 4)] = s <= t ? acc[j][r] * pw[t - s] : 0.f;
            }
    for (int d = tid; d < D; d += 512) a.gend[id * D + d] = pw[ck.n];
}
// BESIDE: with the single tokens of n_small sequences, as beside the delta rule's chunks.  11 chunks and 14 sequences, 16 heads of 128 x 128: 20.9 us in
// launches of their own, 13.2 together.  Chunks alone have a kernel without the other body (58 registers, 94 with it; its bytes bound it where
// chunks are many): 896 of 128 x 128 28.4 us, 31.7 with it, 29.6 in workgroups of four waves; 176 9.5, 9.9 and 12.1.
template <class Tr, bool BESIDE>
__global__ __launch_bounds__(512, 4) void k_tlm_chunk_lightning(TlmLinArgs a, int n_chunk, int n_small, int cgp) {
    MMI_DYN_SHARED(float, sh);
    const int b = (int)blockIdx.x, own = b - n_chunk * a.heads;
    if (!BESIDE || own < 0) tlm_chunk_lightning(a, sh, b % n_chunk, b / n_chunk);
    else tlm_state_step<Tr, false, 8>(a, sh, cgp, own % n_small, own / n_small);
}

// ------------------------------------------------------------------------------------------------
// chunks, delta: P, W, U0, the decayed queries and transposed keys.  grid: chunks, heads; NP: panels of 64 channels, 1, 2 or 4
// Its bytes bound it where chunks are many (896 of 128 x 128: 250 MB, 67 us in a step = 3.7 TB/s; 127 before), the chain of one workgroup's phases
// where they are few (176: 23 us; 47 before).  So: eight waves, two on every SIMD and two workgroups on a CU while the registers (126) allow it; the
// next panel's operands and U0's are asked for a phase ahead; pairs are taken one by one only inside 8 tokens (half the vector work of 16), all
// others by the matrix core; no right side goes through memory: W's stay in the registers of the wave that solves for them.
// ------------------------------------------------------------------------------------------------
constexpr int TLM_SUB = 8;               // tokens whose pairs are taken one by one; decays across them are whole products
inline size_t tlm_chunk_delta_smem() { return (size_t)(3 * TLM_CHUNK * TLM_PST + (3 * (TLM_CHUNK / TLM_SUB) + 1) * 64) * sizeof(float); }
template <int NP>
__device__ __forceinline__ void tlm_chunk_delta(const TlmLinArgs& a, float* sh, int chunk, int h) {
    float *Q = sh, *K = Q + TLM_CHUNK * TLM_PST, *G = K + TLM_CHUNK * TLM_PST;      // [64][TLM_PST] each
    float *tot = G + TLM_CHUNK * TLM_PST, *pre = tot + TLM_CHUNK / TLM_SUB * 64, *suf = pre + TLM_CHUNK / TLM_SUB * 64;      // [8][64] each: decay over 8 tokens, over all 8s before, behind
    float* beta = suf + TLM_CHUNK / TLM_SUB * 64;          // [64]
    float *A = K, *Pl = Q, *part = G, *ti = G;                                      // once the panels are done: [64][TLM_PST] twice; [4][64][4], then [4][16][20]
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = mmi_uniform(tid >> 6);
    int bl = lane & 15, kq = lane >> 4;
    const TlmSeg ck = a.chunk[chunk];
    const int D = a.dim_p, V = a.vdim_p, kh = h / (a.heads / a.kv_heads), nd = D / 16, nv = V / 16;
    const long id = (long)chunk * a.heads + h;
    const float *qp = a.qkv + (long)ck.row0 * a.conv_c + a.q0 + kh * D, *kp = qp + (a.k0 - a.q0), *vp = a.qkv + (long)ck.row0 * a.conv_c + a.v0 + h * V;
    const float *zp = a.decay + ((long)ck.row0 * a.heads + h) * D, *cp = a.decay_c + h * D;
    float *Wg = a.w + id * TLM_CHUNK * D, *Qg = a.qg + id * TLM_CHUNK * D, *Kt = a.kt + id * TLM_CHUNK * D, *Ug = a.u0 + id * TLM_CHUNK * V;
    float* P = a.p + id * (TLM_CHUNK * TLM_CHUNK);
    const float bv = a.in[(long)(ck.row0 + min(lane, ck.n - 1)) * a.in_ld + a.b0 + h];
    // a panel's operands: token lt and the one 32 further on, 4 channels from lc (past the end: a valid address, not used)
    f32x4 qv[2], kv[2], zv[2], zs, zf;
    auto load = [&](int c0, int lt, int lc) __attribute__((always_inline)) {
        const int c = c0 + min(lc, min(64, D - c0) - 4);
        zs = tlm_quad(cp, c);
        zf = tlm_quad(cp + a.heads * D, c);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = min(lt + 32 * i, ck.n - 1);
            zv[i] = tlm_quad(zp, t * a.heads * D + c);
            qv[i] = tlm_quad(qp, t * a.conv_c + c);
            kv[i] = tlm_quad(kp, t * a.conv_c + c);
        }
    };
    load(0, tid >> 4, 4 * (tid & 15));
    if (tid < TLM_CHUNK) beta[tid] = tid < ck.n ? tlm_sigmoid(bv) : 0.f;
    float dA[TLM_SUB], dP[TLM_SUB];                        // pairs (t, t - i), t = 16 (wave % 4) + bl, of this lane's share of the channels
#pragma unroll
    for (int i = 0; i < TLM_SUB; ++i) dA[i] = dP[i] = 0.f;
    // the 16 x 16 blocks that are products: waves 0 .. 5 those below the diagonal, (3,0) (3,1) (3,2) (2,0) (2,1) (1,0); waves 6, 7 the lower left
    // quarters of two blocks on the diagonal each (rows 8 .. 15 of a block against its columns 0 .. 7; the other two quarters are dropped)
    const int bi = wave < 3 ? 3 : (wave < 5 ? 2 : 1), bj = wave < 3 ? wave : (wave < 5 ? wave - 3 : 0);
    auto row = [&](int l) __attribute__((always_inline)) { return wave < 6 ? 16 * bi + l : 32 * (wave - 6) + 16 * (l >> 3) + (l & 7) + 8; };
    auto column = [&](int l) __attribute__((always_inline)) { return wave < 6 ? 16 * bj + l : 32 * (wave - 6) + 16 * (l >> 3) + (l & 7); };
    f32x4 oA = {0.f, 0.f, 0.f, 0.f}, oP = oA;              // transposed: lane (kq, bl) holds columns 4 kq .. 4 kq + 3 of row bl
    // 16-column strips of [W | U0] that this wave solves for: strip 4 p + wave % 4 of W for every other panel p, then every eighth of U0
    constexpr int NS = (NP + 1) / 2;
    f32x4 x[NS + 1][4] = {};
    const int v0 = (wave + 8 - (4 * NP & 7)) & 7;
    auto load_u0 = [&](f32x4* u, int v, int bl, int kq) __attribute__((always_inline)) {       // (past the end: the last strip again, not stored)
        const int at = 16 * min(v, nv - 1) + bl;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) u[i][r] = tlm_quad<float>(vp, min(16 * i + 4 * kq + r, ck.n - 1) * a.conv_c + at);
    };
    auto panel = [&](int c0, bool mine, f32x4* strip) __attribute__((always_inline)) {
        const int cn = min(64, D - c0);                    // a multiple of 16
        int l = lane;
        mmi_here(l);
        const int bl = l & 15, kq = l >> 4, lt = 4 * wave + (l >> 4), lc = 4 * (l & 15);
        if (c0) mmi_meet();
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = lt + 32 * i;
            const bool in = t < ck.n && lc < cn;
            f32x4 g = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float d = tlm_decay(zv[i][e] + zs[e], zf[e]);
                g[e] = in ? d : 1.f;
                qv[i][e] = in ? qv[i][e] : 0.f;
                kv[i][e] = in ? kv[i][e] : 0.f;
            }
            *reinterpret_cast<f32x4*>(Q + t * TLM_PST + lc) = qv[i];
            *reinterpret_cast<f32x4*>(K + t * TLM_PST + lc) = kv[i];
            *reinterpret_cast<f32x4*>(G + t * TLM_PST + lc) = g;
        }
        mmi_meet();
        if (NP <= 2 ? c0 < 64 * (NP - 1) : c0 < 128 || c0 + 64 < D) load(c0 + 64, lt, lc);
        else load_u0(x[NS], v0, bl, kq);
        // pairs inside 8 tokens, with a running decay: token t against t - i.  What t - i before t's 8 gives is dropped at the end: those rows are
        // others of the chunk, or rows of the panel that lies in front in LDS
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int t = 16 * (wave & 3) + bl, c = 32 * (wave >> 2) + 16 * j + 4 * kq;
            const f32x4 kt = *reinterpret_cast<const f32x4*>(K + t * TLM_PST + c), qt = *reinterpret_cast<const f32x4*>(Q + t * TLM_PST + c);
            f32x4 d = *reinterpret_cast<const f32x4*>(G + t * TLM_PST + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) dP[0] = mmi_fma(qt[e], kt[e], dP[0]);
#pragma unroll
            for (int i = 1; i < TLM_SUB; ++i) {
                const f32x4 y = d * *reinterpret_cast<const f32x4*>(K + (t - i) * TLM_PST + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    dA[i] = mmi_fma(kt[e], y[e], dA[i]);
                    dP[i] = mmi_fma(qt[e], y[e], dP[i]);
                }
                if (i + 1 < TLM_SUB) d *= *reinterpret_cast<const f32x4*>(G + (t - i) * TLM_PST + c);
            }
        }
#pragma unroll
        for (int i = 0; i < TLM_SUB; ++i) {
            mmi_here(dA[i]);
            mmi_here(dP[i]);
        }
        mmi_meet();
        {                                                  // K -> k x (decay from the start of its 8), Q likewise, G -> k x (decay to the end)
            const int at = TLM_SUB * wave * TLM_PST + lane;
            float g[TLM_SUB], kk[TLM_SUB], qq[TLM_SUB], run = 1.f;
#pragma unroll
            for (int t = 0; t < TLM_SUB; ++t) {
                kk[t] = K[at + t * TLM_PST];
                qq[t] = Q[at + t * TLM_PST];
                g[t] = G[at + t * TLM_PST];
            }
#pragma unroll
            for (int t = 0; t < TLM_SUB; ++t) {
                run *= g[t];
                K[at + t * TLM_PST] = kk[t] * run;
                Q[at + t * TLM_PST] = qq[t] * run;
            }
            tot[wave * 64 + lane] = run;
            run = 1.f;
#pragma unroll
            for (int t = TLM_SUB - 1; t >= 0; --t) {
                G[at + t * TLM_PST] = kk[t] * run;
                run *= g[t];
            }
        }
        mmi_meet();
        {
            float fp = 1.f, fs = 1.f;                      // this wave's rows of pre and suf
#pragma unroll
            for (int m = 0; m < TLM_CHUNK / TLM_SUB; ++m) {
                const float v = tot[m * 64 + lane];
                fp *= m < wave ? v : 1.f;
                fs *= m > wave ? v : 1.f;
            }
            pre[wave * 64 + lane] = fp;
            suf[wave * 64 + lane] = fs;
            f32x4 mid[4];                                  // decay of the whole 8s between a row's token and a column's
#pragma unroll
            for (int j = 0; j < 4; ++j) mid[j] = f32x4{1.f, 1.f, 1.f, 1.f};
            if (wave < 6)
                for (int m = 2 * bj + 2; m < 2 * bi; ++m)
#pragma unroll
                    for (int j = 0; j < 4; ++j) mid[j] *= *reinterpret_cast<const f32x4*>(tot + m * 64 + 16 * j + 4 * kq);
#pragma unroll
            for (int j = 0; j < 4; ++j) {                  // (channels past the end: zeros)
                const int c = 16 * j + 4 * kq;
                f32x4 kt = *reinterpret_cast<const f32x4*>(K + row(bl) * TLM_PST + c), qt = *reinterpret_cast<const f32x4*>(Q + row(bl) * TLM_PST + c);
                f32x4 ks = *reinterpret_cast<const f32x4*>(G + column(bl) * TLM_PST + c);
                if (wave < 6) {
                    const f32x4 tt = *reinterpret_cast<const f32x4*>(tot + 2 * bi * 64 + c), ts = *reinterpret_cast<const f32x4*>(tot + (2 * bj + 1) * 64 + c);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float f = bl & 8 ? tt[e] : 1.f;
                        kt[e] *= f;
                        qt[e] *= f;
                        ks[e] *= bl & 8 ? 1.f : ts[e];
                    }
                    ks *= mid[j];
                }
                const u32x4 kb = __builtin_bit_cast(u32x4, ks);
                oA = TlmF32::mfma(kb, __builtin_bit_cast(u32x4, kt), oA);
                oP = TlmF32::mfma(kb, __builtin_bit_cast(u32x4, qt), oP);
            }
        }
        mmi_meet();
        if (lc < cn)
#pragma unroll
            for (int i = 0; i < 2; ++i) {                  // decayed queries
                const int t = lt + 32 * i;
                tlm_quad(Qg, (int)tlm_tile(t, c0 + lc, nd)) =
                    *reinterpret_cast<const f32x4*>(Q + t * TLM_PST + lc) * *reinterpret_cast<const f32x4*>(pre + t / TLM_SUB * 64 + lc);
            }
        if (mine && 16 * (wave & 3) < cn) {                // this wave's right sides of W
            const int c = 16 * (wave & 3) + bl;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float f = pre[(2 * i + (kq >> 1)) * 64 + c];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 16 * i + 4 * kq + r;
                    strip[i][r] = K[t * TLM_PST + c] * f * beta[t];
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {                      // transposed fragments: 16 channels x 16 tokens
            const int at = wave + 8 * i, c = 16 * (at >> 2) + bl, t = 16 * (at & 3) + 4 * kq;
            if (at >= cn / 4) continue;
            const float f = suf[t / TLM_SUB * 64 + c];
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = G[(t + e) * TLM_PST + c] * f;
            tlm_quad(Kt, (int)tlm_tile(c0 + c, t, 4)) = v;
        }
        if (tid < cn) a.gend[id * D + c0 + tid] = pre[(TLM_CHUNK / TLM_SUB - 1) * 64 + tid] * tot[(TLM_CHUNK / TLM_SUB - 1) * 64 + tid];
    };
#pragma unroll
    for (int k = 0; k < NS; ++k)
#pragma unroll
        for (int p = 0; p < min(2, NP); ++p)
            if (128 * k + 64 * p < D) panel(128 * k + 64 * p, wave >> 2 == p, x[k]);
    mmi_meet();
    // -A (strictly lower) and P, whole rows in LDS
    int l = lane;
    mmi_here(l);
    bl = l & 15;
    kq = l >> 4;
#pragma unroll
    for (int i = 0; i < TLM_SUB; ++i) {
        dA[i] = mmi_rows_sum(dA[i]);
        dP[i] = mmi_rows_sum(dP[i]);
    }
    f32x4 mine;                                            // lane (kq, bl): pairs t - 2 kq and t - 2 kq - 1
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        mine[i] = kq < 2 ? (kq ? dA[2 + i] : dA[i]) : (kq == 2 ? dA[4 + i] : dA[6 + i]);
        mine[2 + i] = kq < 2 ? (kq ? dP[2 + i] : dP[i]) : (kq == 2 ? dP[4 + i] : dP[6 + i]);
    }
    if (wave >= 4) *reinterpret_cast<f32x4*>(part + ((wave - 4) * 64 + lane) * 4) = mine;
    if (wave < 6 || (bl >> 3) == (kq >> 1)) {              // (a quarter's operands took rows of two blocks: the pairs inside one are wanted)
        const int t = row(bl), s = wave < 6 ? 16 * bj + 4 * kq : 32 * (wave - 6) + 16 * (kq >> 1) + 4 * (kq & 1);
        *reinterpret_cast<f32x4*>(A + t * TLM_PST + s) = oA * -beta[t];
        *reinterpret_cast<f32x4*>(Pl + t * TLM_PST + s) = oP;
    }
    mmi_meet();
    if (wave < 4) {
        mine += *reinterpret_cast<const f32x4*>(part + (wave * 64 + lane) * 4);
        const int t = 16 * wave + bl;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int s = t - 2 * kq - i;
            if (2 * kq + i > (t & 7)) continue;
            if (s < t) A[t * TLM_PST + s] = -beta[t] * mine[i];
            Pl[t * TLM_PST + s] = mine[2 + i];
        }
    }
    mmi_meet();
    if (wave < 4) {                                        // (I + A_ww)^-1, one column per lane
        float y[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float s = t == bl ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < t; j += 4) {
                const f32x4 r = *reinterpret_cast<const f32x4*>(A + (16 * wave + t) * TLM_PST + 16 * wave + j);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (j + e < t) s = mmi_fma(r[e], y[j + e], s);
            }
            y[t] = s;
        }
        if (kq == 0)
#pragma unroll
            for (int t = 0; t < 16; ++t) ti[(wave * 16 + t) * 20 + bl] = y[t];
    } else {
        for (int i = wave - 4; i < 10; i += 4) {           // P's blocks, those right of the diagonal left out
            const int ti_ = i < 1 ? 0 : (i < 3 ? 1 : (i < 6 ? 2 : 3)), si = i - ti_ * (ti_ + 1) / 2, t = 16 * ti_ + bl, s = 16 * si + 4 * kq;
            f32x4 v = *reinterpret_cast<const f32x4*>(Pl + t * TLM_PST + s);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = s + e <= t ? v[e] : 0.f;
            tlm_quad(P, (int)tlm_tile(t, s, 4)) = v;
        }
    }
    auto scale_u0 = [&](f32x4* u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = 16 * i + 4 * kq + r;
                u[i][r] = t < ck.n ? u[i][r] * beta[t] : 0.f;
            }
    };
    scale_u0(x[NS]);
    mmi_meet();
    // forward substitution by blocks of 16, all strips of this wave side by side
    mmi_here(l);
    bl = l & 15;
    kq = l >> 4;
    auto solve = [&](f32x4 (*y)[4], auto count) __attribute__((always_inline)) {
        constexpr int N = decltype(count)::value;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < i; ++j) {
                const u32x4 av = *reinterpret_cast<const u32x4*>(A + (16 * i + bl) * TLM_PST + 16 * j + 4 * kq);
#pragma unroll
                for (int k = 0; k < N; ++k) y[k][i] = TlmF32::mfma(av, __builtin_bit_cast(u32x4, y[k][j]), y[k][i]);
            }
            const u32x4 tv = *reinterpret_cast<const u32x4*>(ti + (i * 16 + bl) * 20 + 4 * kq);
#pragma unroll
            for (int k = 0; k < N; ++k) y[k][i] = TlmF32::mfma(tv, __builtin_bit_cast(u32x4, y[k][i]), f32x4{0.f, 0.f, 0.f, 0.f});
        }
    };
    auto store_u0 = [&](const f32x4* u, int v) __attribute__((always_inline)) {
        if (v < nv)
#pragma unroll
            for (int i = 0; i < 4; ++i) tlm_quad(Ug, ((i * nv + v) * 64 + lane) * 4) = u[i];
    };
    solve(x, std::integral_constant<int, NS + 1>{});
    store_u0(x[NS], v0);
    for (int v = v0 + 8; v < nv; v += 8) {                 // (more than 128 value columns)
        load_u0(x[NS], v, bl, kq);
        scale_u0(x[NS]);
        solve(x + NS, std::integral_constant<int, 1>{});
        store_u0(x[NS], v);
    }
    // W goes out as the walk's left operand: a strip's blocks turn round in LDS
    float* T = sh + wave * (TLM_CHUNK * 20);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        mmi_meet();
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) T[(16 * i + 4 * kq + r) * 20 + bl] = x[k][i][r];
        mmi_meet();
        const int st = 8 * k + wave;
        if (st < nd)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                tlm_quad(Wg, ((i * nd + st) * 64 + lane) * 4) = *reinterpret_cast<const f32x4*>(T + (16 * i + bl) * 20 + 4 * kq);
    }
}
// BESIDE: with the single tokens of n_small sequences, where those take workgroups of 512 too: neither fills the chip, and they share nothing.
// 11 chunks and 14 sequences, 16 heads of 128 x 128: 38.6 us in launches of their own, 26.0 together; 1 - 64 sequences beside 2 - 28 chunks of 16 and
// 32 heads gain as much or more, but 64 beside 16 chunks of 256 x 64 (one workgroup per CU by its registers) break even.  Chunks alone have a kernel without the
// other body: with it, scalar registers spill (896 chunks of 128 x 128 71.0 us, 68.0 without).
template <class Tr, int NP, bool BESIDE>
__global__ __launch_bounds__(512, NP <= 2 ? 4 : 2) void k_tlm_chunk_delta(TlmLinArgs a, int n_chunk, int n_small, int cgp) {
    MMI_DYN_SHARED(float, sh);
    const int b = (int)blockIdx.x, own = b - n_chunk * a.heads;
    if (!BESIDE || own < 0) tlm_chunk_delta<NP>(a, sh, b % n_chunk, b / n_chunk);
    else tlm_state_step<Tr, true, 8>(a, sh, cgp, own % n_small, own / n_small);
}

// ------------------------------------------------------------------------------------------------
// chunks: the walk over a sequence's chunks.  One workgroup per (sequence, head, 16 columns of S).  Wave w owns token block w of every chunk
// and a quarter of the rows of S, in the layout the matrix core leaves them in, which is also the layout it takes them as an operand; S and
// U go round through LDS.  A chunk is 112 matrix instructions of 32 cycles per SIMD and asks a CU for 116 KB: requests in one burst kept the
// waves from issuing for 2400 of 7500 cycles, so they stand between the products, a phase or more before their use, and what follows an exchange
// through LDS does not need it (Q S, P U).  One sequence of 1773 tokens, 32 heads of 128 x 128: 107 us in a step
// before, 78 now (5200 cycles per chunk; with all of it in the L2 no less: what is left is the distance of dependent instructions in one wave
// per SIMD); two of 331 and 294 tokens, 16 heads: 24.2 and 19.8.
// grid: 8 x ceil(sequences x heads / 8) x vdim_p / 16, the column blocks of one head on one XCD (they read the same W, Qg, Kt, P)
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ float tlm_f(unsigned v) { return __builtin_bit_cast(float, v); }
template <bool DELTA, int NDW>
__global__ __launch_bounds__(256, NDW <= 2 ? 2 : 1) void k_tlm_chunk_scan(TlmLinArgs a, int n_units) {
    constexpr int ND = 4 * NDW;                            // 16-row blocks of S; past the model's: zeros
    MMI_SHARED __attribute__((aligned(16))) f32x4 Sl[ND][64], Ul[4][64];
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15, kq = lane >> 4;
    const int ncb = a.vdim_p / 16, j0 = (int)blockIdx.x >> 3;
    const int uh = ((int)blockIdx.x & 7) + 8 * (j0 / ncb), cb = j0 % ncb;
    if (uh >= n_units * a.heads) return;
    const TlmUnit un = a.unit[uh / a.heads];
    const int h = uh % a.heads, D = a.dim_p, V = a.vdim_p, nd = D / 16;
    float* S = a.state + ((long)un.slot * a.heads + h) * D * V + 16 * cb;
    // a chunk's operands in registers: keys, P and decays are asked for while W S is computed, queries again as they are used up, W and U0 of
    // the next chunk while S is brought up to date
    u32x4 w[DELTA ? ND : 1], q[ND], k[NDW][4], p[4];
    f32x4 u0, g[NDW], s[NDW], sl[ND], u[4];
    // (blocks past the end: a valid address, against rows of S that stay zero)
    auto load_w = [&](long id, int d) __attribute__((always_inline)) { w[d] = tlm_quad<u32x4>(a.w + id * TLM_CHUNK * D, ((wave * nd + min(d, nd - 1)) * 64 + lane) * 4); };
    auto load_q = [&](long id, int d) __attribute__((always_inline)) { q[d] = tlm_quad<u32x4>(a.qg + id * TLM_CHUNK * D, ((wave * nd + min(d, nd - 1)) * 64 + lane) * 4); };
    auto load_k = [&](long id, int i, int t) __attribute__((always_inline)) { k[i][t] = tlm_quad<u32x4>(a.kt + id * TLM_CHUNK * D, ((min(wave * NDW + i, nd - 1) * 4 + t) * 64 + lane) * 4); };
    auto load_g = [&](long id, int i) __attribute__((always_inline)) { g[i] = tlm_quad(a.gend + id * D, 16 * min(wave * NDW + i, nd - 1) + 4 * kq); };
    auto load_p = [&](long id, int t) __attribute__((always_inline)) { p[t] = tlm_quad<u32x4>(a.p + id * (TLM_CHUNK * TLM_CHUNK), ((wave * 4 + min(t, wave)) * 64 + lane) * 4); };
    auto load_u = [&](long id, int c) __attribute__((always_inline)) {
        if constexpr (DELTA) {
            u0 = tlm_quad(a.u0 + id * TLM_CHUNK * V, ((wave * ncb + cb) * 64 + lane) * 4);
        } else {
            const int n = min(TLM_CHUNK, un.n - c * TLM_CHUNK);
            const float* v = a.in + (long)(un.row0 + c * TLM_CHUNK) * a.in_ld + a.v0 + h * V + 16 * cb;
#pragma unroll
            for (int r = 0; r < 4; ++r) u0[r] = tlm_quad<float>(v, min(16 * wave + 4 * kq + r, n - 1) * a.in_ld + bl);
        }
    };
    {
        const long id = (long)un.chunk0 * a.heads + h;
        load_u(id, 0);
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            if constexpr (DELTA) load_w(id, d);
            load_q(id, d);
        }
    }
#pragma unroll
    for (int i = 0; i < NDW; ++i) {
        s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int d = wave * NDW + i;
        if (!un.fresh && d < nd)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[i][r] = tlm_quad<float>(S, (16 * d + 4 * kq + r) * V + bl);
        Sl[d][lane] = s[i];
    }
    mmi_meet();
#pragma unroll
    for (int d = 0; d < ND; ++d) sl[d] = Sl[d][lane];
    for (int c = 0; c < un.n_chunks; ++c) {
        const int n = min(TLM_CHUNK, un.n - c * TLM_CHUNK), cn = min(c + 1, un.n_chunks - 1);      // (the last chunk asks for itself again)
        const long id = (long)(un.chunk0 + c) * a.heads + h, next = (long)(un.chunk0 + cn) * a.heads + h;
        // two independent sums, steps in turn: a matrix instruction never waits for the one before it
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        f32x4 x0 = zero, x1 = zero, o0 = zero, o1 = zero;
        auto outputs = [&](int d) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o0 = mmi_mfma_f32_16x16x4(tlm_f(q[d][e]), sl[d][e], o0);
                o1 = mmi_mfma_f32_16x16x4(tlm_f(q[d + 1][e]), sl[d + 1][e], o1);
            }
            mmi_sched_barrier();
            load_q(next, d);
            load_q(next, d + 1);
            mmi_sched_barrier();
        };
        auto rest = [&](int d) __attribute__((always_inline)) {
            load_k(id, d / 4, d % 4);
            if (d % 4 == 0) load_g(id, d / 4);
            if (d < 4) load_p(id, d);
        };
        if constexpr (DELTA) {
#pragma unroll
            for (int d = 0; d < ND; d += 2) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x0 = mmi_mfma_f32_16x16x4(tlm_f(w[d][e]), sl[d][e], x0);
                    x1 = mmi_mfma_f32_16x16x4(tlm_f(w[d + 1][e]), sl[d + 1][e], x1);
                }
                mmi_sched_barrier();
                rest(d);
                rest(d + 1);
                mmi_sched_barrier();
            }
            Ul[wave][lane] = u0 - (x0 + x1);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) u0[r] = 16 * wave + 4 * kq + r < n ? u0[r] : 0.f;
            Ul[wave][lane] = u0;
#pragma unroll
            for (int d = 0; d < ND; ++d) rest(d);
            mmi_sched_barrier();
        }
        // the exchange of U stands between the halves of Q S, that of S between those of P U: what a wave waits for is on its way meanwhile
#pragma unroll
        for (int d = 0; d < ND / 2; d += 2) outputs(d);
        mmi_meet();
#pragma unroll
        for (int t = 0; t < 4; ++t) u[t] = Ul[t][lane];
        mmi_sched_barrier();
#pragma unroll
        for (int d = ND / 2; d < ND; d += 2) outputs(d);
        f32x4 sh[NDW];
#pragma unroll
        for (int i = 0; i < NDW; ++i) {
            s[i] *= g[i];
            sh[i] = zero;
        }
#pragma unroll
        for (int t = 0; t < 4; t += 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < NDW; ++i) {
                    s[i] = mmi_mfma_f32_16x16x4(tlm_f(k[i][t][e]), u[t][e], s[i]);
                    sh[i] = mmi_mfma_f32_16x16x4(tlm_f(k[i][t + 1][e]), u[t + 1][e], sh[i]);
                }
            mmi_sched_barrier();
            if constexpr (DELTA)
#pragma unroll
                for (int d = t * NDW; d < (t + 2) * NDW; ++d) load_w(next, d);
            if (t) load_u(next, cn);
            mmi_sched_barrier();
        }
#pragma unroll
        for (int i = 0; i < NDW; ++i) {
            s[i] += sh[i];
            if (wave * NDW + i >= nd) s[i] = zero;
            Sl[wave * NDW + i][lane] = s[i];
        }
        auto inside = [&](int t) __attribute__((always_inline)) {      // (blocks right of the diagonal: zeros instead)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                o0 = mmi_mfma_f32_16x16x4(t <= wave ? tlm_f(p[t][e]) : 0.f, u[t][e], o0);
                o1 = mmi_mfma_f32_16x16x4(t + 1 <= wave ? tlm_f(p[t + 1][e]) : 0.f, u[t + 1][e], o1);
            }
            mmi_sched_barrier();
        };
        inside(0);
        mmi_meet();
#pragma unroll
        for (int d = 0; d < ND; ++d) sl[d] = Sl[d][lane];
        mmi_sched_barrier();
        inside(2);
        const f32x4 o = o0 + o1;
        float* out = a.o + ((long)(un.row0 + c * TLM_CHUNK) * a.heads + h) * V + 16 * cb;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tok = 16 * wave + 4 * kq + r;
            if (tok < n) tlm_quad<float>(out, tok * a.heads * V + bl) = o[r];
        }
    }
#pragma unroll
    for (int i = 0; i < NDW; ++i) {
        const int d = wave * NDW + i;
        if (d < nd)
#pragma unroll
            for (int r = 0; r < 4; ++r) tlm_quad<float>(S, (16 * d + 4 * kq + r) * V + bl) = s[i][r];
    }
}

// ------------------------------------------------------------------------------------------------
// RMS norm of a head's output (`per_head`) or of all heads' together, weight, gate -> packed operand; one workgroup per row: of the whole
// step, or (`chunk`) 64 per chunk
// ------------------------------------------------------------------------------------------------
template <class Tr>
__global__ __launch_bounds__(256) void k_tlm_gated_norm(TlmLinArgs a, int per_head, const TlmSeg* chunk) {
    MMI_DYN_SHARED(float, inv);                            // [heads], then [4]
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6, V = a.vdim_p, ld = a.heads * V;
    const int b = tlm_row_block((int)blockIdx.x, (int)gridDim.x);
    long row = b;
    if (chunk) {
        const TlmSeg ck = chunk[b >> 6];
        if ((b & 63) >= ck.n) return;
        row = ck.row0 + (b & 63);
    }
    const float* o = a.o + row * ld;
    if (per_head) {
        for (int h = wave; h < a.heads; h += 4) {
            float s = 0.f;
            for (int c = lane; c < V; c += 64) s = mmi_fma(o[h * V + c], o[h * V + c], s);
            s = tlm_wave_sum(s);
            if (lane == 0) inv[h] = 1.0f / sqrtf(s / (float)a.vdim + a.eps);
        }
    } else {
        float s = 0.f;
        for (int c = 4 * tid; c < ld; c += 1024) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(o + c);
            s += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        s = tlm_wave_sum(s);
        float* part = inv + a.heads;
        if (lane == 0) part[wave] = s;
        __syncthreads();
        s = 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)(a.heads * a.vdim) + a.eps);
        for (int h = tid; h < a.heads; h += 256) inv[h] = s;
    }
    __syncthreads();
    for (int c = 4 * tid; c < ld; c += 1024) {
        const int h = c / V;
        const f32x4 w = *reinterpret_cast<const f32x4*>(a.nw + (per_head ? c - h * V : c));
        f32x4 g = *reinterpret_cast<const f32x4*>(a.gate + row * a.gate_ld + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) g[e] = tlm_sigmoid(g[e]);
        Tr::store4((typename Tr::elem*)a.out + tlm_index<Tr>(row, c, a.out_ks), *reinterpret_cast<const f32x4*>(o + c) * inv[h] * w * g);
    }
}
