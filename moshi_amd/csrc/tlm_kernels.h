// Kernels of the token language models (tlm_engine.hip): decoder-only networks over token ids whose layers are described by data
// (mmi_tlm_cfg), served from a paged cache and per-sequence recurrent state, any mixture of prompt portions and single tokens per step.
//
// Every kernel is written once for two number formats: TlmBf16 (bf16 operands on v_mfma_f32_16x16x32_bf16, fp32 accumulation) and
// TlmF32 (fp32 operands on v_mfma_f32_16x16x4_f32, an exact fma chain).  Positions, angles, attention scores and weights, norms, the
// residual stream, gates and recurrent state are fp32 in both.
//
// Data layout in HBM
//   fragment     64 lanes x 16 bytes: 16 rows x KSTEP reduction indices (bf16: 32, fp32: 16); lane (i, kq) = 16 kq + i holds row i,
//                k = V kq .. V kq + V - 1 (V = 8 bf16 / 4 fp32).  It is the A operand (row = output feature), the B operand (row = token)
//                and, at fp32, four 16x16x4 steps at once: element e of every lane is one step (any k order serves, both operands use it).
//   weights      Wp[n-tile][k-step][lane][V]            (16-row tiles, zero padded; the layout of the Moshi LM's 16-row tile)
//   activations  Xp[row / 16][k-step][lane][V]          (tlm_index; written by the producing epilogue)
//   key cache    the same matrix with row = 64 page + offset: k = latent, then the rotated key part
//                There is no second copy for the values (the value IS the latent): the transposed operand of the value product comes out
//                of the matrix core, K x identity (TlmFlip) - lane (d, kq) of its accumulators holds keys 4 kq .. 4 kq + 3, exactly the
//                keys whose scores the same lane holds after S = K Q^T, so the softmax weights become an operand without leaving the lane.
//   residual     x[token][ld] fp32
#pragma once
#include "mmi_common.h"

struct TlmBf16 {
    typedef uint16_t elem;
    static constexpr int V = 8, KSTEP = 32;
    static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) { return mmi_mfma_bf16_16x16x32(a, b, c); }
    static __device__ __forceinline__ uint16_t cvt(float v) { return mmi_f32_to_bf16(v); }
    static __device__ __forceinline__ void store4(uint16_t* p, f32x4 v) {
        u32x2 o = {mmi_pack_bf16x2(v[0], v[1]), mmi_pack_bf16x2(v[2], v[3])};
        *reinterpret_cast<u32x2*>(p) = o;
    }
    static __device__ __forceinline__ void store2(uint16_t* p, float a, float b) { *reinterpret_cast<uint32_t*>(p) = mmi_pack_bf16x2(a, b); }
};
struct TlmF32 {
    typedef float elem;
    static constexpr int V = 4, KSTEP = 16;
    static __device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int e = 0; e < 4; ++e) c = mmi_mfma_f32_16x16x4(fa[e], fb[e], c);
        return c;
    }
    static __device__ __forceinline__ float cvt(float v) { return v; }
    static __device__ __forceinline__ void store4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
    static __device__ __forceinline__ void store2(float* p, float a, float b) { *reinterpret_cast<f32x2*>(p) = f32x2{a, b}; }
};

// element (row, k) of a fragment-packed matrix with `ks` k-steps per row tile
template <class Tr>
MMI_HD long tlm_index(long row, int k, int ks) {
    return (((row >> 4) * ks + k / Tr::KSTEP) * 64 + ((k % Tr::KSTEP) / Tr::V) * 16 + (row & 15)) * Tr::V + k % Tr::V;
}

constexpr int TLM_PAGE = 64;         // tokens per cache page

// 1 / (1 + e^-x) in about half the instructions of expf and a division, as good as theirs (largest error of 20 million 2.6 ulp): 2^-(x log2 e) with the
// product's low part carried along, the reciprocal with one Newton step.  Of e^-x = e 2^n the sum is formed as 2^-n + e where n > 0, so that the
// reciprocal is a normal number (the instruction would flush another one) and results below 2^-126 are rounded like the others.  0 and 1 at
// the infinities, NaN where x is
__device__ __forceinline__ float tlm_sigmoid(float x) {
    constexpr float L = 1.44269504f, LL = 1.92596299e-8f;      // log2 e in two parts
    x = x > 104.f ? 104.f : x;
    x = x < -104.f ? -104.f : x;
    const float nf = rintf(-L * x);
    const int n = (int)nf, m = max(n, 0);
    const float e = mmi_fast_exp2f(mmi_fma(-LL, x, mmi_fma(-L, x, -nf)));
    const float s = ldexpf(1.0f, -m) + ldexpf(e, n - m);
    const float y = mmi_fast_rcpf(s);
    return ldexpf(mmi_fma(y, mmi_fma(-s, y, 1.0f), y), -m);
}
__device__ __forceinline__ float tlm_wave_sum(float x) {
    x = mmi_group_sum<16>(x);
    x += mmi_shfl_xor(x, 16);
    x += mmi_shfl_xor(x, 32);
    return x;
}

// ------------------------------------------------------------------------------------------------
// weight import: bf16 checkpoint tensor -> fragments, through a row and a column map (-1 = zero padding).  Source element
// (row r, column c) is src[r * sr + c * sc], so a transposed operand is the same call with the strides exchanged.
// ------------------------------------------------------------------------------------------------
template <class Tr>
__global__ void k_tlm_pack(const uint16_t* __restrict__ src, long sr, long sc, const int* __restrict__ rowmap, const int* __restrict__ colmap,
                           typename Tr::elem* __restrict__ dst, int NT, int KS, int tmul, int toff, int keep) {
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)NT * KS * 64 * Tr::V) return;
    const int e = (int)(idx % Tr::V);
    const long f = idx / Tr::V;
    const int lane = (int)(f & 63);
    const int ks = (int)((f >> 6) % KS), nt = (int)((f >> 6) / KS);
    const int r = rowmap[nt * 16 + (lane & 15)];
    if (r < 0 && keep) return;                     // (rows another call has filled)
    const int c = colmap[ks * Tr::KSTEP + (lane >> 4) * Tr::V + e];
    const uint16_t h = (r < 0 || c < 0) ? (uint16_t)0 : src[(long)r * sr + (long)c * sc];
    const long at = (((long)nt * tmul + toff) * KS + ks) * 64 * Tr::V + (long)lane * Tr::V + e;      // tile nt of this call is tile nt * tmul + toff of the matrix
    if constexpr (Tr::V == 8) dst[at] = h;
    else dst[at] = mmi_bf16_to_f32(h);
}
// bf16 vector -> fp32, gathered through a map, zero where the map is negative
__global__ void k_tlm_vec(const uint16_t* __restrict__ src, const int* __restrict__ map, float* __restrict__ dst, int n) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) dst[i] = map[i] < 0 ? 0.f : mmi_bf16_to_f32(src[map[i]]);
}

// ------------------------------------------------------------------------------------------------
// step preparation
// ------------------------------------------------------------------------------------------------
struct TlmRope { const float* freq; int half, ld; float* out; };      // out [row][ld][2]: (cos, sin), (1, 0) past `half`
struct TlmPrepArgs {
    int T, n_ropes;
    const int* n_updates;
    const int* htok;          // token per row; negative: the token last sampled for the row's slot
    const int* pos;
    const int* rslot;
    const int* last_tok;      // [slots]
    int* tok;
    const int* updates;       // (block-table index, page) pairs
    int* block_table;
    const TlmRope* rope;
    int buckets; long mul_prev, mul_cur;       // bigram embedding (buckets 0: none)
    const int* prev;          // per row: -1 first token of its sequence, -2 the row before it, otherwise the index of the token in prev_tok
    const int* next;          // per row: where in prev_tok its token goes (the last of an entry), or -1
    int* prev_tok;            // [slots][2]: a step reads one copy and writes the other
    int* brow;                // out: row of the bigram table
};
__global__ void k_tlm_prepare(TlmPrepArgs a) {
    const int i0 = (int)(blockIdx.x * blockDim.x + threadIdx.x), n = (int)(gridDim.x * blockDim.x);
    for (int i = i0; i < *a.n_updates; i += n) a.block_table[a.updates[2 * i]] = a.updates[2 * i + 1];
    for (int i = i0; i < a.T; i += n) {
        const int t = a.htok[i] >= 0 ? a.htok[i] : a.last_tok[a.rslot[i]];
        a.tok[i] = t;
        if (a.buckets > 0) {
            const int w = a.prev[i];
            int b = a.buckets;
            if (w != -1) {
                const int p = w >= 0 ? a.prev_tok[w] : (a.htok[i - 1] >= 0 ? a.htok[i - 1] : a.last_tok[a.rslot[i]]);
                b = (int)(((long)p * a.mul_prev + (long)t * a.mul_cur) % a.buckets);
                if (b < 0) b += a.buckets;
            }
            a.brow[i] = b;
            if (a.next[i] >= 0) a.prev_tok[a.next[i]] = t;
        }
    }
    for (int r = 0; r < a.n_ropes; ++r) {
        const TlmRope q = a.rope[r];
        for (long i = i0; i < (long)a.T * q.ld; i += n) {
            const int row = (int)(i / q.ld), j = (int)(i % q.ld);
            float c = 1.f, s = 0.f;
            if (j < q.half) {
                const float ang = (float)a.pos[row] * q.freq[j];
                c = cosf(ang);
                s = sinf(ang);
            }
            q.out[2 * i] = c;
            q.out[2 * i + 1] = s;
        }
    }
}

// Token-table routing: the experts of a row are table[token][0 .. top).  One workgroup per routed layer sorts the step's
// (row, choice) pairs by expert - the order inside an expert is irrelevant, every pair is computed and stored on its own - and cuts
// each expert's run into tiles of `tile` pairs.
struct TlmRouteLayer { const int* table; int experts, top; };
struct TlmRouteArgs {
    const TlmRouteLayer* layers;
    const int* tok;
    int T, tile;
    int* list;                // [layer][list_ld] pair ids row * top + choice, by expert
    long list_ld;
    int* tiles;               // [layer][tile_ld][3]: expert, first pair, pairs
    long tile_ld;
    int* n_tiles;             // [layer]
};
__global__ __launch_bounds__(1024) void k_tlm_route(TlmRouteArgs a) {
    MMI_DYN_SHARED(unsigned, cnt);                       // [experts] pair counts, then [experts] insertion points
    const TlmRouteLayer L = a.layers[blockIdx.x];
    const int E = L.experts, top = L.top, tid = (int)threadIdx.x, nthr = (int)blockDim.x;
    unsigned* at = cnt + E;
    for (int e = tid; e < E; e += nthr) cnt[e] = 0u;
    __syncthreads();
    const int n = a.T * top;
    for (int i = tid; i < n; i += nthr) mmi_atomic_add(&cnt[L.table[(long)a.tok[i / top] * top + i % top]], 1u);
    __syncthreads();
    if (tid == 0) {
        unsigned s = 0;
        int nt = 0;
        int* tl = a.tiles + (long)blockIdx.x * a.tile_ld * 3;
        for (int e = 0; e < E; ++e) {
            const int c = (int)cnt[e];
            at[e] = s;
            for (int o = 0; o < c; o += a.tile) {
                tl[3 * nt] = e;
                tl[3 * nt + 1] = (int)s + o;
                tl[3 * nt + 2] = c - o < a.tile ? c - o : a.tile;
                ++nt;
            }
            s += (unsigned)c;
        }
        a.n_tiles[blockIdx.x] = nt;
    }
    __syncthreads();
    int* list = a.list + (long)blockIdx.x * a.list_ld;
    for (int i = tid; i < n; i += nthr) list[mmi_atomic_add(&at[L.table[(long)a.tok[i / top] * top + i % top]], 1u)] = i;
}

// Row of a workgroup in the kernels that write a packed operand row by row: 16 rows in a row to one XCD.  A fragment interleaves 16 rows in
// pieces of 16 bytes, so a cache line is written by 8 workgroups; consecutive ones go round the XCDs, whose L2s would each send an
// eighth of the line to memory.  (the rows past the last multiple of 128 as they come: too few to go round)
// 1773 rows: residual and norm of width 4096 48.7 -> 38.0 us, gated norm 30.3 -> 25.1; 2048 rows of 1792 columns' latent part 11.4 -> 8.5
__device__ __forceinline__ int tlm_row_block(int b, int n) {
    if (b >= (n & ~127)) return b;
    const int i = b >> 3;
    return ((i >> 4) * 8 + (b & 7)) * 16 + (i & 15);
}

// n / d for what a launch knows: m = 2^32 / d + 1 makes it one multiplication (exact while n d < 2^32, else 0)
struct TlmDiv { int d; unsigned m; };
inline TlmDiv tlm_divisor(int d, long n_max) { return TlmDiv{d, d > 1 && n_max * d < (1L << 32) ? (unsigned)((1L << 32) / d + 1) : 0u}; }
__device__ __forceinline__ int tlm_div(int n, TlmDiv v) {
    if (v.m) return (int)(((unsigned long)(unsigned)n * v.m) >> 32);
    return v.d == 1 ? n : n / v.d;
}

// ------------------------------------------------------------------------------------------------
// residual update + grouped RMS norm: one workgroup per row
//   x <- x + ls1 * sum_p mix[p] + ls2 * (1 / top) * sum_choice sum_p dn[p]   (the split-K partials of the two sublayers' last products;
//        no ls: factor 1), or x <- sum_p mix[p] (`replace`: the product at the start of a repeated pass)
//   x <- emb[token] (first layer) or x + emb[token] (start of a repeated pass); x <- x + vec; then h = norm(x) * w -> packed operand, and
//   a second one with weights of its own; `raw`: x itself as a packed operand
//   emb[token] = table[token] * scale + bigram[row of (previous, token)] + pos[position]
// ------------------------------------------------------------------------------------------------
enum { TLM_EMB_NONE = 0, TLM_EMB_SET = 1, TLM_EMB_ADD = 2 };
struct TlmEmbArgs {
    const uint16_t* table; const int* tok; float scale;
    const uint16_t* bigram; const int* brow;       // or null
    const uint16_t* pos; const int* at;            // or null
};
struct TlmResidArgs {
    float* x;
    int width, ld;                       // ld: row stride of x, mix, dn (width rounded up to 16)
    const float* mix; int mix_p; long mix_ps; const float* ls1; int replace;
    const float* dn; int dn_p; long dn_ps; int top; const float* ls2;
    TlmEmbArgs emb; int emb_mode;
    const float* vec;
    float* tap;                          // copy of the residual stream before the embedding is added again, or null
    const float* w; int groups; float eps;
    TlmDiv by_group;                     // by width / groups
    void* out; int KS;                   // packed; null: no norm
    const float* w2; void* out2;
    void* rows_out; int rows_ld;         // what experts gather (by w2 if there is one), row-major, or null
    void* raw; int raw_ks;               // packed x, or null
    void* emb_out; int emb_k0;           // TLM_EMB_SET: packed copy of the embedding from column emb_k0 of rows of raw_ks k-steps, or null
    const int* rows;                     // row list (the residual is then not written back), or null
};
// V: vectors of 4 columns per thread, all of them in registers (4 V blockDim >= ld).  A few rows are a chain: what a row reads, the sum over the
// workgroup, what it writes.  So a thread asks for everything at once (V == 1; up to 8 partial sums of each product, those past the last one again, not
// added), and where groups are whole waves' vectors (256 columns) the sums need no copy of the row and one meeting.  Before - the partial sums
// one after the other behind the row, weights cold behind the sums, divisions by the group's width - a row of 2048 took 5.6 us, here 4.4.
// us per launch before / here: 64 rows of 4096 8.6 / 6.4, 2048 of 2048 26.1 / 19.8, 1773 of 4096 38.8 / 33.1 (their bytes: 3.4 TB/s before).
template <class Tr, int V>
__global__ __launch_bounds__(1024) void k_tlm_resid_norm(TlmResidArgs a) {
    MMI_DYN_SHARED(float, sh);           // one partial sum per wave and vector; other groups: [ld] the row, [groups * parts] partial sums, [groups] 1 / rms
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = mmi_uniform(tid >> 6), nthr = (int)blockDim.x, nw = nthr >> 6;
    const int o = tlm_row_block((int)blockIdx.x, (int)gridDim.x), r = a.rows ? a.rows[o] : o;
    float* x = a.x + (long)r * a.ld;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f}, ones = {1.f, 1.f, 1.f, 1.f};
    int k[V];                            // first column; past the row: its last vector again, not stored
    bool mine[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int at = 4 * (tid + i * nthr);
        mine[i] = at < a.ld;
        k[i] = min(at, a.ld - 4);
    }
    f32x4 v[V], d[V], f[V], ev[V], w, w2, l1 = ones, l2 = ones;
#pragma unroll
    for (int i = 0; i < V; ++i) v[i] = d[i] = f[i] = ev[i] = zero;
    const bool update = a.emb_mode != TLM_EMB_SET;
    if (update && !a.replace)
#pragma unroll
        for (int i = 0; i < V; ++i) v[i] = *reinterpret_cast<const f32x4*>(x + k[i]);
    auto mix = [&](int p, int i) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(a.mix + p * a.mix_ps + (long)r * a.ld + k[i]); };
    const int dn_n = a.dn ? a.top * a.dn_p : 0, mix_n = a.mix ? a.mix_p : 0;
    int dc = 0, dp = 0;                  // choice and partial sum that comes next
    auto dn = [&](int i) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(a.dn + dp * a.dn_ps + ((long)r * a.top + dc) * a.ld + k[i]); };
    auto next = [&]() __attribute__((always_inline)) {
        if (++dp == a.dn_p) {
            dp = 0;
            ++dc;
        }
    };
    if constexpr (V == 1) {
        f32x4 m4[8], d4[8];
#pragma unroll
        for (int h = 0; h < 8; h += 4) {
            if (update && mix_n > h)
#pragma unroll
                for (int p = h; p < h + 4; ++p) m4[p] = mix(min(p, mix_n - 1), 0);
            if (update && dn_n > h)
#pragma unroll
                for (int p = h; p < h + 4; ++p) {
                    d4[p] = dn(0);
                    if (p + 1 < dn_n) next();
                }
        }
        if (update && a.ls1) l1 = *reinterpret_cast<const f32x4*>(a.ls1 + k[0]);
        if (update && a.ls2) l2 = *reinterpret_cast<const f32x4*>(a.ls2 + k[0]);
        if (a.out) {
            w = *reinterpret_cast<const f32x4*>(a.w + k[0]);
            w2 = a.w2 ? *reinterpret_cast<const f32x4*>(a.w2 + k[0]) : w;
        }
        if (update) {
#pragma unroll
            for (int p = 0; p < 8; ++p)
                if (p < mix_n) d[0] += m4[p];
#pragma unroll
            for (int p = 0; p < 8; ++p)
                if (p < dn_n) f[0] += d4[p];
#pragma unroll 1
            for (int p0 = 8; p0 < mix_n; p0 += 4) {
                f32x4 t[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) t[p] = mix(min(p0 + p, mix_n - 1), 0);
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    if (p0 + p < mix_n) d[0] += t[p];
            }
#pragma unroll 1
            for (int p0 = 8; p0 < dn_n; p0 += 4) {
                f32x4 t[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    t[p] = dn(0);
                    if (p0 + p + 1 < dn_n) next();
                }
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    if (p0 + p < dn_n) f[0] += t[p];
            }
        }
    } else if (update) {
        int p = 0;
        for (; p + 2 <= mix_n; p += 2) {
            f32x4 t[2][V];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < V; ++i) t[q][i] = mix(p + q, i);
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < V; ++i) d[i] += t[q][i];
        }
        if (p < mix_n)
#pragma unroll
            for (int i = 0; i < V; ++i) d[i] += mix(p, i);
        p = 0;
        for (; p + 2 <= dn_n; p += 2) {
            f32x4 t[2][V];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
#pragma unroll
                for (int i = 0; i < V; ++i) t[q][i] = dn(i);
                next();
            }
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int i = 0; i < V; ++i) f[i] += t[q][i];
        }
        if (p < dn_n)
#pragma unroll
            for (int i = 0; i < V; ++i) f[i] += dn(i);
    }
    if (a.emb_mode != TLM_EMB_NONE) {
        const TlmEmbArgs& E = a.emb;
        const uint16_t* e = E.table + (long)E.tok[r] * a.width;
        const uint16_t* eb = E.bigram ? E.bigram + (long)E.brow[r] * a.width : nullptr;
        const uint16_t* ep = E.pos ? E.pos + (long)E.at[r] * a.width : nullptr;
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (k[i] + q < a.width) {
                    ev[i][q] = mmi_bf16_to_f32(e[k[i] + q]) * E.scale;
                    if (eb) ev[i][q] += mmi_bf16_to_f32(eb[k[i] + q]);
                    if (ep) ev[i][q] += mmi_bf16_to_f32(ep[k[i] + q]);
                }
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
        if (!update) {
            v[i] = ev[i];
            if (a.emb_out && mine[i]) Tr::store4((typename Tr::elem*)a.emb_out + tlm_index<Tr>(o, a.emb_k0 + k[i], a.raw_ks), ev[i]);
        } else {
            if (V > 1 && a.ls1) l1 = *reinterpret_cast<const f32x4*>(a.ls1 + k[i]);
            if (a.mix && a.ls1) d[i] *= l1;
            if (a.dn) {
                f[i] *= 1.0f / (float)a.top;
                if (V > 1 && a.ls2) l2 = *reinterpret_cast<const f32x4*>(a.ls2 + k[i]);
                d[i] += a.ls2 ? f[i] * l2 : f[i];
            }
            v[i] += d[i];
            if (a.tap && mine[i]) *reinterpret_cast<f32x4*>(a.tap + (long)r * a.ld + k[i]) = v[i];
            if (a.emb_mode == TLM_EMB_ADD) v[i] += ev[i];
        }
        if (a.vec) v[i] += *reinterpret_cast<const f32x4*>(a.vec + k[i]);
        if (!mine[i]) continue;
        if (a.raw) Tr::store4((typename Tr::elem*)a.raw + tlm_index<Tr>(o, k[i], a.raw_ks), v[i]);
        if (!a.rows) *reinterpret_cast<f32x4*>(x + k[i]) = v[i];
    }
    if (!a.out) return;                                       // uniform over the grid
    const int gs = a.by_group.d;
    float inv[V][4];
    if (a.groups == 1 || gs % 256 == 0) {                     // a wave's vector lies in one group
        float ss[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
            ss[i] = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (mine[i] && k[i] + q < a.width) ss[i] = mmi_fma(v[i][q], v[i][q], ss[i]);
            if (a.groups > 1) {
                ss[i] = tlm_wave_sum(ss[i]);
                if (lane == 0) sh[wave + i * nw] = ss[i];
            } else if (i) {
                ss[0] += ss[i];
            }
        }
        if (a.groups == 1) {
            ss[0] = tlm_wave_sum(ss[0]);
            if (lane == 0) sh[wave] = ss[0];
        }
        __syncthreads();
        const int n = a.groups == 1 ? nw : gs / 256;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            if (i && a.groups == 1) {
                inv[i][0] = inv[0][0];
            } else {
                const float* part = sh + (a.groups == 1 ? 0 : tlm_div(mmi_uniform(min(256 * (wave + i * nw), a.width - 1)), a.by_group) * n);
                float t = 0.f;
                for (int p = 0; p < n; ++p) t += part[p];
                inv[i][0] = 1.0f / sqrtf(t / (float)gs + a.eps);
            }
#pragma unroll
            for (int q = 1; q < 4; ++q) inv[i][q] = inv[i][0];
        }
    } else {
        const int parts = a.groups < nw ? nw / a.groups : 1;        // waves per group
        float *row = sh, *part = row + a.ld, *rms = part + a.groups * parts;
#pragma unroll
        for (int i = 0; i < V; ++i)
            if (mine[i]) *reinterpret_cast<f32x4*>(row + k[i]) = v[i];
        __syncthreads();
        const int per = (gs + parts - 1) / parts;
        for (int t = wave; t < a.groups * parts; t += nw) {
            const int g = t / parts, p = t - g * parts;
            const int lo = p * per, hi = lo + per < gs ? lo + per : gs;
            float s = 0.f;
            for (int c = lo + lane; c < hi; c += 64) s = mmi_fma(row[g * gs + c], row[g * gs + c], s);
            s = tlm_wave_sum(s);
            if (lane == 0) part[t] = s;
        }
        __syncthreads();
        for (int g = tid; g < a.groups; g += nthr) {
            float s = 0.f;
            for (int p = 0; p < parts; ++p) s += part[g * parts + p];
            rms[g] = 1.0f / sqrtf(s / (float)gs + a.eps);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) inv[i][q] = rms[min(tlm_div(k[i] + q, a.by_group), a.groups - 1)];
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
        if (!mine[i]) continue;
        if constexpr (V > 1) {
            w = *reinterpret_cast<const f32x4*>(a.w + k[i]);
            w2 = a.w2 ? *reinterpret_cast<const f32x4*>(a.w2 + k[i]) : w;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) v[i][q] = k[i] + q < a.width ? v[i][q] * inv[i][q] : 0.f;
        Tr::store4((typename Tr::elem*)a.out + tlm_index<Tr>(o, k[i], a.KS), v[i] * w);
        if (a.rows_out) Tr::store4((typename Tr::elem*)a.rows_out + (long)o * a.rows_ld + k[i], v[i] * w2);
        if (a.out2) Tr::store4((typename Tr::elem*)a.out2 + tlm_index<Tr>(o, k[i], a.KS), v[i] * w2);
    }
}

// ------------------------------------------------------------------------------------------------
// matrix products: up to three of them per launch, each dense, grouped (per head) or routed (per expert)
// ------------------------------------------------------------------------------------------------
enum { TLM_EPI_F32 = 0, TLM_EPI_PACK = 1, TLM_EPI_ROPE = 2, TLM_EPI_GRU = 3, TLM_EPI_LOGITS = 4, TLM_EPI_SILU = 5, TLM_EPI_GLU = 6, TLM_EPI_QKV = 7 };
enum { TLM_ACT_NONE = 0, TLM_ACT_RELU2 = 1 };
// queries, keys and values of grouped attention: head by head, every head padded to whole tiles; keys and values go to the cache
struct TlmQkv {
    void *kc, *vc;
    const int* crow;                     // cache row of the token: 64 page + offset
    int q_nt, k_nt, h_nt, v_nt;          // tiles of all query heads, of all key heads, per query / key head, per value head
    int heads, kv_heads;
};
struct TlmJob {
    const u32x4* wp; long wgs;           // packed weights; fragments x 64 per group
    const u32x4* xp; int xks, xkg;       // packed activations, their k-steps per row tile; k-step offset per group
    int KS, NT, groups, ksplit;
    int rows, rblocks;                   // dense rows; row blocks (routed: the bound on the number of tiles)
    int in_mul, in_gadd;                 // activation row of row r in group g: r * in_mul + g * in_gadd
    const int* list;                     // routed: pair list, tiles (expert, first, pairs), their number; activation row = pair / in_div
    const int* tiles;
    const int* n_tiles;
    int in_div;
    // routed: rows by their place in the list instead of by pair (activations in / out): the experts' hidden rows lie in the order in which
    // the down projection reads them, so that nothing is gathered there.  xrow: the activations are row-major (their k-steps xks wide), for
    // gathered rows: of a fragment-packed matrix a row's k-step is four pieces in four cache lines shared with seven other rows
    int in_pos, out_pos, xrow;
    int epi, act, act_nt;                // SILU: the first act_nt tiles
    void* out; int out_ld; long out_ps;  // fp32: row stride, stride per K split; packed: k-steps per row tile
    int out_mul, out_gadd, out_k0, out_kg;
    const float* bias;                   // GRU: [2][width]
    TlmQkv qkv;
    const float* gate; int gate_ld;      // PACK: factor per (row, group), or null
    const float* rope; int rope_ld;      // ROPE: (cos, sin) per row
    int n_valid;                         // LOGITS: columns
    float scale;                         // LOGITS: factor; GLU: limit
    int blocks;
};
struct TlmJobs {
    TlmJob j[3];
    int n;
    int height;                          // k_tlm_gemm_wide: rows per block, a multiple of 32
};

// cached values of grouped attention: the transposed operand of the value product, [page][kv head][keys / KSTEP][16-wide value blocks]
// fragments whose reduction order is the one the softmax weights have in the registers after S = K Q^T (bf16: keys 4 kq .. 4 kq + 3 of
// both 16-key halves)
template <class Tr>
MMI_HD long tlm_value_index(int crow, int g, int kv_heads, int d, int nd) {
    const int o = crow & (TLM_PAGE - 1), ko = o % Tr::KSTEP, half = ko >> 4;
    const long blk = ((long)(crow / TLM_PAGE) * kv_heads + g) * (TLM_PAGE / Tr::KSTEP) + o / Tr::KSTEP;
    return ((blk * nd + (d >> 4)) * 64 + ((ko & 15) >> 2) * 16 + (d & 15)) * Tr::V + 4 * half + (ko & 3);
}

template <class Tr, int EPI>
__device__ __forceinline__ void tlm_epilogue(const TlmJob& j, int g, int split, int id, int nt, int quad, f32x4 v) {
    const int n0 = nt * 16 + 4 * quad;
    const long orow = (long)id * j.out_mul + (long)g * j.out_gadd;
    if constexpr (EPI == TLM_EPI_F32) {
        *reinterpret_cast<f32x4*>((float*)j.out + split * j.out_ps + orow * j.out_ld + n0) = v;
    } else if constexpr (EPI == TLM_EPI_PACK) {
        if (j.act == TLM_ACT_RELU2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float r = v[e] > 0.f ? v[e] : 0.f;
                v[e] = r * r;
            }
        }
        if (j.gate) v *= j.gate[(long)id * j.gate_ld + g];
        Tr::store4((typename Tr::elem*)j.out + tlm_index<Tr>(orow, j.out_k0 + g * j.out_kg + n0, j.out_ld), v);
    } else if constexpr (EPI == TLM_EPI_ROPE) {
        // rotation pairs are adjacent (the weight rows are interleaved at load)
        const f32x4 cs = *reinterpret_cast<const f32x4*>(j.rope + ((long)id * j.rope_ld + n0 / 2) * 2);
        const f32x4 o = {v[0] * cs[0] - v[1] * cs[1], v[1] * cs[0] + v[0] * cs[1], v[2] * cs[2] - v[3] * cs[3], v[3] * cs[2] + v[2] * cs[3]};
        Tr::store4((typename Tr::elem*)j.out + tlm_index<Tr>(orow, j.out_k0 + g * j.out_kg + n0, j.out_ld), o);
    } else if constexpr (EPI == TLM_EPI_GRU) {
        // n-tiles alternate gate, candidate, output gate of the same 16 channels
        const int kind = nt % 3, c = (nt / 3) * 16 + 4 * quad;
        const int w = j.out_ld;
        f32x4 o;
        if (kind == 2) {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = v[e] * tlm_sigmoid(v[e]);
        } else {
            v += *reinterpret_cast<const f32x4*>(j.bias + kind * w + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (kind == 1 && v[e] >= 0.f) ? v[e] + 0.5f : tlm_sigmoid(v[e]);
        }
        *reinterpret_cast<f32x4*>((float*)j.out + orow * 3 * w + n0) = o;      // (in the order of the tiles: whole cache lines)
    } else if constexpr (EPI == TLM_EPI_SILU) {
        if (nt < j.act_nt) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= tlm_sigmoid(v[e]);
        }
        *reinterpret_cast<f32x4*>((float*)j.out + orow * j.out_ld + n0) = v;
    } else if constexpr (EPI == TLM_EPI_GLU) {
        // gate and up rows alternate (the weight rows are interleaved at load)
        float y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float g = fminf(v[2 * e], j.scale), u = fminf(fmaxf(v[2 * e + 1], -j.scale), j.scale);
            y[e] = g * tlm_sigmoid(1.702f * g) * (u + 1.0f);
        }
        Tr::store2((typename Tr::elem*)j.out + tlm_index<Tr>(orow, n0 / 2, j.out_ld), y[0], y[1]);
    } else if constexpr (EPI == TLM_EPI_QKV) {
        const TlmQkv& z = j.qkv;
        if (nt < z.q_nt) {
            const int h = nt / z.h_nt;
            Tr::store4((typename Tr::elem*)j.out + tlm_index<Tr>((long)id * z.heads + h, n0 - h * z.h_nt * 16, j.out_ld), v);
        } else if (nt < z.q_nt + z.k_nt) {
            const int g = (nt - z.q_nt) / z.h_nt, cr = z.crow[id];
            const long row = ((long)(cr / TLM_PAGE) * z.kv_heads + g) * TLM_PAGE + (cr & (TLM_PAGE - 1));
            Tr::store4((typename Tr::elem*)z.kc + tlm_index<Tr>(row, n0 - (z.q_nt + g * z.h_nt) * 16, j.out_ld), v);
        } else {
            const int t = nt - z.q_nt - z.k_nt, g = t / z.v_nt, cr = z.crow[id], d = n0 - (z.q_nt + z.k_nt + g * z.v_nt) * 16;
            typename Tr::elem* o = (typename Tr::elem*)z.vc + tlm_value_index<Tr>(cr, g, z.kv_heads, d, z.v_nt);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e * Tr::V] = Tr::cvt(v[e]);
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n0 + e < j.n_valid) ((float*)j.out)[orow * j.out_ld + n0 + e] = v[e] * j.scale;
    }
}

template <int E>
struct TlmEpi { static constexpr int value = E; };
// f(TlmEpi<kind>()) once per workgroup: the kinds' code is laid out one after the other, not interleaved per tile
template <class F>
__device__ __forceinline__ void tlm_with_epilogue(int epi, F f) {
    if (epi == TLM_EPI_F32) f(TlmEpi<TLM_EPI_F32>());
    else if (epi == TLM_EPI_PACK) f(TlmEpi<TLM_EPI_PACK>());
    else if (epi == TLM_EPI_ROPE) f(TlmEpi<TLM_EPI_ROPE>());
    else if (epi == TLM_EPI_GRU) f(TlmEpi<TLM_EPI_GRU>());
    else if (epi == TLM_EPI_SILU) f(TlmEpi<TLM_EPI_SILU>());
    else if (epi == TLM_EPI_GLU) f(TlmEpi<TLM_EPI_GLU>());
    else if (epi == TLM_EPI_QKV) f(TlmEpi<TLM_EPI_QKV>());
    else f(TlmEpi<TLM_EPI_LOGITS>());
}

// k-step 0 of activation row `in` for a lane
__device__ __forceinline__ const u32x4* tlm_row(const TlmJob& j, long in, int g, int lane) {
    return j.xp + (j.xrow ? in * j.xks * 4 + (lane >> 4) : ((in >> 4) * j.xks + (long)g * j.xkg) * 64 + (in & 15) + (lane >> 4) * 16);
}

// Few rows (<= 16 MT per block): the weights are an HBM stream.  A workgroup owns NTW n-tiles; its waves split K, each with U k-steps
// of weight fragments in flight per register buffer; partial tiles are summed through LDS in a fixed order.  Every activation fragment
// (an L2 read) meets NTW weight fragments, so that with many rows the activations do not cost more than the weights.
template <class Tr, int MT, int NTW, int WAVES, int U>
__global__ __launch_bounds__(WAVES * 64, WAVES == 4 ? 2 : 1) void k_tlm_gemm_rows(TlmJobs jobs) {
    int b = (int)blockIdx.x, ji = 0;
    while (ji + 1 < jobs.n && b >= jobs.j[ji].blocks) b -= jobs.j[ji++].blocks;
    const TlmJob j = jobs.j[ji];             // (a copy: its fields live in scalar registers)
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15;
    const int ntb = (j.NT + NTW - 1) / NTW, nt0 = (b % ntb) * NTW;
    b /= ntb;
    const int split = b % j.ksplit;
    b /= j.ksplit;
    int g = b % j.groups, rb = b / j.groups, r0 = rb * 16 * MT, n;
    if (j.list) {
        if (rb >= *j.n_tiles) return;
        g = j.tiles[3 * rb];
        r0 = j.tiles[3 * rb + 1];
        n = j.tiles[3 * rb + 2];
    } else {
        n = j.rows - r0 < 16 * MT ? j.rows - r0 : 16 * MT;
    }
    const u32x4* xq[MT];                                      // rows past n repeat the last one, and are dropped at the end
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int i = m * 16 + bl < n ? m * 16 + bl : n - 1;
        const int id = j.list ? j.list[r0 + i] : r0 + i;
        const long in = j.in_pos ? r0 + i : (j.list ? id / j.in_div : (long)id * j.in_mul + (long)g * j.in_gadd);
        xq[m] = tlm_row(j, in, g, lane);
    }
    const int xs = j.xrow ? 4 : 64;
    // K range of this split, then of this wave
    const int sper = (j.KS + j.ksplit - 1) / j.ksplit;
    const int s0 = min(j.KS, split * sper), s1 = min(j.KS, s0 + sper);
    const int wper = (s1 - s0 + WAVES - 1) / WAVES;
    const int k0 = min(s1, s0 + wave * wper), nk = min(s1, k0 + wper) - k0;
    const u32x4* wq[NTW];
#pragma unroll
    for (int t = 0; t < NTW; ++t) wq[t] = j.wp + (long)g * j.wgs + ((long)min(nt0 + t, j.NT - 1) * j.KS + k0) * 64 + lane;
    f32x4 acc[NTW][MT];
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 wA[U][NTW], wB[U][NTW], xA[U][MT], xB[U][MT];
#define TLM_LOAD(W_, X_, base)                                                                              \
    _Pragma("unroll") for (int u = 0; u < U; ++u) {                                                         \
        _Pragma("unroll") for (int t = 0; t < NTW; ++t) W_[u][t] = mmi_load_nt(wq[t] + (long)((base) + u) * 64); \
        _Pragma("unroll") for (int m = 0; m < MT; ++m) X_[u][m] = xq[m][(long)(k0 + (base) + u) * xs];      \
    }
#define TLM_MMA1(W_, X_, u)                                                                                 \
        _Pragma("unroll") for (int m = 0; m < MT; ++m)                                                      \
            _Pragma("unroll") for (int t = 0; t < NTW; ++t) acc[t][m] = Tr::mfma(W_[u][t], X_[u][m], acc[t][m]);
#define TLM_MMA(W_, X_)                                                                                     \
    _Pragma("unroll") for (int u = 0; u < U; ++u) { TLM_MMA1(W_, X_, u) }
    // no load of the steady state is conditional, so that the wait before a product only covers the older buffer
    const int nfull = nk / U, rem = nk - nfull * U;
    if (nfull > 0) {
        TLM_LOAD(wA, xA, 0);
        int i = 0;
        for (; i + 2 < nfull; i += 2) {
            TLM_LOAD(wB, xB, (i + 1) * U);
            mmi_sched_barrier();
            TLM_MMA(wA, xA);
            TLM_LOAD(wA, xA, (i + 2) * U);
            mmi_sched_barrier();
            TLM_MMA(wB, xB);
        }
        if (nfull - i == 2) {
            TLM_LOAD(wB, xB, (i + 1) * U);
            mmi_sched_barrier();
            TLM_MMA(wA, xA);
            TLM_MMA(wB, xB);
        } else {
            TLM_MMA(wA, xA);
        }
    }
    if (rem > 0) {                                            // fewer than U k-steps: requested together, from valid addresses
#pragma unroll
        for (int u = 0; u < U - 1; ++u) {
            const int k = nfull * U + min(u, rem - 1);
#pragma unroll
            for (int t = 0; t < NTW; ++t) wA[u][t] = mmi_load_nt(wq[t] + (long)k * 64);
#pragma unroll
            for (int m = 0; m < MT; ++m) xA[u][m] = xq[m][(long)(k0 + k) * xs];
        }
#pragma unroll
        for (int u = 0; u < U - 1; ++u)
            if (u < rem) { TLM_MMA1(wA, xA, u) }
    }
#undef TLM_MMA1
#undef TLM_LOAD
#undef TLM_MMA
    MMI_SHARED __attribute__((aligned(16))) f32x4 red[WAVES * NTW * MT * 64];
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) red[((wave * NTW + t) * MT + m) * 64 + lane] = acc[t][m];
    __syncthreads();
    tlm_with_epilogue(j.epi, [&](auto epi) __attribute__((always_inline)) {
#pragma unroll 1
        for (int q = wave; q < NTW * MT; q += WAVES) {
            const int t = q / MT, i = (q - t * MT) * 16 + bl;
            if (i >= n || nt0 + t >= j.NT) continue;
            f32x4 v = red[q * 64 + lane];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) v += red[(w * NTW * MT + q) * 64 + lane];
            tlm_epilogue<Tr, decltype(epi)::value>(j, g, split, j.list && !j.out_pos ? j.list[r0 + i] : r0 + i, nt0 + t, lane >> 4, v);
        }
    });
}

// Many rows: WN x WM waves, each over FN x FM fragments, i.e. 16 FN WN features x 16 FM WM rows per workgroup.  Operands go from global
// memory straight into a ring of ST stages of one k-step in LDS (whole fragments, so that both sides are conflict-free without a swizzle),
// ST - 2 stages ahead of the step that reads them into registers, which is one step ahead of the products that use them: a step is one
// meeting of the waves, its loads and LDS reads lie between the products of the step before.  KK = 2: a stage is two k-steps, with one meeting
// for both, where a wave has 8 products or fewer in a k-step (the blocks of 64 features).
// Bound by the matrix core's power (it runs at 0.95 - 1.2 PFLOP/s where a 16384^3 library product reaches 1.29) and, with few blocks, by
// the latency of a step (0.3 - 0.56 us).  Against the same tiles staged through registers: 1773 x 38912 x 4096 602 -> 543 us, 1773 x 4096 x
// (11264 + 4096) 263 -> 203.
template <class Tr, int FN, int FM, int WN, int WM, int ST, int KK>
struct TlmTile {
    static constexpr int NW = WN * WM, NFN = WN * FN, NFM = WM * FM, NF = NFN + NFM;
    static constexpr int NIN = KK * NFN / NW, NIM = KK * NFM / NW, NI = NIN + NIM;      // fragments that a wave brings to a stage
    static_assert(NFN % NW == 0 && (NFM % NW == 0 || (NW % NFM == 0 && KK * NFM % NW == 0)) && (ST == 3 || ST == 4), "every wave brings whole fragments; the waits are for one or two stages");
    static_assert(KK == 1 || KK == 2, "k-steps per stage: the register sets go round in pairs");
    static constexpr size_t smem() { return (size_t)ST * KK * NF * 1024; }
};
template <class Tr, int FN, int FM, int WN, int WM, int ST, int OCC, int KK>
__global__ __launch_bounds__(WN * WM * 64, OCC) void k_tlm_gemm_tile(TlmJobs jobs) {
    typedef TlmTile<Tr, FN, FM, WN, WM, ST, KK> P;
    MMI_DYN_SHARED(u32x4, lds);
    // consecutive workgroups go round the 8 XCDs: give each XCD a contiguous run of EVERY job's tiles - its L2 sees the shared operand, and no
    // XCD has the long tiles, or the experts' unused row blocks, to itself
    const int xcd = (int)blockIdx.x & 7;
    int b = (int)blockIdx.x >> 3, ji = 0;
    for (;; ++ji) {
        if (ji == jobs.n) return;
        const int lo = (int)((long)jobs.j[ji].blocks * xcd >> 3), mine = (int)((long)jobs.j[ji].blocks * (xcd + 1) >> 3) - lo;
        if (b < mine) {
            b += lo;
            break;
        }
        b -= mine;
    }
    const TlmJob j = jobs.j[ji];             // (a copy: its fields live in scalar registers)
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15;
    const int ntb = (j.NT + P::NFN - 1) / P::NFN, rb = b % j.rblocks;
    b /= j.rblocks;
    const int nb0 = b % ntb;
    b /= ntb;
    const int split = b % j.ksplit;
    int g = b / j.ksplit, n, r0;
    if (j.list) {
        if (rb >= *j.n_tiles) return;
        g = j.tiles[3 * rb];
        r0 = j.tiles[3 * rb + 1];
        n = j.tiles[3 * rb + 2];
    } else {
        r0 = rb * 16 * P::NFM;
        n = j.rows - r0 < 16 * P::NFM ? j.rows - r0 : 16 * P::NFM;
    }
    const int nt0 = nb0 * P::NFN, sper = (j.KS + j.ksplit - 1) / j.ksplit, k0 = min(j.KS, split * sper), ns = min(j.KS, k0 + sper) - k0;
    // fragment i of this wave, of one of the stage's k-steps: weights at a scalar address, activations (gathered rows) at one per lane
    const u32x4 *wq[P::NIN], *xq[P::NIM];
    constexpr auto kn = [](int i) { return P::NW * i / P::NFN; };
    auto km = [&](int i) __attribute__((always_inline)) { return P::NFM % P::NW == 0 ? P::NW * i / P::NFM : (wave + P::NW * i) / P::NFM; };
#pragma unroll
    for (int i = 0; i < P::NIN; ++i) wq[i] = j.wp + (long)g * j.wgs + ((long)min(nt0 + wave + P::NW * i - kn(i) * P::NFN, j.NT - 1) * j.KS + k0 + kn(i)) * 64;
    const int xs = j.xrow ? 4 : 64;
#pragma unroll
    for (int i = 0; i < P::NIM; ++i) {                        // (rows past n repeat the last one, and are dropped at the end)
        const int m = (wave + P::NW * i - km(i) * P::NFM) * 16 + bl, ii = m < n ? m : n - 1;
        const int id = j.list ? j.list[r0 + ii] : r0 + ii;
        const long in = j.in_pos ? r0 + ii : (j.list ? id / j.in_div : (long)id * j.in_mul + (long)g * j.in_gadd);
        xq[i] = tlm_row(j, in, g, lane) + (long)(k0 + km(i)) * xs;
    }
    const int stages = KK == 1 ? ns : (ns + 1) / 2;
    int to = 0, from = 0, left = stages;                      // places in the ring: of the next stage to load, of the next k-step to read; stages to load
    auto fetch_all = [&]() __attribute__((always_inline)) {
        // (an odd number of k-steps: the last stage gets the last one twice - stages are counted in loads)
        const int back = KK == 2 && --left == 0 && (ns & 1) ? 1 : 0;
#pragma unroll
        for (int i = 0; i < P::NIN; ++i) {
            mmi_load_lds(KK == 1 ? wq[i] : wq[i] - back * kn(i) * 64, lane * 16, lds, (to * KK * P::NF + wave + P::NW * i + kn(i) * P::NFM) * 64);
            wq[i] += KK * 64;
        }
#pragma unroll
        for (int i = 0; i < P::NIM; ++i) {
            mmi_load_lds(KK == 1 ? xq[i] : xq[i] - back * km(i) * xs, lds, (to * KK * P::NF + wave + P::NW * i + (km(i) + 1) * P::NFN) * 64);
            xq[i] += KK * xs;
        }
        to = to + 1 < ST ? to + 1 : 0;
    };
    const int wn = wave % WN, wm = wave / WN;
    const int ny = (n - wm * FM * 16 + 15) / 16;              // row fragments that hold rows (fp32: 512 cycles each and k-step, worth the branch)
    u32x4 av[2][FN], bv[2][FM];
    f32x4 acc[FN][FM];
#pragma unroll
    for (int x = 0; x < FN; ++x)
#pragma unroll
        for (int y = 0; y < FM; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto read = [&](int set, int i) __attribute__((always_inline)) {      // fragment i of FN + FM: rows first, they meet every feature
        const u32x4* base = lds + from * P::NF * 64 + lane;
        if (i < FM) bv[set][i < FM ? i : 0] = base[(P::NFN + wm * FM + i) * 64];
        else av[set][i < FM ? 0 : i - FM] = base[(wn * FN + i - FM) * 64];
    };
    auto wait = [&](int behind) __attribute__((always_inline)) {          // until only the last `behind` stages are in flight
        if (ST > 3 && behind == 2) mmi_wait_loads<(ST > 3 ? 2 : 0) * P::NI>();
        else if (behind == 1) mmi_wait_loads<P::NI>();
        else mmi_wait_loads<0>();
    };
    // products of k-step s (register set `cur`); between them the LDS reads of k-step s + 1 and, where that one begins a stage, the loads
    // of the stage ST - 2 behind it
    auto step = [&](auto set, int s) __attribute__((always_inline)) {
        constexpr int cur = decltype(set)::value;
        const bool more = s + 1 < ns;
        if (KK == 1 || cur == KK - 1) {
            const int c = KK == 1 ? s : s / KK;              // this stage
            if (more) {
                wait(ST == 3 ? 0 : min(stages - 1, c + ST - 2) - (c + 1));
                mmi_meet();
            }
            if (c + ST - 1 < stages) fetch_all();
        }
#pragma unroll
        for (int x = 0; x < FN; ++x) {
            if (more) {
#pragma unroll
                for (int i = x * (FN + FM) / FN; i < (x + 1) * (FN + FM) / FN; ++i) read(cur ^ 1, i);
            }
            mmi_sched_barrier();
#pragma unroll
            for (int y = 0; y < FM; ++y)
                if (Tr::V == 8 || y < ny) acc[x][y] = Tr::mfma(av[cur][x], bv[cur][y], acc[x][y]);
        }
        from = from + 1 < ST * KK ? from + 1 : 0;
    };
    if (ns > 0) {
        const int first = min(stages, ST - 1);
        for (int s = 0; s < first; ++s) fetch_all();
        wait(first - 1);
        mmi_meet();
#pragma unroll
        for (int i = 0; i < FN + FM; ++i) read(0, i);
        from = 1;
        int s = 0;
#pragma unroll 1
        for (; s + 1 < ns; s += 2) {
            step(std::integral_constant<int, 0>(), s);
            step(std::integral_constant<int, 1>(), s + 1);
        }
        if (s < ns) step(std::integral_constant<int, 0>(), s);
    }
    __syncthreads();
    tlm_with_epilogue(j.epi, [&](auto epi) __attribute__((always_inline)) {
#pragma unroll
        for (int y = 0; y < FM; ++y) {
            const int m = (wm * FM + y) * 16 + bl;
            if (m >= n) continue;
            const int id = j.list && !j.out_pos ? j.list[r0 + m] : r0 + m;
            // through LDS (a lane reads what it wrote), so that the epilogue's code is there once per y and not once per tile
            f32x4* buf = reinterpret_cast<f32x4*>(lds) + wave * FN * 64 + lane;
#pragma unroll
            for (int x = 0; x < FN; ++x) buf[x * 64] = acc[x][y];
            const int nx = min(FN, j.NT - nt0 - wn * FN);
#pragma unroll 1
            for (int x = 0; x < nx; ++x) tlm_epilogue<Tr, decltype(epi)::value>(j, g, split, id, nt0 + wn * FN + x, lane >> 4, buf[x * 64]);
        }
    });
}

// Dense products of many rows at bf16: 256 features x up to 256 rows per workgroup of 8 waves, 4 along the features and 2 along the rows, one
// workgroup per CU.  A wave has 64 features x 16 FM rows, FM = 1 .. 8 by the rows the block has: rows are cut evenly into blocks of a height
// that suits the chip (plan_jobs).  Operands as in k_tlm_gemm_tile; here a stage's place in the ring is loaded again as soon as its last
// k-step is in registers.  KK = 2 (two k-steps per meeting) where a wave has 12 products or fewer in a k-step.
// What bounds it: a CU has some 26 KB of loads on their way, whatever is asked for, so that a k-step takes the time in which its operands
// pass (64 rows: 0.36 us, most of them behind weights that come from HBM) unless its products take longer (256 rows: 0.78 us, 1.3 PFLOP/s).
// 256 x 256 loads 8 KB per MFLOP, 256 x 128 11, 128 x 64 24; against those, one workgroup per CU leaves its first loads and its last stores
// bare (8 us, and 8 - 19 us for 256 rows).  Width 2048, 639 rows, 14336 - 19456 features: 63.5 - 79.3 us in 128 x 64 blocks, 56.6 - 68.6 here;
// width 4096, 420 rows, 4096 x 11264 and 4096 x 4096 together: 95.5 and 83.8; 1773 rows: 282 and 238.
struct TlmWide {
    static constexpr int FN = 4, NFN = 16;                   // feature fragments of a wave, of the block
    static constexpr int kk(int fm) { return fm <= 3 ? 2 : 1; }
    static constexpr int stages(int fm) { return fm <= 3 ? 3 : 4; }
    static constexpr size_t smem() { return (size_t)3 * 2 * (NFN + 2 * 3) * 1024; }      // the largest ring: FM = 3 (8: 4 x 32 KB)
};
template <class Tr>
__global__ __launch_bounds__(512, 2) void k_tlm_gemm_wide(TlmJobs jobs) {
    constexpr int FN = TlmWide::FN, NFN = TlmWide::NFN, FMAX = 8;
    MMI_DYN_SHARED(u32x4, lds);
    const int xcd = (int)blockIdx.x & 7;                      // (every XCD a run of every job's blocks: k_tlm_gemm_tile)
    int b = (int)blockIdx.x >> 3, ji = 0;
    for (;; ++ji) {
        if (ji == jobs.n) return;
        const int lo = (int)((long)jobs.j[ji].blocks * xcd >> 3), mine = (int)((long)jobs.j[ji].blocks * (xcd + 1) >> 3) - lo;
        if (b < mine) {
            b += lo;
            break;
        }
        b -= mine;
    }
    const TlmJob j = jobs.j[ji];             // (a copy: its fields live in scalar registers)
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15;
    const int ntb = (j.NT + NFN - 1) / NFN, rb = b % j.rblocks;
    b /= j.rblocks;
    const int nt0 = b % ntb * NFN;
    const int split = b / ntb, r0 = rb * jobs.height, n = min(j.rows - r0, jobs.height);
    const int fm = (n + 31) / 32;                             // row fragments of a wave
    const int sper = (j.KS + j.ksplit - 1) / j.ksplit, k0 = min(j.KS, split * sper), ns = min(j.KS, k0 + sper) - k0;
    const int wn = wave & 3, wm = wave >> 2;
    f32x4 acc[FN][FMAX];
#pragma unroll
    for (int x = 0; x < FN; ++x)
#pragma unroll
        for (int y = 0; y < FMAX; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto products = [&](auto fmc) __attribute__((always_inline)) {
        constexpr int FM = decltype(fmc)::value, KK = TlmWide::kk(FM), ST = TlmWide::stages(FM), NF = NFN + 2 * FM;
        static_assert((size_t)ST * KK * NF * 1024 <= TlmWide::smem(), "the ring");
        // fragments that this wave brings to a stage: NW of the weights, NX of the KK x 2 FM of the activations, the last one in the first REST waves
        constexpr int NW = 2 * KK, AF = KK * 2 * FM, NX = (AF + 7) / 8, REST = AF % 8;
        const bool all = REST == 0 || wave < REST;
        auto act = [&](int i) __attribute__((always_inline)) { return min(wave + 8 * i, AF - 1); };
        const u32x4 *wq[NW], *xq[NX];
#pragma unroll
        for (int i = 0; i < NW; ++i) wq[i] = j.wp + ((long)min(nt0 + wave + 8 * (i / KK), j.NT - 1) * j.KS + k0 + i % KK) * 64;
#pragma unroll
        for (int i = 0; i < NX; ++i) {                        // (rows past n repeat the last one, and are dropped at the end)
            xq[i] = tlm_row(j, r0 + min(act(i) % (2 * FM) * 16 + bl, n - 1), 0, lane) + (long)(k0 + act(i) / (2 * FM)) * 64;
        }
        const int stages = (ns + KK - 1) / KK;
        int to = 0, from = 0, left = stages;                  // places in the ring: of the next stage to load, of the next k-step to read; stages to load
        auto fetch = [&]() __attribute__((always_inline)) {
            // (an odd number of k-steps: the last stage gets the last one twice - stages are counted in loads)
            const int back = KK == 2 && --left == 0 && (ns & 1) ? 1 : 0;
#pragma unroll
            for (int i = 0; i < NW; ++i) {
                mmi_load_lds(i % KK ? wq[i] - back * 64 : wq[i], lane * 16, lds, ((to * KK + i % KK) * NF + wave + 8 * (i / KK)) * 64);
                wq[i] += KK * 64;
            }
#pragma unroll
            for (int i = 0; i < NX; ++i)
                if (i + 1 < NX || all) {
                    const int k = act(i) / (2 * FM);
                    mmi_load_lds(k ? xq[i] - back * 64 : xq[i], lds, ((to * KK + k) * NF + NFN + act(i) - k * 2 * FM) * 64);
                    xq[i] += KK * 64;
                }
            to = to + 1 < ST ? to + 1 : 0;
        };
        auto wait = [&](int behind) __attribute__((always_inline)) {      // until only the last `behind` stages are in flight
            if (all) {
                if (ST > 3 && behind == 3) mmi_wait_loads<(ST > 3 ? 3 : 0) * (NW + NX)>();
                else if (behind == 2) mmi_wait_loads<2 * (NW + NX)>();
                else if (behind == 1) mmi_wait_loads<NW + NX>();
                else mmi_wait_loads<0>();
            } else {
                if (ST > 3 && behind == 3) mmi_wait_loads<(ST > 3 ? 3 : 0) * (NW + NX - 1)>();
                else if (behind == 2) mmi_wait_loads<2 * (NW + NX - 1)>();
                else if (behind == 1) mmi_wait_loads<NW + NX - 1>();
                else mmi_wait_loads<0>();
            }
        };
        u32x4 av[2][FN], bv[2][FM];
        auto read = [&](int set, int i) __attribute__((always_inline)) {      // fragment i of FN + FM: rows first, they meet every feature
            const u32x4* base = lds + from * NF * 64 + lane;
            if (i < FM) bv[set][i < FM ? i : 0] = base[(NFN + wm * FM + i) * 64];
            else av[set][i < FM ? 0 : i - FM] = base[(wn * FN + i - FM) * 64];
        };
        // products of k-step s (register set `cur`); between them the LDS reads of k-step s + 1.  Where that one begins a stage, every wave has
        // the stage in hand in its registers: its place is loaded again
        auto step = [&](auto set, int s) __attribute__((always_inline)) {
            constexpr int cur = decltype(set)::value;
            const bool more = s + 1 < ns;
            if ((KK == 1 || cur == 1) && more) {
                const int c = s / KK;                         // this stage
                wait(min(stages - 1, c + ST - 1) - (c + 1));
                mmi_meet();
                if (c + ST < stages) fetch();
            }
#pragma unroll
            for (int x = 0; x < FN; ++x) {
                if (more) {
#pragma unroll
                    for (int i = x * (FN + FM) / FN; i < (x + 1) * (FN + FM) / FN; ++i) read(cur ^ 1, i);
                }
                mmi_sched_barrier();
#pragma unroll
                for (int y = 0; y < FM; ++y) acc[x][y] = Tr::mfma(av[cur][x], bv[cur][y], acc[x][y]);
            }
            from = from + 1 < ST * KK ? from + 1 : 0;
        };
        const int first = min(stages, ST);
        for (int s = 0; s < first; ++s) fetch();
        wait(first - 1);
        mmi_meet();
#pragma unroll
        for (int i = 0; i < FN + FM; ++i) read(0, i);
        from = 1;
        int s = 0;
#pragma unroll 1
        for (; s + 1 < ns; s += 2) {
            step(std::integral_constant<int, 0>(), s);
            step(std::integral_constant<int, 1>(), s + 1);
        }
        if (s < ns) step(std::integral_constant<int, 0>(), s);
    };
    if (ns > 0) {
        if (fm == 8) products(std::integral_constant<int, 8>());
        else if (fm == 7) products(std::integral_constant<int, 7>());
        else if (fm == 6) products(std::integral_constant<int, 6>());
        else if (fm == 5) products(std::integral_constant<int, 5>());
        else if (fm == 4) products(std::integral_constant<int, 4>());
        else if (fm == 3) products(std::integral_constant<int, 3>());
        else if (fm == 2) products(std::integral_constant<int, 2>());
        else products(std::integral_constant<int, 1>());
    }
    __syncthreads();
    tlm_with_epilogue(j.epi, [&](auto epi) __attribute__((always_inline)) {
        const int nx = min(FN, j.NT - nt0 - wn * FN);
        f32x4* buf = reinterpret_cast<f32x4*>(lds) + wave * FN * 64 + lane;
#pragma unroll 1
        for (int y = 0; y < fm; ++y) {                        // through LDS (a lane reads what it wrote): the epilogue's code is there once
#pragma unroll
            for (int c = 0; c < FMAX; ++c)
                if (c == y)
#pragma unroll
                    for (int x = 0; x < FN; ++x) buf[x * 64] = acc[x][c];
            const int m = (wm * fm + y) * 16 + bl;
            if (m >= n) continue;
#pragma unroll 1
            for (int x = 0; x < nx; ++x) tlm_epilogue<Tr, decltype(epi)::value>(j, 0, split, r0 + m, nt0 + wn * FN + x, lane >> 4, buf[x * 64]);
        }
    });
}

// ------------------------------------------------------------------------------------------------
// latent attention
// ------------------------------------------------------------------------------------------------
// One workgroup per token, on the columns [query latent | latent | rotated key part | head gates] of the input projection (fp32
// split-K partials): the two RMS norms, the rotation of the key part, the cache write and the sigmoid of the gates.
struct TlmLatentArgs {
    const float* in; int in_p; long in_ps; int ld;       // ld: columns per row (every section rounded up to 16)
    int q_rank, kv_rank, rot, heads;
    int qp, kvp, rp;                                     // section widths
    const float* qw; const float* cw; float eps;
    const float* rope; int rope_ld;
    const int* crow;                                     // cache row of the token: 64 page + offset
    void* q; int q_ks;
    void* kc; int k_ks, rot_k0;
    float* gate; int gate_ld;
};
template <class Tr>
__global__ __launch_bounds__(256) void k_tlm_latent(TlmLatentArgs a) {
    typedef typename Tr::elem elem;
    MMI_DYN_SHARED(float, row);                          // [ld]
    MMI_SHARED float part[2][4];
    const int t = tlm_row_block((int)blockIdx.x, (int)gridDim.x), tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float sq = 0.f, sc = 0.f;
    for (int k = 4 * tid; k < a.ld; k += 1024) {
        f32x4 v = *reinterpret_cast<const f32x4*>(a.in + (long)t * a.ld + k);
#pragma unroll 4
        for (int p = 1; p < a.in_p; ++p) v += *reinterpret_cast<const f32x4*>(a.in + p * a.in_ps + (long)t * a.ld + k);
        *reinterpret_cast<f32x4*>(row + k) = v;
        const float s = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];     // the padding columns are zero
        if (k < a.qp) sq += s;
        else if (k < a.qp + a.kvp) sc += s;
    }
    sq = tlm_wave_sum(sq);
    sc = tlm_wave_sum(sc);
    if (lane == 0) {
        part[0][wave] = sq;
        part[1][wave] = sc;
    }
    __syncthreads();
    const float iq = 1.0f / sqrtf((part[0][0] + part[0][1] + part[0][2] + part[0][3]) / (float)a.q_rank + a.eps);
    const float ic = 1.0f / sqrtf((part[1][0] + part[1][1] + part[1][2] + part[1][3]) / (float)a.kv_rank + a.eps);
    const long cr = a.crow[t];
    for (int k = 4 * tid; k < a.ld; k += 1024) {
        f32x4 v = *reinterpret_cast<const f32x4*>(row + k);
        if (k < a.qp) {
            v *= iq * *reinterpret_cast<const f32x4*>(a.qw + k);
            Tr::store4((elem*)a.q + tlm_index<Tr>(t, k, a.q_ks), v);
        } else if (k < a.qp + a.kvp) {
            const int d = k - a.qp;
            v *= ic * *reinterpret_cast<const f32x4*>(a.cw + d);
            Tr::store4((elem*)a.kc + tlm_index<Tr>(cr, d, a.k_ks), v);
        } else if (k < a.qp + a.kvp + a.rp) {
            const int d = k - a.qp - a.kvp;
            const f32x4 cs = *reinterpret_cast<const f32x4*>(a.rope + ((long)t * a.rope_ld + d / 2) * 2);
            const f32x4 o = {v[0] * cs[0] - v[1] * cs[1], v[1] * cs[0] + v[0] * cs[1], v[2] * cs[2] - v[3] * cs[3], v[3] * cs[2] + v[2] * cs[3]};
            Tr::store4((elem*)a.kc + tlm_index<Tr>(cr, a.rot_k0 + d, a.k_ks), o);
        } else {
            const int h = k - a.qp - a.kvp - a.rp;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (h + e < a.heads) a.gate[(long)t * a.gate_ld + h + e] = tlm_sigmoid(v[e]);
        }
    }
}

// Attention over the latent cache.  All heads share one key per position - (latent, rotated part) against the queries absorbed
// through the key projection - and the value is the latent itself, so (token, head) pairs are the columns of one product and a key
// fragment serves 16 of them.  A column tile never mixes sequences.  Keys are walked in blocks of 32; a column sees key j of its
// token at position i when 0 <= i - j < window.
// which keys a position sees, and the factor of the scores (times log2(e)): the last `window` ones (0: all), and the first `keep`
struct TlmMask { int window, keep; float scale; };
// pages of a sequence: the block table's first `keep` entries are for the pages that no window releases, the others are a ring
struct TlmPages { const int* table; int ld, keep; };
__device__ __forceinline__ int tlm_page(const TlmPages& p, const int* row, int i) { return mmi_load_const(row + (i < p.keep ? i : p.keep + (i - p.keep) % (p.ld - p.keep))); }

struct TlmAttnArgs {
    const void* q;                       // packed rows token * heads + head
    const void* kc;
    void* out; int out_rows;             // packed rows head * out_rows + token, latent columns (the value projection reads head by head)
    int heads, q_ks, nd, out_ks;
    TlmMask mask;
    int n_entries, n_tiles, nsplit;
    const int* tile0;                    // [entries + 1] first column tile (k_tlm_attn_tile: column group) of each entry
    const int* erow0; const int* elen; const int* epos0; const int* eslot;
    TlmPages pages;                      // table [slot][ld]
    float* po;                           // nsplit > 1: [tile][split][nd][64] f32x4 un-normalised sums
    float* pml;                          // [tile][split][2][16]: running maximum, sum of weights
};
struct TlmCols { int entry, c0, ncol; };
template <class Args>
__device__ __forceinline__ TlmCols tlm_find_tile(const Args& a, int tile) {
    // the last entry whose first tile is <= tile: all prefixes compared at once (a binary search would be a chain of dependent loads)
    unsigned below = 0;
    for (int e = mmi_lane(); e < a.n_entries; e += 64) below += a.tile0[e] <= tile ? 1u : 0u;
    const int lo = mmi_uniform((int)mmi_wave_sum_u32(below) - 1);
    TlmCols c;
    c.entry = lo;
    c.c0 = (tile - a.tile0[lo]) * 16;
    c.ncol = a.elen[lo] * a.heads;
    return c;
}

template <class Tr>
__device__ __forceinline__ void tlm_attn_store(const TlmAttnArgs& a, const TlmCols& c, int bl, int kq, int db, f32x4 v) {
    const int col = c.c0 + bl;
    if (col >= c.ncol) return;
    const int t = col / a.heads;
    const long orow = (long)(col - t * a.heads) * a.out_rows + a.erow0[c.entry] + t;
    Tr::store4((typename Tr::elem*)a.out + tlm_index<Tr>(orow, db * 16 + 4 * kq, a.out_ks), v);
}

// Shapes are template bounds - ND 16-wide latent blocks, RK k-steps of the rotated part - and the loops run over the bounds without a
// branch, so that a block's loads are all in flight together: fragments past the model's own sizes repeat a valid address against zero
// query fragments, value blocks past them are dropped at the end.
template <class Tr, int ND, int RK>
struct TlmQuery {
    static constexpr int LK = ND * 16 / Tr::KSTEP, NK = LK + RK;
    static constexpr int NB = 32 / (4 * Tr::V);                    // value fragments per 32 keys and latent block
    u32x4 f[NK];
    static __device__ __forceinline__ u32x4 fragment(const TlmAttnArgs& a, const u32x4* qp, int s) {
        const int o = s < LK ? s : a.out_ks + s - LK;
        const u32x4 zero = {0u, 0u, 0u, 0u};
        return (s < LK ? s < a.out_ks : o < a.q_ks) ? qp[o * 64] : zero;
    }
    __device__ __forceinline__ void load(const TlmAttnArgs& a, long qrow, int kq) {
        const u32x4* qp = (const u32x4*)a.q + (qrow >> 4) * a.q_ks * 64 + kq * 16 + (qrow & 15);
#pragma unroll
        for (int s = 0; s < NK; ++s) f[s] = fragment(a, qp, s);
    }
};
// 32 (16 at fp32) keys x KSTEP latent dimensions -> the transposed operand, through the matrix core: K x identity is exact
template <class Tr>
struct TlmFlip {
    static constexpr int H = Tr::KSTEP / 16;                       // 16-wide latent blocks per k-step
    u32x4 id[H];
    __device__ __forceinline__ void init(int bl, int kq) {
#pragma unroll
        for (int h = 0; h < H; ++h) {
            if constexpr (Tr::V == 8) {
                const int e = 16 * h + bl - 8 * kq;                // k = 8 kq + e meets column bl where k = 16 h + bl
#pragma unroll
                for (int i = 0; i < 4; ++i) id[h][i] = e == 2 * i ? 0x00003f80u : (e == 2 * i + 1 ? 0x3f800000u : 0u);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) id[h][i] = 4 * kq + i == bl ? 0x3f800000u : 0u;
            }
        }
    }
    // bf16: latent block h of the two 16-key fragments of a k-step; fp32: of one
    __device__ __forceinline__ u32x4 turn(u32x4 k0, u32x4 k1, int h) const {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        const f32x4 a = Tr::mfma(k0, id[h], zero);
        if constexpr (Tr::V == 8) {
            const f32x4 b = Tr::mfma(k1, id[h], zero);
            return u32x4{mmi_pack_bf16x2(a[0], a[1]), mmi_pack_bf16x2(a[2], a[3]), mmi_pack_bf16x2(b[0], b[1]), mmi_pack_bf16x2(b[2], b[3])};
        } else {
            return __builtin_bit_cast(u32x4, a);
        }
    }
};
// k-step of the cache that fragment s of the bound stands for
template <int LK>
__device__ __forceinline__ int tlm_kstep_of(const TlmAttnArgs& a, int s) {
    return s < LK ? min(s, a.out_ks - 1) : min(a.out_ks + s - LK, a.q_ks - 1);
}
// Scores of 32 keys and QT column tiles -> softmax weights as operand fragments, the running maxima, sums and outputs moved on (the lane's
// keys are k0 .. k0 + 3 and k0 + 16 .. k0 + 19, its column of tile t is at position k0 + d0[t]).
// In the prompts' kernels the vector unit and its latencies stood in the matrix cores' way (845 vector instructions per block of 32 keys
// and 32 columns against 72 products; now some 200), so what is not needed is left out: the mask is looked at only where some key of some
// column lies outside it, the exponential is the hardware's, the maxima cross lanes in registers, and sums are rescaled only where some
// maximum has grown.  (Not only once it has grown by 2^8, which would save 0.2 - 0.4 % of a prompt: the largest weight is then no longer
// exactly one, and its rounding to bf16 does not cancel against the sum, which is of unrounded weights.  Mean error against 64 bits over 64 steps of
// Bibapel at widths 1024 and 2048: 0.003033 with that slack, 0.003030 without; Kesirax' logits are the library exponential's, bit for bit.)
template <class Tr, int ND, int QT>
__device__ __forceinline__ void tlm_softmax_block(const TlmMask& a, f32x4 (&s)[QT][2], int k0, const int (&d0)[QT], float (&m)[QT], float (&l)[QT],
                                                  u32x4 (&pf)[QT][32 / (4 * Tr::V)], f32x4 (&acc)[QT][ND]) {
    constexpr int NB = 32 / (4 * Tr::V);
    bool edge = false, moved = false;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        edge = edge || d0[t] < 19 || (a.window > 0 && d0[t] >= a.window);
        s[t][0] *= a.scale;
        s[t][1] *= a.scale;
    }
    if (mmi_any(edge)) {
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e0 = d0[t] - r, e1 = d0[t] - r - 16;
                s[t][0][r] = e0 >= 0 && (a.window <= 0 || e0 < a.window || k0 + r < a.keep) ? s[t][0][r] : -INFINITY;
                s[t][1][r] = e1 >= 0 && (a.window <= 0 || e1 < a.window || k0 + r + 16 < a.keep) ? s[t][1][r] : -INFINITY;
            }
    }
    float mx[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        float x = m[t];
#pragma unroll
        for (int r = 0; r < 4; ++r) x = fmaxf(x, fmaxf(s[t][0][r], s[t][1][r]));
        mx[t] = mmi_rows_max(x);
        moved = moved || mx[t] > m[t];
    }
    if (mmi_any(moved)) {
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            const float al = mmi_fast_exp2f(m[t] - mx[t]);
            m[t] = mx[t];
            l[t] *= al;
#pragma unroll
            for (int d = 0; d < ND; ++d) acc[t][d] *= al;
        }
    }
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        f32x4 p0, p1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p0[r] = mmi_fast_exp2f(s[t][0][r] - m[t]);
            p1[r] = mmi_fast_exp2f(s[t][1][r] - m[t]);
            l[t] += p0[r] + p1[r];
        }
        if constexpr (NB == 1) {
            pf[t][0] = u32x4{mmi_pack_bf16x2(p0[0], p0[1]), mmi_pack_bf16x2(p0[2], p0[3]), mmi_pack_bf16x2(p1[0], p1[1]), mmi_pack_bf16x2(p1[2], p1[3])};
        } else {
            pf[t][0] = __builtin_bit_cast(u32x4, p0);
            pf[t][NB - 1] = __builtin_bit_cast(u32x4, p1);
        }
    }
}

template <class Tr, int ND>
__device__ __forceinline__ void tlm_softmax_block(const TlmMask& a, f32x4 s0, f32x4 s1, int k0, int d0, float& m, float& l, u32x4 (&pf)[32 / (4 * Tr::V)], f32x4 (&acc)[ND]) {
    f32x4 s[1][2] = {{s0, s1}};
    const int d[1] = {d0};
    tlm_softmax_block<Tr, ND, 1>(a, s, k0, d, reinterpret_cast<float (&)[1]>(m), reinterpret_cast<float (&)[1]>(l), reinterpret_cast<u32x4 (&)[1][32 / (4 * Tr::V)]>(pf),
                                 reinterpret_cast<f32x4 (&)[1][ND]>(acc));
}

// One block of 32 keys as a stream of fragments out of LDS - keys 0-15 and 16-31 of every k-step, then the turned values - consumed in
// groups of G, the next group read while one is used.
template <class Tr, int ND, int RK, int QT, int G>
struct TlmAttnStream {
    typedef TlmQuery<Tr, ND, RK> Q;
    static constexpr int NB = Q::NB, NK = Q::NK, F = 2 * NK + ND * NB, NG = ((F + G - 1) / G + 1) / 2 * 2;      // an even number of groups: group g always meets buffer g & 1
    u32x4 fr[2][G];
    f32x4 s[QT][2];
    u32x4 pf[QT][NB];
    float m[QT], l[QT];
    f32x4 acc[QT][ND];
    __device__ __forceinline__ void clear(float m0 = -1e30f) {
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            m[t] = m0;
            l[t] = 0.f;
#pragma unroll
            for (int d = 0; d < ND; ++d) acc[t][d] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // at(f): address of fragment f for this lane
    template <class At>
    __device__ __forceinline__ void load(int buf, int g, At at) {
#pragma unroll
        for (int i = 0; i < G; ++i)
            if (g * G + i < F) fr[buf][i] = *at(g * G + i);
    }
    // q(t, k): query fragment k of column tile t
    template <class Qf>
    __device__ __forceinline__ void use(const TlmMask& a, Qf q, int buf, int g, int k0, const int (&d0)[QT]) {
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const int f = g * G + i;
            if (f >= F) continue;
            if (f < 2 * NK) {
#pragma unroll
                for (int t = 0; t < QT; ++t) s[t][f & 1] = Tr::mfma(fr[buf][i], q(t, f >> 1), f < 2 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[t][f & 1]);
                if (f == 2 * NK - 1) tlm_softmax_block<Tr, ND, QT>(a, s, k0, d0, m, l, pf, acc);
            } else {
                const int d = (f - 2 * NK) / NB;
#pragma unroll
                for (int t = 0; t < QT; ++t) acc[t][d] = Tr::mfma(fr[buf][i], pf[t][(f - 2 * NK) % NB], acc[t][d]);
            }
        }
    }
};

// Few column tiles (decoding): the four waves of a workgroup share one column tile, each takes every 4th key block straight from the
// cache, and their sums meet in LDS.  gridDim.y > 1: the keys are also split over workgroups (k_tlm_attn_combine).
template <class Tr, int ND, int RK>
__global__ __launch_bounds__(256, Tr::V == 8 && ND <= 16 ? 2 : 1) void k_tlm_attn(TlmAttnArgs a) {      // two workgroups per CU where the registers allow it
    typedef TlmQuery<Tr, ND, RK> Q;
    constexpr int NB = Q::NB, WK = 4;
    MMI_SHARED float ml[2][4][16];
    MMI_SHARED __attribute__((aligned(16))) f32x4 ob[4 * 8 * 64];
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15, kq = lane >> 4, split = (int)blockIdx.y;
    // consecutive workgroups go round the 8 XCDs: neighbouring tiles (heads of one sequence read the same keys) to one XCD's L2
    const int tile = ((int)blockIdx.x & 7) * ((int)gridDim.x >> 3) + ((int)blockIdx.x >> 3);
    if (tile >= a.n_tiles) return;
    const TlmCols c = tlm_find_tile(a, tile);
    const int col = c.c0 + bl < c.ncol ? c.c0 + bl : c.ncol - 1;
    const int pos0 = a.epos0[c.entry];
    const int pc = pos0 + col / a.heads;                           // position of this lane's column
    const int plo = pos0 + c.c0 / a.heads, phi = pos0 + (min(c.c0 + 15, c.ncol - 1)) / a.heads;
    const int klo = a.mask.window > 0 && plo - a.mask.window + 1 > 0 ? plo - a.mask.window + 1 : 0;
    int b0 = klo / 32, b1 = phi / 32 + 1;
    if (a.nsplit > 1) {
        const int per = (b1 - b0 + a.nsplit - 1) / a.nsplit;
        b0 = min(b1, b0 + split * per);
        b1 = min(b1, b0 + per);
    }
    const int* bt = a.pages.table + (long)a.eslot[c.entry] * a.pages.ld;
    f32x4 acc[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -1e30f, l = 0.f;
    TlmFlip<Tr> flip;
    flip.init(bl, kq);
    // the waves share the column tile: its query fragments stay in LDS, the registers are for keys in flight
    MMI_SHARED __attribute__((aligned(16))) u32x4 ql[Q::NK * 64];
    {
        const long qrow = (long)a.erow0[c.entry] * a.heads + col;
        const u32x4* qp = (const u32x4*)a.q + (qrow >> 4) * a.q_ks * 64 + kq * 16 + (qrow & 15);
        for (int s = wave; s < Q::NK; s += WK) ql[s * 64 + lane] = Q::fragment(a, qp, s);
        __syncthreads();
    }
    // A block's key fragments stay in registers from the scores to the values (turned there), and each one's register asks for the next
    // block's fragment as soon as it has been used: a block is read once, and nearly a whole block is always in flight.
    constexpr int NK = Q::NK, LK = Q::LK, FH = TlmFlip<Tr>::H, GK = 4;
    u32x4 fr[NK][2];
    const u32x4* kp = (const u32x4*)a.kc;
    auto block = [&](int kb) __attribute__((always_inline)) {
        const long page = tlm_page(a.pages, bt, min(kb, b1 - 1) >> 1);    // (past the end: the last block again)
        kp = (const u32x4*)a.kc + (page * 4 + (kb & 1) * 2) * a.q_ks * 64 + lane;
    };
    auto load = [&](int k) __attribute__((always_inline)) {
        const int o = tlm_kstep_of<LK>(a, k);
        fr[k][0] = kp[o * 64];
        fr[k][1] = kp[(a.q_ks + o) * 64];
    };
    if (b0 + wave < b1) {
        block(b0 + wave);
#pragma unroll
        for (int k = 0; k < NK; ++k) load(k);
    }
    for (int kb = b0 + wave; kb < b1; kb += WK) {
        block(kb + WK);
        f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            const u32x4 qv = ql[k * 64 + lane];
            s0 = Tr::mfma(fr[k][0], qv, s0);
            s1 = Tr::mfma(fr[k][1], qv, s1);
        }
#pragma unroll
        for (int k = LK; k < NK; ++k) load(k);
        mmi_sched_barrier();
        u32x4 pf[NB];
        tlm_softmax_block<Tr, ND>(a.mask, s0, s1, kb * 32 + 4 * kq, pc - (kb * 32 + 4 * kq), m, l, pf, acc);
#pragma unroll
        for (int k0 = 0; k0 < LK; k0 += GK) {
#pragma unroll
            for (int k = k0; k < k0 + GK && k < LK; ++k)
#pragma unroll
                for (int h = 0; h < FH; ++h) {
                    acc[k * FH + h] = Tr::mfma(flip.turn(fr[k][0], fr[k][1], h), pf[0], acc[k * FH + h]);
                    if constexpr (NB == 2) acc[k * FH + h] = Tr::mfma(flip.turn(fr[k][1], fr[k][1], h), pf[NB - 1], acc[k * FH + h]);
                }
#pragma unroll
            for (int k = k0; k < k0 + GK && k < LK; ++k) load(k);
            mmi_sched_barrier();
        }
    }
    l += mmi_shfl_xor(l, 16);
    l += mmi_shfl_xor(l, 32);
    if (kq == 0) {
        ml[0][wave][bl] = m;
        ml[1][wave][bl] = l;
    }
    __syncthreads();
    float M = -1e30f, L = 0.f;
#pragma unroll
    for (int w = 0; w < WK; ++w) M = fmaxf(M, ml[0][w][bl]);
#pragma unroll
    for (int w = 0; w < WK; ++w) L += ml[1][w][bl] * exp2f(ml[0][w][bl] - M);
    const float f = exp2f(m - M);
    const float inv = a.nsplit > 1 ? 1.f : 1.0f / L;
#pragma unroll
    for (int d0 = 0; d0 < ND; d0 += 8) {
        if (d0 >= a.nd) break;
        if (d0) __syncthreads();
#pragma unroll
        for (int d = 0; d < 8; ++d)
            if (d0 + d < ND) ob[(wave * 8 + d) * 64 + lane] = acc[d0 + d < ND ? d0 + d : 0] * f;
        __syncthreads();
#pragma unroll
        for (int d = wave; d < 8; d += WK) {
            if (d0 + d >= a.nd) break;
            f32x4 v = ob[d * 64 + lane];
#pragma unroll
            for (int w = 1; w < WK; ++w) v += ob[(w * 8 + d) * 64 + lane];
            if (a.nsplit > 1) *reinterpret_cast<f32x4*>(a.po + ((((long)tile * a.nsplit + split) * a.nd + d0 + d) * 64 + lane) * 4) = v;
            else tlm_attn_store<Tr>(a, c, bl, kq, d0 + d, v * inv);
        }
    }
    if (a.nsplit > 1 && wave == 0 && kq == 0) {
        float* p = a.pml + ((long)tile * a.nsplit + split) * 32;
        p[bl] = M;
        p[16 + bl] = L;
    }
}

// Many columns (prompts): four waves x QT column tiles of one sequence walk the same keys; a block's fragments are staged through LDS
// once for all of them (NBUF buffers, the next block in flight in registers while this one is used).
// QT: as many tiles as leave room for a second workgroup on the CU (256 registers per wave), whose products fill the waits of this one's
// softmax; with 512 registers the compiler also moved the sums between the two register files in every block.  2048 tokens, 16 heads, 256
// latent columns, window 1024: two tiles and one workgroup per CU 89 us (and 114 before the softmax was trimmed), one tile and two 70.
template <class Tr, int ND, int RK>
struct TlmAttnTile {
    static constexpr int QT = ND <= 8 ? 2 : 1;
    static constexpr int NF = 2 * TlmQuery<Tr, ND, RK>::NK + ND * TlmQuery<Tr, ND, RK>::NB;      // fragments per 32 keys
    static constexpr int NBUF = 2 * NF <= 152 ? 2 : 1;
    static constexpr size_t smem() { return (size_t)NBUF * NF * 1024; }
};
template <class Tr, int ND, int RK>
__global__ __launch_bounds__(256, Tr::V == 8 && ND <= 16 ? 2 : 1) void k_tlm_attn_tile(TlmAttnArgs a) {
    typedef TlmQuery<Tr, ND, RK> Q;
    typedef TlmAttnTile<Tr, ND, RK> P;
    constexpr int NB = Q::NB, NK = Q::NK, QT = P::QT, NF = P::NF, NBUF = P::NBUF, NI = (NK + 3) / 4, FH = TlmFlip<Tr>::H;
    MMI_DYN_SHARED(u32x4, lds);
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15, kq = lane >> 4;
    int g = (int)blockIdx.x;
    TlmCols c;                                                     // (tile0 counts groups of 64 QT columns here)
    {
        c = tlm_find_tile(a, g);
        c.c0 *= 4 * QT;
    }
    const int pos0 = a.epos0[c.entry];
    const int plo = pos0 + c.c0 / a.heads, phi = pos0 + min(c.c0 + 64 * QT - 1, c.ncol - 1) / a.heads;
    const int klo = a.mask.window > 0 && plo - a.mask.window + 1 > 0 ? plo - a.mask.window + 1 : 0;
    const int b0 = klo / 32, b1 = phi / 32 + 1;
    const int* bt = a.pages.table + (long)a.eslot[c.entry] * a.pages.ld;
    typedef TlmAttnStream<Tr, ND, RK, QT, (ND >= 16 ? 4 : 8)> S;
    Q q[QT];
    S sm;
    sm.clear();
    TlmFlip<Tr> flip;
    flip.init(bl, kq);
    int pc[QT], c0[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        c0[t] = c.c0 + (wave * QT + t) * 16;
        const int col = c0[t] + bl < c.ncol ? c0[t] + bl : c.ncol - 1;
        pc[t] = pos0 + col / a.heads;
        q[t].load(a, (long)a.erow0[c.entry] * a.heads + col, kq);
    }
    // fragments of a block in LDS: keys 0-15 and 16-31 of each k-step, then the turned values; wave w brings k-steps w, w + 4, ..
    u32x4 st[NI][2];
    auto page_of = [&](int kb) __attribute__((always_inline)) { return tlm_page(a.pages, bt, min(kb, b1 - 1) >> 1); };
    long page = page_of(b0);                                       // of the block fetched next
    auto fetch = [&](int kb) __attribute__((always_inline)) {
        const u32x4* kp = (const u32x4*)a.kc + (page * 4 + (kb & 1) * 2) * a.q_ks * 64 + lane;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int o = tlm_kstep_of<Q::LK>(a, min(wave + 4 * i, NK - 1));
            st[i][0] = kp[o * 64];
            st[i][1] = kp[(a.q_ks + o) * 64];
        }
        page = page_of(kb + 1);
    };
    auto stage = [&](int buf) __attribute__((always_inline)) {
        u32x4* base = lds + buf * NF * 64 + lane;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int k = wave + 4 * i;
            if (4 * i + 3 >= NK && k >= NK) continue;
            base[(2 * k) * 64] = st[i][0];
            base[(2 * k + 1) * 64] = st[i][1];
            if (4 * i + 3 >= Q::LK && k >= Q::LK) continue;          // the rotated part has no value
#pragma unroll
            for (int h = 0; h < FH; ++h) {
                const int d = k * FH + h;
                if constexpr (NB == 1) {
                    base[(2 * NK + d) * 64] = flip.turn(st[i][0], st[i][1], h);
                } else {
                    base[(2 * NK + d * NB) * 64] = flip.turn(st[i][0], st[i][0], h);
                    base[(2 * NK + d * NB + NB - 1) * 64] = flip.turn(st[i][1], st[i][1], h);
                }
            }
        }
    };
    fetch(b0);
    stage(0);
    __syncthreads();
    int cur = 0;
    for (int kb = b0; kb < b1; ++kb) {
        fetch(kb + 1);                                             // (past the end: the last block's page again)
        mmi_sched_barrier();
        const u32x4* base = lds + cur * NF * 64 + lane;
        auto at = [&](int f) __attribute__((always_inline)) -> const u32x4* { return base + f * 64; };
        auto qf = [&](int t, int k) __attribute__((always_inline)) { return q[t].f[k]; };
        int d0[QT];
#pragma unroll
        for (int t = 0; t < QT; ++t) d0[t] = pc[t] - (kb * 32 + 4 * kq);
        sm.load(0, 0, at);
#pragma unroll
        for (int g = 0; g < S::NG; ++g) {
            if (g + 1 < S::NG) sm.load((g + 1) & 1, g + 1, at);
            mmi_sched_barrier();
            sm.use(a.mask, qf, g & 1, g, kb * 32 + 4 * kq, d0);
        }
        if constexpr (NBUF == 1) __syncthreads();
        else cur ^= 1;
        stage(cur);
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        float l = sm.l[t];
        l += mmi_shfl_xor(l, 16);
        l += mmi_shfl_xor(l, 32);
        const float inv = 1.0f / l;
        TlmCols o = c;
        o.c0 = c0[t];
#pragma unroll
        for (int d = 0; d < ND; ++d)
            if (d < a.nd) tlm_attn_store<Tr>(a, o, bl, kq, d, sm.acc[t][d] * inv);
    }
}

// the splits of one column tile -> output; one workgroup per tile, waves over the latent blocks
template <class Tr>
__global__ __launch_bounds__(256) void k_tlm_attn_combine(TlmAttnArgs a) {
    const int lane = (int)threadIdx.x & 63, wave = mmi_uniform((int)threadIdx.x >> 6), bl = lane & 15, kq = lane >> 4, tile = (int)blockIdx.x;
    const TlmCols c = tlm_find_tile(a, tile);
    const float* q = a.pml + (long)tile * a.nsplit * 32;
    float M = -1e30f, L = 0.f;
#pragma unroll 4
    for (int s = 0; s < a.nsplit; ++s) M = fmaxf(M, q[s * 32 + bl]);
#pragma unroll 4
    for (int s = 0; s < a.nsplit; ++s) L += q[s * 32 + 16 + bl] * exp2f(q[s * 32 + bl] - M);
    const float inv = 1.0f / L;
    for (int d = wave + 4 * (int)blockIdx.y; d < a.nd; d += 4 * (int)gridDim.y) {
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int s = 0; s < a.nsplit; ++s)
            v += *reinterpret_cast<const f32x4*>(a.po + ((((long)tile * a.nsplit + s) * a.nd + d) * 64 + lane) * 4) * exp2f(q[s * 32 + bl] - M);
        tlm_attn_store<Tr>(a, c, bl, kq, d, v * inv);
    }
}

// ------------------------------------------------------------------------------------------------
// minimal gated recurrence: S_t = (1 - z_t) S_(t-1) + z_t c_t, output S_t * g_t, from the fp32 gates the projection's epilogue stored.
// A step's sequences are cut into segments of at most TLM_SEG tokens.  The recurrence is linear in S, so a segment is the pair
// (A, B) with S_end = A S_begin + B: the first launch computes the pairs (only when some sequence has more than one segment), the
// second starts every segment from its predecessors' pairs.  State is [slot][2][width]: read one copy, write the other, so that a
// segment's write cannot be seen by another segment of the same sequence.
// ------------------------------------------------------------------------------------------------
constexpr int TLM_SEG = 32;
struct TlmSeg { int row0, n, slot, par, index, last, fresh, pad; };      // index: number of the segment in its sequence; fresh: position 0
struct TlmScanArgs {
    const float* zcg;             // [row][width / 16][3][16]
    int width;                    // padded to 16
    const TlmSeg* seg;
    float* state;
    float* pair;                  // [segment][2][width]
    void* out; int out_ks;
};
__global__ __launch_bounds__(256) void k_tlm_scan_pairs(TlmScanArgs a) {
    const int c = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const TlmSeg s = a.seg[blockIdx.y];
    if (c >= a.width || s.last) return;
    const float* p = a.zcg + (long)s.row0 * 3 * a.width + c / 16 * 48 + c % 16;
    float A = 1.f, B = 0.f;
    for (int i0 = 0; i0 < s.n; i0 += 8) {
        float z[8], u[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const long o = (long)(i0 + i < s.n ? i0 + i : s.n - 1) * 3 * a.width;
            z[i] = p[o];
            u[i] = p[o + 16];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i0 + i < s.n) {
                A *= 1.0f - z[i];
                B = mmi_fma(1.0f - z[i], B, z[i] * u[i]);
            }
    }
    a.pair[(long)blockIdx.y * 2 * a.width + c] = A;
    a.pair[((long)blockIdx.y * 2 + 1) * a.width + c] = B;
}
template <class Tr>
__global__ __launch_bounds__(256) void k_tlm_scan(TlmScanArgs a) {
    const int c = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    const TlmSeg s = a.seg[blockIdx.y];
    if (c >= a.width) return;
    const float* p = a.zcg + (long)s.row0 * 3 * a.width + c / 16 * 48 + c % 16;
    typename Tr::elem* out = (typename Tr::elem*)a.out;
    float S = s.fresh ? 0.f : a.state[((long)s.slot * 2 + s.par) * a.width + c];
    const float* q = a.pair + (long)((int)blockIdx.y - s.index) * 2 * a.width + c;
    for (int i0 = 0; i0 < s.index; i0 += 8) {                      // (a step waits for the one before it, its loads need not: 2048 rows, 28.0 -> 17.2 us)
        float A[8], B[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const long o = (long)min(i0 + i, s.index - 1) * 2 * a.width;
            A[i] = q[o];
            B[i] = q[o + a.width];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i0 + i < s.index) S = mmi_fma(A[i], S, B[i]);
    }
    for (int i0 = 0; i0 < s.n; i0 += 8) {
        float z[8], u[8], g[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const long o = (long)(i0 + i < s.n ? i0 + i : s.n - 1) * 3 * a.width;
            z[i] = p[o];
            u[i] = p[o + 16];
            g[i] = p[o + 32];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (i0 + i < s.n) {
                S = mmi_fma(1.0f - z[i], S, z[i] * u[i]);
                out[tlm_index<Tr>(s.row0 + i0 + i, c, a.out_ks)] = Tr::cvt(S * g[i]);
            }
    }
    if (s.last) a.state[((long)s.slot * 2 + (s.par ^ 1)) * a.width + c] = S;
}

// ------------------------------------------------------------------------------------------------
// sampling helpers
// ------------------------------------------------------------------------------------------------
// greedy: index of the largest logit, the lowest index on ties; out[map[row]] (map: row -> slot)
__global__ __launch_bounds__(256) void k_tlm_argmax(const float* __restrict__ logits, int V, const int* __restrict__ map, int* __restrict__ out,
                                                    int* __restrict__ last_tok) {
    MMI_SHARED float bv[256];
    MMI_SHARED int bi[256];
    const int tid = (int)threadIdx.x;
    const float* p = logits + (long)blockIdx.x * V;
    float best = -INFINITY;
    int at = 0;
    for (int i = tid; i < V; i += 256)
        if (p[i] > best) { best = p[i]; at = i; }
    bv[tid] = best;
    bi[tid] = at;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (tid < s && (bv[tid + s] > bv[tid] || (bv[tid + s] == bv[tid] && bi[tid + s] < bi[tid]))) {
            bv[tid] = bv[tid + s];
            bi[tid] = bi[tid + s];
        }
        __syncthreads();
    }
    if (tid == 0) {
        out[blockIdx.x] = bi[0];
        last_tok[map[blockIdx.x]] = bi[0];
    }
}
// fp32 logits -> the sampler's bf16 rows of ld columns (padding: -inf, never drawn)
__global__ void k_tlm_sample_rows(const float* __restrict__ logits, int V, uint16_t* __restrict__ dst, int ld, int n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)n * ld) return;
    const int c = (int)(i % ld);
    dst[i] = c < V ? mmi_f32_to_bf16(logits[(i / ld) * V + c]) : (uint16_t)0xff80u;
}
__global__ void k_tlm_last_tok(const int* __restrict__ out, const int* __restrict__ map, int* __restrict__ last_tok, int n) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i < n) last_tok[map[i]] = out[i];
}
