// Mimi codec engine behind the C ABI (include/moshi_mi.h): MimiModel.encode / decode in streaming mode
// (reference: moshi/moshi/models/compression.py:338-433) as a fixed per-frame launch list over the kernels
// of mimi_kernels.h, captured into one hipGraph per direction.
#include "mimi_kernels.h"
#include "mmi_graph.h"

#include <math.h>
#include <algorithm>
#include <mutex>

namespace {

struct ConvW {          // one conv / linear as an implicit GEMM: rows = Cout, reduction = Cin*K
    float* wpk = nullptr;
    float* wpk_h = nullptr;   // 1x1 convs: the same matrix packed in the hidden-tile order of k_resblock's second stage
    float* bias = nullptr;
    int Cin = 0, Cout = 0, K = 1, S = 1, Mt = 0, Q = 0;
};

struct LinW {           // a transformer's linear, rows = M (k_pack_lin)
    float* w = nullptr;
    int M = 0, K = 0, J = 0;
};
struct TrLayerW {
    LinW in_proj, out_proj, lin1, lin2;
    float *n1w = nullptr, *n1b = nullptr, *n2w = nullptr, *n2b = nullptr;       // operand order (k_pack_ln)
    float *ls1 = nullptr, *ls2 = nullptr;
};

struct Buf {            // activation buffer [B][C][ld]; first H columns = causal history of its consumer
    float* p = nullptr;
    int C = 0, ld = 0, H = 0;
    int lead = 0;          // floats in front of row 0 (alloc_buf: alignment of the new columns)
    // ELU hoisted into the producers (ConvGemmArgs::elu_out / out2, mimi_kernels.h):
    float* pe = nullptr;   // twin of the same geometry holding ELU(values) - what the ELU-fronted consumer conv reads
    bool elu = false;      // `p` itself holds ELU(values) (no reader wants the raw ones)
    float* conv_src() const { return pe ? pe : p; }                    // what an ELU-fronted conv reads
    bool needs_elu_at_load() const { return !pe && !elu; }
};

// Scratch of a group program (below): one reservation of what the largest program so far needs.  A program is built on what there is; where
// that is too little, the build goes on without launches (`over`) to learn what it needs, and is repeated on a larger reservation.
struct MimiSlab {
    char* base = nullptr;
    size_t size = 0, need = 0;
    bool over = false;
    void* alloc(size_t nb) {
        const size_t at = need;
        need += (nb + 255) & ~(size_t)255;
        over = over || need > size;
        return over ? (char*)this : base + at;         // (not null, which means "none" to the plans; no launch is given it)
    }
    void rewind() { need = 0; over = false; }
    bool release() {                           // false: kept, the runtime does not free while another thread captures
        if (base && hipFree(base) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        base = nullptr;
        size = 0;
        rewind();
        return true;
    }
    void drop() {                              // with the handle: freed now or later
        if (!release()) mmi_free(base);
        base = nullptr;
    }
    hipError_t reserve(size_t nb) {            // never beside the old one: nothing of it may be in flight
        if (!release()) return hipErrorOutOfMemory;
        hipError_t e = mmi_malloc((void**)&base, nb);
        if (e == hipSuccess) size = nb;
        return e;
    }
};

// Where a program's buffers come from: the stream's arena (zeroed, part of the stream's snapshot), or a slab, which holds what it held.
// A group's histories, activations, partial sums and tables are written before they are read; the rows that fill a packed operand's last
// quad up are not (clear_operand): they meet zero weights, but 0 x NaN is NaN.
struct MimiMem {
    MmiArena* arena = nullptr;
    MimiSlab* slab = nullptr;
    int frames = 1;                            // of the program that is built
    hipStream_t stream = nullptr;
    template <class T>
    hipError_t alloc(T** p, size_t n) {
        if (arena) return arena->alloc(p, n);
        *p = (T*)slab->alloc((n ? n : 1) * sizeof(T));
        const char* pz = getenv("MMI_DEBUG_POISON");                          // as in MmiArena::alloc, behind what still runs in the slab
        return pz && (pz[0] == '1' || pz[0] == '0') && there() ? hipMemsetAsync(*p, pz[0] == '1' ? 0xFF : 0x00, (n ? n : 1) * sizeof(T), stream) : hipSuccess;
    }
    bool there() const { return arena || !slab->over; }                       // false: a build that only counts
    template <class T>
    hipError_t zero(T* p, size_t n, hipStream_t s) {
        return !arena || (arena->cut(p) && !getenv("MMI_DEBUG_POISON")) ? hipSuccess : hipMemsetAsync(p, 0, n * sizeof(T), s);      // (a chunk starts zeroed)
    }
    // a packed operand of `tiles` x Q fragments of `deep` reduction indices whose producer stores K rows
    hipError_t clear_operand(float* p, int tiles, int Q, int K, int deep = 8) {
        const size_t n = (size_t)tiles * Q * 256;
        return arena ? zero(p, n, stream) : (Q * deep == K || !there() ? hipSuccess : hipMemsetAsync(p, 0, n * sizeof(float), stream));
    }
};

// operands of the quantiser's launches, `rows` latents at once
struct RvqScratch {
    float* xq = nullptr;                       // 2 x [rows][2*Dq] residuals (first | rest)
    double* best_d = nullptr;                  // 4 x [rows][nchunk] (two of each half)
    int* best_i = nullptr;
    int* codes = nullptr;                      // [rows][n_q]
    float *qin_bp = nullptr, *qin_part = nullptr;
    int rows = 0;
};
struct DequantScratch {
    int* codes = nullptr;                      // [rows][n_q]
    float* q2 = nullptr;                       // [rows][2*Dq]
    float *qout_bp = nullptr, *qout_part = nullptr;
};

// Several consecutive frames of every stream through the network at once: the same launch list as a frame's with `frames` times the
// columns, so that a launch is worth its latency.  The streaming state stays where the frame program keeps it: the histories are copied
// in front of the group's rows before its launches and back behind them, everything else is shared.
// Measured on one stream, 129 frames encoded and decoded (10.3 s of audio): 140 ms frame by frame (176 dependent launches per frame, most of
// them at the ~4.7 us a dependent launch costs; 136 launches and 90 ms now), 2.9 ms in one group of 129.
struct MimiGroup {
    int frames = 0;                            // 0: not built (for this stream)
    bool earlier = false;                      // built for an earlier file, and not used by this one yet
    bool refused = false;                      // building failed (shapes, memory): this stream goes frame by frame
    MimiSlab slab;
    MmiProgram prog;
    Buf in, out;                               // encoder: samples, latents; decoder: latents, samples
    int* codes = nullptr;
    HistTable hist;
};

}  // namespace

struct mmi_mimi {
    int device = -1;                // HIP device the handle lives on (current at create); see MmiDeviceGuard
    int* dec_k_dev = nullptr;       // number of codebooks of the current decode call (read by the captured decoder program)
    int dec_k_host = 0, dec_k_cur = 0;
    mmi_mimi_cfg cfg;
    int max_batch = 0;
    int n_codebooks = 8;
    MmiArena wts;
    // SEANet
    std::vector<ConvW> enc_convs, dec_convs;   // in execution order
    std::vector<TrLayerW> enc_tr, dec_tr;
    ConvW downsample;
    float* upsample_w = nullptr;               // [C][2*stride]
    // RVQ
    ConvW q_in, q_out;                         // stacked first|rest projections
    float* E_all = nullptr;                    // [n_q][bins][D]  (0 = rvq_first.layers.0, 1.. = rvq_rest.layers.*)
    double* e2_all = nullptr;                  // [n_q][bins]
    // RVQ scratch (max_batch rows); the decoder side has its own: an encode of the next frame may run on another stream while a decode
    // is in flight (duplex.hip)
    RvqScratch rvq;
    DequantScratch deq;
    int nchunk = 0;
    // streaming state
    bool streaming = false;
    int batch = 0;
    MmiArena st;
    uint8_t* exec = nullptr;
    uint8_t* first = nullptr;
    long* counters = nullptr;                  // [2][B]: encoder / decoder transformer offsets
    Buf enc_in, latent, dec_codes_lat, dec_out;
    float* enc_kv = nullptr;
    float* dec_kv = nullptr;
    std::vector<float*> partials;              // conv-transpose partial buffers
    std::vector<long> partial_sizes;           // elements per batch row
    HistDesc* enc_hist = nullptr;
    HistDesc* dec_hist = nullptr;
    HistTable enc_tab, dec_tab;                // the same tables on the host
    MimiGroup enc_grp, dec_grp;
    int all_exec = 1;                          // does every stream run?  1: yes, 0: no, -1: what `exec` says (mask_changes, all_run)
    bool mask_in_graph = false;                // a call that changes the mask has been captured: a replay may change it at any time
    int enc_nhist = 0, dec_nhist = 0, enc_hist_rows = 0, dec_hist_rows = 0;
    MmiProgram enc_prog, dec_prog;
    hipStream_t cap_stream = nullptr;
    bool use_graph = true;
    bool parked = false;                       // not streaming; the state and the programs of the last file's stream are still here ...
    int parked_k = 0;                          // ... built for so many codebooks
    bool unfinished = false;                   // the wait behind that stream has failed: work on the device may still use what it has left
};

namespace {

// ---- weight import ---------------------------------------------------------------------------
int need(const MmiWeights& W, const std::string& name, int ndim, const mmi_tensor_desc** out) {
    const mmi_tensor_desc* d = W.find(name);
    if (!d) return mmi_fail(MMI_ERR_MISSING_WEIGHT, "missing weight: " + name);
    if (d->dtype != MMI_F32) return mmi_fail(MMI_ERR_UNSUPPORTED, "Mimi weights must be fp32: " + name);
    if (d->ndim != ndim) return mmi_fail(MMI_ERR_SHAPE, "unexpected rank for " + name);
    *out = d;
    return MMI_OK;
}

int pack_matrix(mmi_mimi* m, const float* W, int M, int Kd, long sm, long sk, ConvW* cw) {
    cw->Mt = mmi_cdiv(M, 32);
    cw->Q = mmi_cdiv(Kd, 8);
    size_t n = (size_t)cw->Mt * cw->Q * 256;
    MMI_HIP_CHECK(m->wts.alloc(&cw->wpk, n));
    int blocks = (int)mmi_cdiv64((int64_t)n, 256);
    MMI_LAUNCH(k_pack_a_f32, blocks, 256, 0, (hipStream_t)0, W, cw->wpk, M, Kd, sm, sk, cw->Mt, cw->Q);
    MMI_CHECK_LAUNCH();
    return MMI_OK;
}

int copy_vec(mmi_mimi* m, const mmi_tensor_desc* d, int n, float** out) {
    MMI_HIP_CHECK(m->wts.alloc(out, (size_t)n));
    MMI_HIP_CHECK(hipMemcpy(*out, d->data, (size_t)n * sizeof(float), hipMemcpyDeviceToDevice));
    return MMI_OK;
}

// nn.Conv1d weight [Cout][Cin][K] (+ bias)
int load_conv(mmi_mimi* m, const MmiWeights& W, const std::string& prefix, int Cin, int Cout, int K, int S, bool bias,
              ConvW* cw) {
    const mmi_tensor_desc* w;
    int rc = need(W, prefix + ".weight", 3, &w);
    if (rc) return rc;
    if (w->shape[0] != Cout || w->shape[1] != Cin || w->shape[2] != K)
        return mmi_fail(MMI_ERR_SHAPE, "shape mismatch for " + prefix + ".weight");
    cw->Cin = Cin; cw->Cout = Cout; cw->K = K; cw->S = S;
    rc = pack_matrix(m, (const float*)w->data, Cout, Cin * K, (long)Cin * K, 1, cw);
    if (rc) return rc;
    if (K == 1) {   // the second conv of a residual block (k_resblock reads its reduction index permuted)
        const size_t n = (size_t)cw->Mt * cw->Q * 256;
        MMI_HIP_CHECK(m->wts.alloc(&cw->wpk_h, n));
        MMI_LAUNCH(k_pack_a_f32_hperm, (int)mmi_cdiv64((int64_t)n, 256), 256, 0, (hipStream_t)0, (const float*)w->data, cw->wpk_h, Cout, Cin,
                   cw->Mt, cw->Q);
        MMI_CHECK_LAUNCH();
    }
    if (bias) {
        const mmi_tensor_desc* b;
        rc = need(W, prefix + ".bias", 1, &b);
        if (rc) return rc;
        if (b->shape[0] != Cout) return mmi_fail(MMI_ERR_SHAPE, "shape mismatch for " + prefix + ".bias");
        rc = copy_vec(m, b, Cout, &cw->bias);
        if (rc) return rc;
    }
    return MMI_OK;
}

// nn.ConvTranspose1d weight [Cin][Cout][K] as a GEMM with rows (co,k): out rows = Cout*K, reduction = Cin
int load_convtr(mmi_mimi* m, const MmiWeights& W, const std::string& prefix, int Cin, int Cout, int K, int S,
                ConvW* cw) {
    const mmi_tensor_desc* w;
    int rc = need(W, prefix + ".weight", 3, &w);
    if (rc) return rc;
    if (w->shape[0] != Cin || w->shape[1] != Cout || w->shape[2] != K)
        return mmi_fail(MMI_ERR_SHAPE, "shape mismatch for " + prefix + ".weight");
    if (K != 2 * S) return mmi_fail(MMI_ERR_UNSUPPORTED, "transposed conv needs kernel == 2*stride: " + prefix);
    cw->Cin = Cin; cw->Cout = Cout * K; cw->K = 1; cw->S = 1;
    rc = pack_matrix(m, (const float*)w->data, Cout * K, Cin, 1, (long)Cout * K, cw);
    if (rc) return rc;
    const mmi_tensor_desc* b;
    rc = need(W, prefix + ".bias", 1, &b);
    if (rc) return rc;
    return copy_vec(m, b, Cout, &cw->bias);
}

// nn.Linear weight [out][in], no bias
int load_linear(mmi_mimi* m, const MmiWeights& W, const std::string& name, int in, int out, LinW* lw) {
    const mmi_tensor_desc* w;
    int rc = need(W, name, 2, &w);
    if (rc) return rc;
    if (w->shape[0] != out || w->shape[1] != in) return mmi_fail(MMI_ERR_SHAPE, "shape mismatch for " + name);
    lw->M = out; lw->K = in; lw->J = mmi_cdiv(in, 16);
    const int Mt = mmi_cdiv(out, 16);
    const size_t n = (size_t)Mt * lw->J * 256;
    MMI_HIP_CHECK(m->wts.alloc(&lw->w, n));
    MMI_LAUNCH(k_pack_lin, (int)mmi_cdiv64((int64_t)n, 256), 256, 0, (hipStream_t)0, (const float*)w->data, lw->w, out, in, Mt, lw->J);
    MMI_CHECK_LAUNCH();
    return MMI_OK;
}

int load_vec(mmi_mimi* m, const MmiWeights& W, const std::string& name, int n, float** out) {
    const mmi_tensor_desc* d;
    int rc = need(W, name, 1, &d);
    if (rc) return rc;
    if (d->shape[0] != n) return mmi_fail(MMI_ERR_SHAPE, "shape mismatch for " + name);
    return copy_vec(m, d, n, out);
}

int load_transformer(mmi_mimi* m, const MmiWeights& W, const std::string& prefix, std::vector<TrLayerW>* layers) {
    const mmi_mimi_cfg& c = m->cfg;
    const int d = c.tr_d_model, ff = c.tr_dim_feedforward;
    layers->resize(c.tr_num_layers);
    for (int l = 0; l < c.tr_num_layers; ++l) {
        TrLayerW& L = (*layers)[l];
        std::string p = prefix + ".transformer.layers." + std::to_string(l);
        int rc;
        if ((rc = load_linear(m, W, p + ".self_attn.in_projs.0.weight", d, 3 * d, &L.in_proj))) return rc;
        if ((rc = load_linear(m, W, p + ".self_attn.out_projs.0.weight", d, d, &L.out_proj))) return rc;
        if ((rc = load_linear(m, W, p + ".linear1.weight", d, ff, &L.lin1))) return rc;
        if ((rc = load_linear(m, W, p + ".linear2.weight", ff, d, &L.lin2))) return rc;
        struct { const char* name; float** dst; } norms[] = {{".norm1.weight", &L.n1w}, {".norm1.bias", &L.n1b}, {".norm2.weight", &L.n2w}, {".norm2.bias", &L.n2b}};
        for (auto& e : norms) {
            float* v = nullptr;
            if ((rc = load_vec(m, W, p + e.name, d, &v))) return rc;
            MMI_HIP_CHECK(m->wts.alloc(e.dst, (size_t)mmi_cdiv(d, 16) * 16));
            MMI_LAUNCH(k_pack_ln, mmi_cdiv(d, 256), 256, 0, (hipStream_t)0, (const float*)v, *e.dst, d & ~15);      // (widths that are no multiple: add_lin)
            MMI_CHECK_LAUNCH();
        }
        if ((rc = load_vec(m, W, p + ".layer_scale_1.scale", d, &L.ls1))) return rc;
        if ((rc = load_vec(m, W, p + ".layer_scale_2.scale", d, &L.ls2))) return rc;
    }
    return MMI_OK;
}

int load_rvq(mmi_mimi* m, const MmiWeights& W) {
    const mmi_mimi_cfg& c = m->cfg;
    const int D = c.q_dimension, dim = c.dimension, bins = c.q_bins, nq = c.q_n_q;
    // stacked input projection [2D][dim]: rows 0..D-1 = rvq_first.input_proj, D..2D-1 = rvq_rest.input_proj
    const mmi_tensor_desc *wf, *wr, *of, *orr;
    int rc;
    if ((rc = need(W, "quantizer.rvq_first.input_proj.weight", 3, &wf))) return rc;
    if ((rc = need(W, "quantizer.rvq_rest.input_proj.weight", 3, &wr))) return rc;
    if ((rc = need(W, "quantizer.rvq_first.output_proj.weight", 3, &of))) return rc;
    if ((rc = need(W, "quantizer.rvq_rest.output_proj.weight", 3, &orr))) return rc;
    if (wf->shape[0] != D || wf->shape[1] != dim || of->shape[0] != dim || of->shape[1] != D)
        return mmi_fail(MMI_ERR_SHAPE, "RVQ projection shape mismatch");
    float* tmp = nullptr;
    MMI_HIP_CHECK(mmi_malloc((void**)&tmp, (size_t)2 * D * dim * sizeof(float)));
    MMI_HIP_CHECK(hipMemcpy(tmp, wf->data, (size_t)D * dim * sizeof(float), hipMemcpyDeviceToDevice));
    MMI_HIP_CHECK(hipMemcpy(tmp + (size_t)D * dim, wr->data, (size_t)D * dim * sizeof(float), hipMemcpyDeviceToDevice));
    m->q_in.Cin = dim; m->q_in.Cout = 2 * D; m->q_in.K = 1; m->q_in.S = 1;
    rc = pack_matrix(m, tmp, 2 * D, dim, dim, 1, &m->q_in);
    if (rc) { mmi_free(tmp); return rc; }
    MMI_HIP_CHECK(hipDeviceSynchronize());
    // stacked output projection [dim][2D]: columns 0..D-1 = first, D..2D-1 = rest
    int blocks = mmi_cdiv(dim * D, 256);
    MMI_LAUNCH(k_copy2d_f32, blocks, 256, 0, (hipStream_t)0, (const float*)of->data, (long)D, tmp, (long)2 * D, dim, D);
    MMI_LAUNCH(k_copy2d_f32, blocks, 256, 0, (hipStream_t)0, (const float*)orr->data, (long)D, tmp + D, (long)2 * D, dim, D);
    MMI_CHECK_LAUNCH();
    m->q_out.Cin = 2 * D; m->q_out.Cout = dim; m->q_out.K = 1; m->q_out.S = 1;
    rc = pack_matrix(m, tmp, dim, 2 * D, 2 * D, 1, &m->q_out);
    MMI_HIP_CHECK(hipDeviceSynchronize());
    mmi_free(tmp);
    if (rc) return rc;

    MMI_HIP_CHECK(m->wts.alloc(&m->E_all, (size_t)nq * bins * D));
    MMI_HIP_CHECK(m->wts.alloc(&m->e2_all, (size_t)nq * bins));
    for (int k = 0; k < nq; ++k) {
        std::string p = k < c.q_n_q_semantic
                            ? "quantizer.rvq_first.vq.layers." + std::to_string(k) + "._codebook."
                            : "quantizer.rvq_rest.vq.layers." + std::to_string(k - c.q_n_q_semantic) + "._codebook.";
        const mmi_tensor_desc *es, *cu;
        if ((rc = need(W, p + "embedding_sum", 2, &es))) return rc;
        if ((rc = need(W, p + "cluster_usage", 1, &cu))) return rc;
        if (es->shape[0] != bins || es->shape[1] != D || cu->shape[0] != bins)
            return mmi_fail(MMI_ERR_SHAPE, "codebook shape mismatch: " + p);
        MMI_LAUNCH(k_codebook_prepare, bins, 64, 0, (hipStream_t)0, (const float*)es->data, (const float*)cu->data,
                   m->E_all + (size_t)k * bins * D, m->e2_all + (size_t)k * bins, bins, D, 1e-5f);
    }
    MMI_CHECK_LAUNCH();
    return MMI_OK;
}

// ---- launch helpers ---------------------------------------------------------------------------
// A conv becomes one of these launch sequences, chosen when the program is built (mimi_kernels.h; the transformers' linears: add_lin):
//   N = B*T_out > 128 columns : k_conv_wide, in groups of frames also k_conv_cols [-> k_conv_finish when K is split over workgroups]
//   N <= 128                  : k_conv_few [-> k_conv_finish], or [k_pack_b_f32] -> k_gemm_f32 [-> k_conv_finish when K is split over workgroups]
struct ConvPlan {
    bool wide = false;
    bool few = false;                 // k_conv_few
    bool cols = false;                // k_conv_cols
    int MTB = 1, W = 1;               // wide
    bool group = false;
    int NSUB = 1, waves = 4, ksplit = 1, nz = 1;
    bool pack = false;
};

template <int MTB, int U, bool ELU_IN, bool GROUP>
void launch_wide_e(hipStream_t s, const ConvGemmArgs& a, int W, dim3 grid) {
    const size_t smem = (size_t)W * MTB * 16 * 64 * sizeof(float);
    switch (W) {
        case 1: MMI_LAUNCH((k_conv_wide<MTB, 1, U, ELU_IN, GROUP>), grid, 64, 0, s, a); break;
        case 2: MMI_LAUNCH((k_conv_wide<MTB, 2, U, ELU_IN, GROUP>), grid, 128, smem, s, a); break;
        case 4: MMI_LAUNCH((k_conv_wide<MTB, 4, U, ELU_IN, GROUP>), grid, 256, smem, s, a); break;
        default: MMI_LAUNCH((k_conv_wide<MTB, 8, U, ELU_IN, GROUP>), grid, 512, smem, s, a); break;
    }
}
template <int MTB, int U>
void launch_wide_w(hipStream_t s, const ConvGemmArgs& a, int W, bool group, dim3 grid) {
    if (group && a.elu_in) launch_wide_e<MTB, U, true, true>(s, a, W, grid);
    else if (group) launch_wide_e<MTB, U, false, true>(s, a, W, grid);
    else if (a.elu_in) launch_wide_e<MTB, U, true, false>(s, a, W, grid);      // ELU at the load (inputs nobody pre-activated)
    else launch_wide_e<MTB, U, false, false>(s, a, W, grid);
}

int launch_conv_plan(hipStream_t s, const ConvGemmArgs& a, const ConvPlan& p) {
    if (p.cols) {
        const dim3 grid(mmi_cdiv(a.Ntot, 128), mmi_cdiv(a.Mt, p.MTB), p.ksplit);
        ConvGemmArgs w = a;
        if (p.ksplit > 1) w.out_mode = MMI_GOUT_PARTIAL;
        const bool fours = mmi_cdiv(w.q_blk, p.W) % 4 == 0;          // (a group ends with its piece)
        if (p.MTB == 4) MMI_LAUNCH((k_conv_cols<4, 2>), grid, 256, 0, s, w, p.W);
        else if (p.MTB == 2 && fours) MMI_LAUNCH((k_conv_cols<2, 4>), grid, 256, 0, s, w, p.W);
        else if (p.MTB == 2) MMI_LAUNCH((k_conv_cols<2, 2>), grid, 256, 0, s, w, p.W);
        else if (fours) MMI_LAUNCH((k_conv_cols<1, 4>), grid, 256, 0, s, w, p.W);
        else MMI_LAUNCH((k_conv_cols<1, 2>), grid, 256, 0, s, w, p.W);
        if (p.ksplit > 1) MMI_LAUNCH(k_conv_finish, (int)mmi_cdiv64((int64_t)a.Cout * a.Ntot, 256), 256, 0, s, a, p.ksplit);
        MMI_CHECK_LAUNCH();
        return MMI_OK;
    }
    if (p.wide) {
        const dim3 grid(mmi_cdiv(a.Ntot, 32), mmi_cdiv(a.Mt, p.MTB), p.ksplit);
        ConvGemmArgs w = a;
        if (p.ksplit > 1) w.out_mode = MMI_GOUT_PARTIAL;
        switch (p.MTB) {
            case 1: launch_wide_w<1, 4>(s, w, p.W, p.group, grid); break;
            case 2: launch_wide_w<2, 4>(s, w, p.W, p.group, grid); break;
            default: launch_wide_w<4, 2>(s, w, p.W, p.group, grid); break;
        }
        if (p.ksplit > 1) MMI_LAUNCH(k_conv_finish, (int)mmi_cdiv64((int64_t)a.Cout * a.Ntot, 256), 256, 0, s, a, p.ksplit);
        MMI_CHECK_LAUNCH();
        return MMI_OK;
    }
    if (p.pack) {
        const long n = (long)mmi_cdiv(a.Ntot, 32) * a.Q * 64;
        MMI_LAUNCH(k_pack_b_f32, (int)mmi_cdiv64(n, 256), 256, 0, s, a, const_cast<float*>(a.bp));
    }
    ConvGemmArgs g = a;
    if (p.ksplit > 1) g.out_mode = MMI_GOUT_PARTIAL;
    const dim3 grid(a.Mt, p.ksplit, p.nz), grid_few(mmi_cdiv(a.Cout, 16), mmi_cdiv(a.Ntot, 16), p.ksplit);
    if (p.few) {
        g.q_blk = mmi_cdiv(a.Q, p.ksplit);
        if (a.x_packed) MMI_LAUNCH((k_conv_few<true, false>), grid_few, p.waves * 64, 0, s, g);
        else if (a.first) MMI_LAUNCH((k_conv_few<false, true>), grid_few, p.waves * 64, 0, s, g);
        else MMI_LAUNCH((k_conv_few<false, false>), grid_few, p.waves * 64, 0, s, g);
    } else if (p.NSUB == 1) {
        if (p.waves == 8) MMI_LAUNCH((k_gemm_f32<1, 8, 2>), grid, 512, 0, s, g);
        else MMI_LAUNCH((k_gemm_f32<1, 4, 2>), grid, 256, 0, s, g);
    } else if (p.NSUB == 2) {
        if (p.waves == 8) MMI_LAUNCH((k_gemm_f32<2, 8, 2>), grid, 512, 0, s, g);
        else MMI_LAUNCH((k_gemm_f32<2, 4, 2>), grid, 256, 0, s, g);
    } else {
        MMI_LAUNCH((k_gemm_f32<4, 4, 2>), grid, 256, 0, s, g);
    }
    if (p.ksplit > 1) MMI_LAUNCH(k_conv_finish, (int)mmi_cdiv64((int64_t)a.Cout * a.Ntot, 256), 256, 0, s, a, p.ksplit);
    MMI_CHECK_LAUNCH();
    return MMI_OK;
}

// k_conv_wide on N columns: m-tiles per wave and waves that split the reduction
void wide_rule(const ConvGemmArgs& a, int N, int* mtb_out, int* w_out) {
    const int nsub = mmi_cdiv(N, 32);
    // m-tiles per wave (each gathered + ELU'd operand element is reused MTB times) vs. waves in flight:
    // aim for >= 1024 waves, taking the parallelism from split-K waves (W) before shrinking MTB
    int MTB = 4;                         // 8 m-tiles per wave needs > 256 registers per lane: one wave per SIMD, slower
    while (MTB > a.Mt) MTB >>= 1;
    int W = 1;
    auto waves = [&](int mtb, int w) { return nsub * mmi_cdiv(a.Mt, mtb) * w; };
    auto wmax = [&](int mtb) { int w = 1; while (w < 8 && w * 2 * mtb <= 16 && a.Q / (w * 2) >= 4) w <<= 1; return w; };
    while (MTB > 1 && waves(MTB, wmax(MTB)) < 1024) MTB >>= 1;
    while (W < wmax(MTB) && waves(MTB, W) < 1024) W <<= 1;
    // Measured tilings of the codec's own layer shapes (profiles/r02_logs/conv_wide_tiling_sweep_b{8,32,64}.txt: every
    // (MTB, W) forced on every layer, per-site times from the kernel trace).  The rule above is within a few percent of the
    // best at 8 sessions but leaves 72 us per frame at 32 sessions and 114 us at 64: what it does not see is the workgroup
    // count against the 256 CUs (a strided conv of 16 column tiles at MTB = 2 is 128 workgroups - half the chip) and the
    // 64-value epilogue of an unsplit MTB = 4 wave.  Shapes not listed (other codecs, other batch classes) keep the rule.
    // Same fp32 results up to summation order (W waves split the reduction), like any other tiling.
    {
        struct Tune { int Cin, Cout, K, S, nsub, MTB, W; };
        static const Tune kTune[] = {
            // 32 sessions (column tiles of the layer at 32 sessions)
            {128, 256, 10, 5, 96, 4, 4},    // enc.down1   45.9 -> 34.1 us
            {256, 512, 12, 6, 16, 1, 8},    // enc.down2   47.4 -> 30.8
            {128, 64, 3, 1, 480, 1, 4},     // resblock 128 ch (enc.res1 / dec.res2), first conv
            {64, 128, 1, 1, 480, 1, 4},     //   second conv                      32.9 -> 31.9, 32.7 -> 31.2
            {256, 128, 3, 1, 96, 1, 4},     // resblock 256 ch (enc.res2 / dec.res1)
            {128, 256, 1, 1, 96, 1, 4},     //                                    24.6 -> 23.3, 26.0 -> 23.0
            {512, 256, 3, 1, 16, 1, 8},     // resblock 512 ch (enc.res3 / dec.res0)
            {256, 512, 1, 1, 16, 1, 8},     //                                    21.4 -> 19.4, 21.9 -> 20.1
            {512, 3072, 1, 1, 16, 1, 8},    // dec.convtr1 (rows = Cout * K)      41.5 -> 34.2 (with its combine)
            {256, 1280, 1, 1, 96, 4, 4},    // dec.convtr2                        49.1 -> 47.0
            {128, 512, 1, 1, 480, 1, 2},    // dec.convtr3                        76.6 -> 55.6
            {64, 1, 7, 1, 1920, 1, 4},      // dec.final                          18.9 -> 16.6
            // 64 sessions
            {128, 256, 10, 5, 192, 2, 8},   // enc.down1   78.2 -> 64.1
            {256, 512, 12, 6, 32, 2, 8},    // enc.down2   54.8 -> 49.0
            {256, 128, 3, 1, 192, 1, 4},    // resblock 256 ch                    42.3 -> 34.9, 41.4 -> 34.1
            {128, 256, 1, 1, 192, 1, 4},
            {512, 256, 3, 1, 32, 1, 8},     // resblock 512 ch                    34.1 -> 22.5, 36.3 -> 22.5
            {256, 512, 1, 1, 32, 1, 8},
            {512, 3072, 1, 1, 32, 1, 8},    // dec.convtr1                        61.1 -> 58.9
            {256, 1280, 1, 1, 192, 4, 4},   // dec.convtr2                       100.2 -> 82.3
            {128, 512, 1, 1, 960, 1, 2},    // dec.convtr3                       128.8 -> 99.5
            {64, 1, 7, 1, 3840, 1, 4},      // dec.final                          31.5 -> 28.1
        };
        for (const Tune& t : kTune)
                if (t.Cin == a.Cin && t.Cout == a.Cout && t.K == a.K && t.S == a.S && 4 * nsub >= 3 * t.nsub && 2 * nsub < 3 * t.nsub) {
                    MTB = t.MTB; W = t.W;
                    while (MTB > a.Mt) MTB >>= 1;
                    break;
                }
    }
    if (const char* e = getenv("MMI_CONV_MTB")) { const int v = atoi(e); if (v == 1 || v == 2 || v == 4) MTB = v; }   // test hooks
    if (const char* e = getenv("MMI_CONV_W")) { const int v = atoi(e); if (v == 1 || v == 2 || v == 4 || v == 8) W = v; }
    while (W * MTB > 16) W >>= 1;          // split-K reduction buffer: W * MTB * 4 KiB of LDS, keep it within 64 KiB
    *mtb_out = MTB; *w_out = W;
}

// k_gemm_f32 on N <= 128 columns: subtiles per workgroup, waves that split the reduction, workgroups that do
void gemm_rule(const ConvGemmArgs& a, int N, ConvPlan* p) {
    const int nsub = mmi_cdiv(N, 32);
    p->NSUB = nsub <= 1 ? 1 : (nsub == 2 ? 2 : 4);
    // small weight matrices (<= 8 MB - the released codec's last encoder conv, resampling, quantiser projections): one workgroup per n-subtile, 4 or 8
    // waves splitting K
    const bool spread = nsub >= 2 && (size_t)a.Mt * a.Q * 1024 <= ((size_t)8 << 20);
    int ks = 1;
    if (a.out_mode == MMI_GOUT_NATURAL) {
        // only the large strided convs (>= 2048-deep reductions, tens of MB of weights) are worth a finishing launch
        while (a.Q >= 256 && ks < 8 && a.Mt * ks * 2 <= 256 && a.Q / (ks * 2) >= 32) ks <<= 1;
    }
    if (const char* e = getenv("MMI_CONV_KSPLIT")) {   // test hook
        const int v = atoi(e);
        if (a.out_mode == MMI_GOUT_NATURAL && v >= 1 && v <= 8 && a.Q >= v) ks = v;
    }
    p->ksplit = ks;
    const int qblk = a.Q / ks;
    if (spread) {
        p->NSUB = 1;
        p->nz = nsub;
        p->waves = qblk >= 16 ? 8 : 4;
    } else {
        p->waves = (p->NSUB <= 2 && qblk >= 32) ? 8 : 4;
    }
}

// Decide the launch sequence of one conv and allocate its scratch (packed operand / partials) from
// `mem`.  `a.x_packed`: the producer writes a.bp itself.
// A group's conv (mem.frames > 1) forms every sum in the order in which the frame program forms it - its reduction is cut into the same
// pieces, over the waves and over the workgroups - so that frames give the same bits however many are run at once; only what each
// workgroup covers follows the group's own number of columns.
int plan_conv(MimiMem& mem, ConvGemmArgs& a, ConvPlan* p) {
    const int N = a.Ntot, N1 = N / mem.frames;
    // (T_shift is the group kernels' alone: a frame's columns divide by fewer than 2^11; inputs are addressed by 32 bits of bytes)
    if ((unsigned long)a.B * (unsigned long)a.x_bstride >= (1ul << 30)) return mmi_fail(MMI_ERR_UNSUPPORTED, "a conv's input of 4 GiB and more: lower max_batch");
    if (a.Cin * a.K >= (1 << 17) || N1 >= (1 << 17) || N >= (1 << 19) || a.T_out / mem.frames >= (1 << 11) || a.K >= (1 << 11))
        return mmi_fail(MMI_ERR_UNSUPPORTED, "conv dimensions outside the range of the kernels' index arithmetic (sessions x samples per frame "
                                             "must stay below 131072: 68 sessions per handle at 1920 samples per frame; a frame below 2048 samples)");
    // (a group's layers that the frame program streams the weights of do so for several column groups, up to 512 columns)
    if (N > (mem.frames > 1 && N1 <= 128 ? 512 : 128)) {
        if (a.first || a.x_packed || a.out_mode != MMI_GOUT_NATURAL)
            return mmi_fail(MMI_ERR_UNSUPPORTED, "more than 128 columns (sessions x time steps per frame) on a conv with replicate padding or packed "
                                                 "operands: lower max_batch (the 25 Hz layers of the released codec take 64 sessions)");
        p->wide = true;
        a.q_blk = a.Q;
        wide_rule(a, N1 > 128 ? N1 : N, &p->MTB, &p->W);
        p->group = mem.frames > 1;
        if (mem.frames > 1) {
            if (N1 <= 128) {
                gemm_rule(a, N1, p);
                p->W = p->waves;
            }
            // as many m-tiles per wave as leave 2048 waves
            p->MTB = 4;
            while (p->MTB > 1 && (p->MTB > a.Mt || p->W * p->MTB > 16 || (long)mmi_cdiv(N, 32) * mmi_cdiv(a.Mt, p->MTB) * p->W * p->ksplit < 2048)) p->MTB >>= 1;
            a.q_blk = mmi_cdiv(a.Q, p->ksplit);
            if (p->ksplit > 1) {
                a.Npad = mmi_cdiv(N, 32) * 32;
                MMI_HIP_CHECK(mem.alloc(&a.partial, (size_t)p->ksplit * a.Mt * 32 * a.Npad));
            }
        }
        // a group's waves each take a whole reduction where there are tiles enough to give most SIMDs one; several m-tiles share a gathered value
        // (128 -> 256, K 10 on 12384 columns with 1, 2, 4 of them: 144, 123, 115 us), except for reductions so short that the stores count (K 32 on
        // 247680: 40 and 52 us).  With fewer tiles the waves of k_conv_wide share a reduction (512 -> 256, K 3 on 2064 columns: 42 against 53 us)
        const long tiles = (long)mmi_cdiv(N, 32) * p->ksplit;
        long enough = 700;
        if (const char* e = getenv("MMI_CONV_COLS")) enough = atol(e);         // test hook: the tiny shapes
        p->cols = mem.frames > 1 && !a.elu_in && tiles * a.Mt >= enough;
        if (p->cols) {
            p->MTB = a.Q < 8 ? 1 : 4;
            while (p->MTB > 1 && (p->MTB > a.Mt || tiles * mmi_cdiv(a.Mt, p->MTB) < enough)) p->MTB >>= 1;
        }
        return MMI_OK;
    }
    p->wide = false;                    // (at most 512 columns: T_shift is 0)
    const int nsub = mmi_cdiv(N, 32);
    gemm_rule(a, N, p);
    a.Npad = (nsub <= 1 ? 1 : (nsub == 2 ? 2 : 4)) * 32;
    if (mem.frames > 1) {
        ConvPlan f;
        gemm_rule(a, N1, &f);
        p->ksplit = f.ksplit;
        p->waves = f.waves;
        if (f.waves == 8 && p->NSUB == 4) p->NSUB = 2;          // (four subtiles of eight waves are not built)
        p->nz = mmi_cdiv(nsub, p->NSUB);
        a.Npad = p->nz * p->NSUB * 32;
    }
    // 16 x 16 tiles while the chip holds them all at once (two workgroups per CU) and a load of 16 columns reaches few streams' rows (a frame of 4
    // streams 778 -> 763 us against the launch that packs in front, of 8 streams 845 -> 847).  With a packed operand there is no such launch to
    // save: only where 32 x 32 tiles leave CUs idle (512 -> 512 on 2 columns 6.1 -> 4.8 us; 1024 -> 8192 on 2 columns 9.4 -> 11.8)
    const long tiles = (long)mmi_cdiv(a.Cout, 16) * mmi_cdiv(N, 16);
    p->few = mem.frames == 1 && !a.elu_in && (a.x_packed ? tiles <= 256 : tiles <= 512 && a.B <= 4) && !getenv("MMI_MIMI_PACK_LAUNCHES");
    if (!a.x_packed && !p->few) {
        if (!a.bp) {
            float* bp = nullptr;
            MMI_HIP_CHECK(mem.alloc(&bp, (size_t)nsub * a.Q * 256));
            a.bp = bp;
        }
        p->pack = true;
    }
    if (p->ksplit > 1 && !a.partial) {
        float* part = nullptr;
        MMI_HIP_CHECK(mem.alloc(&part, (size_t)p->ksplit * a.Mt * 32 * a.Npad));
        a.partial = part;
    }
    return MMI_OK;
}

ConvGemmArgs conv_args(const ConvW& w, const Buf& in, int x_off, int T_out, const Buf& out, int out_off, int B,
                       bool elu_in) {
    ConvGemmArgs a;
    memset(&a, 0, sizeof(a));
    // an ELU-fronted conv reads the producer's pre-activated values when they exist (Buf::pe / Buf::elu)
    a.x = elu_in ? in.conv_src() : in.p;
    if (elu_in && !in.needs_elu_at_load()) elu_in = false;
    a.x_ld = in.ld; a.x_bstride = (long)in.C * in.ld; a.x_off = x_off; a.H = in.H;
    a.wpk = w.wpk; a.bias = w.bias;
    a.out = out.p; a.out_ld = out.ld; a.out_off = out_off;
    a.out2 = out.pe; a.elu_out = out.elu ? 1 : 0;
    a.B = B; a.Cin = w.Cin; a.Cout = w.Cout; a.K = w.K; a.S = w.S; a.T_out = T_out;
    a.T_magic = mmi_div_magic(T_out, mmi_div_shift(T_out)); a.T_shift = mmi_div_shift(T_out); a.K_magic = mmi_div_magic(w.K);
    a.Mt = w.Mt; a.Q = w.Q; a.Ntot = B * T_out;
    a.elu_in = elu_in ? 1 : 0;
    a.out_mode = MMI_GOUT_NATURAL;
    return a;
}

// Audio-rate buffers (T >= 32 new columns per row): the row stride is a multiple of 32 floats and the allocation leads with
// `lead` floats so that the T NEW columns of every row start on a 128-byte line (the H history columns sit right in front of
// them).  A 32-column tile of a conv's output is then exactly one cache line per row: consecutive workgroups run on different
// XCDs (different L2s), and with rows starting at arbitrary 8-byte offsets every line was written in part by two of them.
// MMI_MIMI_NO_ALIGN=1 keeps the dense layout (A/B).  Nothing else knows: every kernel takes (pointer, row stride, H).
int alloc_buf(MimiMem& mem, int B, int C, int H, int T, Buf* b, hipStream_t s) {
    b->C = C; b->H = H; b->ld = H + T; b->lead = 0;
    if (T >= 32 && !getenv("MMI_MIMI_NO_ALIGN")) {
        b->lead = (32 - H % 32) % 32;
        b->ld = ((b->lead + H + T + 31) / 32) * 32;
    }
    size_t n = (size_t)B * C * b->ld + b->lead;
    float* base = nullptr;
    MMI_HIP_CHECK(mem.alloc(&base, n));
    MMI_HIP_CHECK(mem.zero(base, n, s));
    b->p = base + b->lead;
    return MMI_OK;
}

// ELU twin of a buffer (same geometry, zero history: ELU(0) = 0)
int alloc_twin(MimiMem& mem, int B, Buf* b, hipStream_t s) {
    size_t n = (size_t)B * b->C * b->ld + b->lead;
    float* base = nullptr;
    MMI_HIP_CHECK(mem.alloc(&base, n));
    MMI_HIP_CHECK(mem.zero(base, n, s));
    b->pe = base + b->lead;
    return MMI_OK;
}

// the history a consumer conv reads lives in the buffer it reads: the ELU twin when there is one
HistDesc hist_of(const Buf& b, int T);
HistDesc hist_of_src(const Buf& b, int T) {
    Buf c = b;
    c.p = b.conv_src();
    return hist_of(c, T);
}

int add_conv(MimiMem& mem, MmiProgram& prog, ConvGemmArgs a) {
    ConvPlan p;
    int rc = plan_conv(mem, a, &p);
    if (rc) return rc;
    prog.add([a, p](hipStream_t s) { return launch_conv_plan(s, a, p); });
    return MMI_OK;
}

// SEANet residual block (conv K -> hidden, conv 1x1 -> channels, + input): ONE launch (k_resblock) at audio rate when the block
// has the shape the kernel is built for and enough columns to fill the chip with 32-column workgroups; else the two convs.
int add_resblock(MimiMem& mem, MmiProgram& prog, ConvGemmArgs a1, ConvGemmArgs a2, const ConvW& w2) {
    const int nblk = mmi_cdiv(a1.Ntot, 32);
    long min_waves = 256;                        // below that the two-launch path (split-K over waves) fills the chip better
    if (const char* e = getenv("MMI_MIMI_RES_FUSION_MIN")) min_waves = atol(e);      // test hook: the tiny shapes
    // Measured on MI355X (profiles/r02_logs/resblock_*): the 64-channel blocks (one hidden tile, 1920 one-wave workgroups) gain
    // 8-13 us each over two launches; the 128 / 256-channel blocks (480 / 96 workgroups of 2 / 4 waves: one wave per SIMD on part of
    // the chip) lost 2-15 us to the two-launch path's split-K over waves and are not instantiated.
    const bool fuse = a1.Ntot / mem.frames > 128 && a1.S == 1 && a2.K == 1 && a2.S == 1 && a1.Cout == a2.Cin && a1.Ntot == a2.Ntot &&
                      a1.T_out == a2.T_out && a1.Mt == 1 && w2.wpk_h && a2.Q <= 4 * a1.Mt &&
                      a2.Mt >= a1.Mt && (long)mmi_cdiv(a1.Ntot / mem.frames, 32) * a1.Mt >= min_waves && !a1.first && !a2.first && !a1.res &&
                      a1.T_out / mem.frames % 32 == 0 && a1.Cin <= 64 * a1.Mt && a1.K <= 33;
    if (!fuse) {
        int rc = add_conv(mem, prog, a1);
        if (rc) return rc;
        return add_conv(mem, prog, a2);
    }
    a2.wpk = w2.wpk_h;
    a2.elu_in = 0;                               // the hidden tensor never exists un-activated
    ResBlockArgs ra;
    ra.a1 = a1; ra.a2 = a2;
    const int mt1 = a1.Mt;
    // LDS: input window Cin x (32 + K - 1) | offset table | the waves' hand-off mailbox
    const size_t smem = ((size_t)((a1.Cin * (32 + a1.K - 1) + 3) & ~3) + (size_t)a1.Q * 8 + (mt1 > 1 ? (size_t)mt1 * 1024 : 0)) * sizeof(float);
    if (smem > 65536) return mmi_fail(MMI_ERR_UNSUPPORTED, "k_resblock: input window does not fit in LDS");
    const bool group = mem.frames > 1;
    prog.add([ra, nblk, smem, group](hipStream_t s) {
        if (group) MMI_LAUNCH((k_resblock<1, 4, true>), nblk, 64, smem, s, ra);
        else MMI_LAUNCH((k_resblock<1, 4, false>), nblk, 64, smem, s, ra);
        MMI_CHECK_LAUNCH();
        return (int)MMI_OK;
    });
    return MMI_OK;
}

// residual vector quantiser: latent [B][dim] (column `lat_off` of rows of length lat_ld) -> r.codes [B][n_q]
// latent_packed: the producer of the latent also wrote it as the packed operand r.qin_bp (ConvGemmArgs::outp): no pack launch
int add_quantize_ops(mmi_mimi* m, MimiMem& mem, const RvqScratch& r, MmiProgram& prog, const float* latent, int lat_ld, int lat_off, int B,
                     bool latent_packed = false) {
    const mmi_mimi_cfg& c = m->cfg;
    const int D = c.q_dimension, bins = c.q_bins;
    Buf in; in.p = const_cast<float*>(latent); in.C = c.dimension; in.ld = lat_ld; in.H = lat_off;
    Buf out; out.p = r.xq; out.C = 2 * D; out.ld = 1; out.H = 0;
    {
        ConvGemmArgs a = conv_args(m->q_in, in, lat_off, 1, out, 0, B, false);
        a.bp = r.qin_bp; a.partial = r.qin_part;
        a.x_packed = latent_packed ? 1 : 0;
        int rc = add_conv(mem, prog, a);
        if (rc) return rc;
    }
    const int K = m->n_codebooks;
    const int nchunk = m->nchunk;
    const size_t smem = (size_t)8 * D * sizeof(double);
    int depth[2] = {0, 0};                                // levels of the acoustic / semantic half so far
    // the next level of its half: two buffers of residuals and two of chunk winners, one read and one written by a launch
    auto level = [&](int k, bool sem) {
        const int n = depth[sem]++;
        const auto buf = [&](int i) { return r.xq + (size_t)(i & 1) * r.rows * 2 * D + (sem ? 0 : D); };
        const auto slot = [&](int i) { return (size_t)((sem ? 2 : 0) + (i & 1)) * nchunk * r.rows; };
        RvqLevel L;
        memset(&L, 0, sizeof(L));
        L.x = buf(n > 0 ? n - 1 : 0); L.x_next = buf(n);
        L.best_d = r.best_d + slot(n); L.best_i = r.best_i + slot(n);
        L.E = m->E_all + (size_t)k * bins * D;
        L.e2 = m->e2_all + (size_t)k * bins;
        if (n > 0) {
            L.prev_E = L.E - (size_t)bins * D;
            L.prev_d = r.best_d + slot(n - 1); L.prev_i = r.best_i + slot(n - 1);
            L.prev_level = k - 1;
        }
        return L;
    };
    int* codes = r.codes; const int nq = c.q_n_q;
    // rows per workgroup: as few as leave the chip two workgroups per CU (32 rows: 9.0 us with 8, 8.0 with 4); more of them share a code's load
    int group = 1;
    while (group < 8 && (long)nchunk * mmi_cdiv(B, group) > 512) group *= 2;
    // the semantic quantiser's single level and the first acoustic level share a launch (independent, see RvqLevel)
    const bool pair = c.q_n_q_semantic == 1 && K >= 2 && !getenv("MMI_RVQ_NO_PAIR");
    for (int k = 0; k < K; ++k) {
        const RvqLevel a0 = level(k, k < c.q_n_q_semantic);
        const bool two = pair && k == 0;
        const RvqLevel a1 = two ? level(++k, false) : a0;
        const int nz = two ? 2 : 1;
        prog.add([=](hipStream_t s) {
            MMI_LAUNCH(k_rvq_level, dim3(nchunk, mmi_cdiv(B, group), nz), 256, smem, s, a0, a1, 2 * D, B, group, D, bins, nchunk, codes, nq);
            MMI_CHECK_LAUNCH();
            return (int)MMI_OK;
        });
    }
    RvqLevel end[2];
    int ends = 0;
    for (int sem = 0; sem < 2; ++sem)
        if (depth[sem] > 0) end[ends++] = level(sem ? std::min(K, c.q_n_q_semantic) : K, sem);       // (its prev_* is the half's last level)
    const RvqLevel e0 = end[0], e1 = end[ends > 1 ? 1 : 0];
    prog.add([=](hipStream_t s) {
        MMI_LAUNCH(k_rvq_last, dim3(mmi_cdiv(B, 4), ends), 256, 0, s, e0, e1, B, nchunk, codes, nq);
        MMI_CHECK_LAUNCH();
        return (int)MMI_OK;
    });
    return MMI_OK;
}

// d.codes [B * T][n_q] (first K used; row b * T + t) -> latents t of stream b, written to out buffer column out_off + t
// k_from_device: the streaming decoder's captured program (K of each call comes from m->dec_k_dev); the one-shot programs of
// decode_latent bake their K in
int add_dequant_ops(mmi_mimi* m, MimiMem& mem, const DequantScratch& d, MmiProgram& prog, int K, const Buf& out, int out_off, int B, int T = 1,
                    bool k_from_device = false) {
    const mmi_mimi_cfg& c = m->cfg;
    const int D = c.q_dimension, bins = c.q_bins, nq = c.q_n_q, nsem = c.q_n_q_semantic, rows = B * T;
    float* q2 = d.q2; const int* codes = d.codes; const float* E = m->E_all; const int* kdev = k_from_device ? m->dec_k_dev : nullptr;
    const bool packed = (rows <= 128 || T > 1) && m->q_out.Q * 8 == 2 * D && !getenv("MMI_MIMI_PACK_LAUNCHES");
    if (T > 1 && !packed) return mmi_fail(MMI_ERR_UNSUPPORTED, "dequantising several frames needs the packed operand");
    float* qp = packed ? d.qout_bp : nullptr; const int qQ = m->q_out.Q;
    prog.add([=](hipStream_t s) {
        MMI_LAUNCH(k_rvq_gather, mmi_cdiv(rows * D, 64), 64, 0, s, codes, nq, K, E, bins, D, nsem, q2, rows, kdev, qp, qQ);
        MMI_CHECK_LAUNCH();
        return (int)MMI_OK;
    });
    Buf in; in.p = d.q2; in.C = 2 * D; in.ld = 1; in.H = 0;
    ConvGemmArgs a = conv_args(m->q_out, in, 0, T, out, out_off, B, false);
    a.bp = d.qout_bp; a.partial = d.qout_part;
    a.x_packed = packed ? 1 : 0;                 // the gather wrote the operand
    return add_conv(mem, prog, a);
}

// the residual stream of a transformer as its linears' operand (mmi_lin_index); who produces the stream's input stores it there
struct TrStream { float* p = nullptr; int J = 0; };
int alloc_tr_stream(mmi_mimi* m, MimiMem& mem, int N, TrStream* x) {
    const int d = m->cfg.tr_d_model;
    x->J = mmi_cdiv(d, 16);
    MMI_HIP_CHECK(mem.alloc(&x->p, (size_t)mmi_cdiv(N, 16) * x->J * 256));
    MMI_HIP_CHECK(mem.clear_operand(x->p, mmi_cdiv(N, 16), x->J, d, 16));
    return MMI_OK;
}

template <int FM, int FN, int U, bool NT>
void launch_lin(hipStream_t s, const MimiLinArgs& a) {
    MMI_LAUNCH((k_mimi_lin<FM, FN, U, false, NT>), dim3(mmi_cdiv(a.M, 16 * FM) << (FM == 1 ? a.share : 0), mmi_cdiv(a.N, 16 * FN)), 512, 0, s, a);
}
template <int FM, int FN, bool NT>
void launch_lin_norm(hipStream_t s, const MimiLinArgs& a) {
    const dim3 grid(mmi_cdiv(a.M, 16 * FM) << (FM == 1 ? a.share : 0), mmi_cdiv(a.N, 16 * FN));
    if (a.J <= 32) MMI_LAUNCH((k_mimi_lin<FM, FN, 4, true, NT>), grid, 512, 0, s, a);
    else MMI_LAUNCH((k_mimi_lin<FM, FN, 8, true, NT>), grid, 512, 0, s, a);
}

int add_lin(MmiProgram& prog, MimiLinArgs a, int K) {
    if (a.ln_w && (a.J > 64 || a.J * 16 != K)) return mmi_fail(MMI_ERR_UNSUPPORTED, "Mimi transformer: a width of at most 1024, a multiple of 16");
    // 16 x 16 tiles while the chip holds all workgroups at once (two per CU); with a norm 32 rows share it from 256 tiles on (32 streams 1203 -> 1186
    // us a frame; with 192 - 256 tiles, 16 streams, 973 -> 1000).  Beyond that 32 x 32 in rings of four fragments (258 columns, K = 2048: 17.5 -> 13.0
    // us, 16 x 16 13.9), with a norm 128 rows per workgroup where those fill half the chip.  Rings of 4 fragments, of 8 for long reductions: with K = 512 a wave
    // has 4 (groups of 4 against 8: one stream 717 -> 688 us a frame, 16 streams 973 -> 946).  Weights that one tile of columns reads leave no line behind, others' are read
    // again (32 streams 1211 -> 1201 us).
    const long tiles = (long)mmi_cdiv(a.M, 16) * mmi_cdiv(a.N, 16);
    const bool rows = a.ln_w && a.J <= 60 && (long)mmi_cdiv(a.M, 128) * mmi_cdiv(a.N, 16) >= 128;      // (J KB of LDS and a little more, below 64)
    int waves = 8;                                           // more of them where that gives every workgroup a CU of its own (2048 x 258: 19.5 -> 15.6 us)
    while (waves < 12 && (long)mmi_cdiv(a.M, 16 * waves) * mmi_cdiv(a.N, 16) > 256) ++waves;
    if ((long)mmi_cdiv(a.M, 16 * waves) * mmi_cdiv(a.N, 16) > 256) waves = 8;
    // two workgroups to a tile of a long reduction while that is one per CU: us a frame of 1, 4, 8, 16, 32 streams 671, 707, 790, 911, 1112 -> 669, 705, 780, 904,
    // 1104 (four: 672, 709, 784, 905, 1108; short reductions and those with a norm, shared likewise: no faster)
    a.share = !a.ln_w && a.J > 32 && 2 * tiles <= 256 ? 1 : 0;
    prog.add([=](hipStream_t s) {
        if (rows) {
            const dim3 grid(mmi_cdiv(a.M, 16 * waves), mmi_cdiv(a.N, 16));
            const size_t smem = (size_t)a.J * 64 * sizeof(f32x4);
            if (a.J <= 32) MMI_LAUNCH((k_mimi_lin_rows<4>), grid, 64 * waves, smem, s, a);
            else MMI_LAUNCH((k_mimi_lin_rows<8>), grid, 64 * waves, smem, s, a);
        } else if (!a.ln_w) {
            if (a.N <= 16 && a.J > 32) launch_lin<1, 1, 8, true>(s, a);
            else if (a.N <= 16) launch_lin<1, 1, 4, true>(s, a);
            else if (tiles <= 512 && a.J > 32) launch_lin<1, 1, 8, false>(s, a);
            else if (tiles <= 512) launch_lin<1, 1, 4, false>(s, a);
            else launch_lin<2, 2, 4, false>(s, a);
        } else {
            if (a.N <= 16 && tiles <= 512) launch_lin_norm<1, 1, true>(s, a);
            else if (tiles <= 256) launch_lin_norm<1, 1, false>(s, a);
            else if (tiles <= 512) launch_lin_norm<2, 1, false>(s, a);
            else launch_lin_norm<1, 2, false>(s, a);
        }
        MMI_CHECK_LAUNCH();
        return (int)MMI_OK;
    });
    return MMI_OK;
}

// one streaming transformer (ProjectedTransformer with conv_layout, transformer.py:932-983) on the residual stream x, whose result goes to
// buf[:, :, off:off+T] as well, T = frames * (steps per frame)
int add_transformer(mmi_mimi* m, MimiMem& mem, MmiProgram& prog, const std::vector<TrLayerW>& layers, const TrStream& x, const Buf& xb, int off, int T,
                    float* kv, const long* offsets, int B, int frames, hipStream_t init_stream) {
    const mmi_mimi_cfg& c = m->cfg;
    const int d = c.tr_d_model, H = c.tr_num_heads, Dh = d / H, ff = c.tr_dim_feedforward, cap = c.tr_context;
    const int N = B * T;
    Buf qkv;
    int rc;
    if ((rc = alloc_buf(mem, B, 3 * d, 0, T, &qkv, init_stream))) return rc;
    float *attp = nullptr, *hbp = nullptr;
    const int nt = mmi_cdiv(N, 16), Jd = x.J, Jff = mmi_cdiv(ff, 16);
    MMI_HIP_CHECK(mem.alloc(&attp, (size_t)nt * Jd * 256));
    MMI_HIP_CHECK(mem.alloc(&hbp, (size_t)nt * Jff * 256));
    MMI_HIP_CHECK(mem.clear_operand(attp, nt, Jd, d, 16));
    MMI_HIP_CHECK(mem.clear_operand(hbp, nt, Jff, ff, 16));
    const size_t kv_layer = (size_t)B * H * cap * Dh;
    if (T / frames > 2 || (Dh != 16 && Dh != 32 && Dh != 64))
        return mmi_fail(MMI_ERR_UNSUPPORTED, "Mimi attention: head dim 16/32/64 and 1 or 2 steps per frame are built");
    const size_t attn_smem = ((size_t)T * Dh + (((size_t)T * cap + 3) & ~(size_t)3) + (size_t)(256 / (Dh / 4)) * T * Dh + 8) * sizeof(float);
    // one memory round trip when a thread's 8 row slots cover the ring (the Mimi shape: 250 slots of 64 floats)
    const bool one_pass = cap <= 8 * (512 / (Dh / 4)) && !getenv("MMI_MIMI_ATTN_TWO_PASS");
    // several frames at once: queries, keys and values row by row (the layers' keys and values until the ring takes them all at the end)
    const size_t rows_d = (size_t)B * H * T * Dh;
    float *qr = nullptr, *kvn = nullptr;
    if (frames > 1) {
        if (!one_pass) return mmi_fail(MMI_ERR_UNSUPPORTED, "Mimi attention: a too long context for several frames at once");
        MMI_HIP_CHECK(mem.alloc(&qr, rows_d));
        MMI_HIP_CHECK(mem.alloc(&kvn, 2 * rows_d * layers.size()));
    }
    auto lin = [&](const LinW& w, const float* in, int mode) {
        MimiLinArgs a;
        memset(&a, 0, sizeof(a));
        a.w = w.w; a.x = in; a.M = w.M; a.N = N; a.J = w.J; a.mode = mode;
        a.T = T; a.T_shift = mmi_div_shift(T); a.T_magic = mmi_div_magic(T, a.T_shift);
        a.ln_eps = 1e-5f;
        return a;
    };
    for (size_t l = 0; l < layers.size(); ++l) {
        const TrLayerW& L = layers[l];
        {   // x = x + ls1 * out_proj(attn(norm1(x)))
            MimiLinArgs ai = lin(L.in_proj, x.p, MIMI_LIN_ROWS);
            ai.ln_w = L.n1w; ai.ln_b = L.n1b;
            ai.out = qkv.p; ai.out_ld = qkv.ld;
            if ((rc = add_lin(prog, ai, L.in_proj.K))) return rc;
            MimiAttnArgs aa;
            aa.qkv = qkv.p; aa.kc = kv + (2 * l) * kv_layer; aa.vc = kv + (2 * l + 1) * kv_layer;
            aa.offsets = offsets; aa.B = B; aa.H = H; aa.D = Dh; aa.T = T; aa.cap = cap;
            aa.context = c.tr_context; aa.max_period = c.tr_max_period;
            aa.outp = attp; aa.outJ = Jd;
            if (frames > 1) {
                MimiGroupRows gr;
                gr.T = T; gr.qkv_ld = qkv.ld; gr.q = qr; gr.kn = kvn + 2 * l * rows_d; gr.vn = gr.kn + rows_d;
                const int tpf = T / frames;
                const dim3 grid_r(B * H, mmi_cdiv(T, MIMI_ROPE_T)), grid_a(B * H, frames);
                prog.add([=](hipStream_t s) {
#define MMI_ATT(D_, T_) do { MMI_LAUNCH((k_mimi_group_rope<D_>), grid_r, 256, 0, s, aa, gr); \
                             MMI_LAUNCH((k_mimi_attn_1pass<D_, T_, true>), grid_a, 512, 0, s, aa, gr); } while (0)
                    if (Dh == 64 && tpf == 2) MMI_ATT(64, 2);
                    else if (Dh == 64) MMI_ATT(64, 1);
                    else if (Dh == 32 && tpf == 2) MMI_ATT(32, 2);
                    else if (Dh == 32) MMI_ATT(32, 1);
                    else if (tpf == 2) MMI_ATT(16, 2);
                    else MMI_ATT(16, 1);
#undef MMI_ATT
                    MMI_CHECK_LAUNCH();
                    return (int)MMI_OK;
                });
            } else prog.add([=](hipStream_t s) {
#define MMI_ATT(D_, T_) do { if (one_pass) MMI_LAUNCH((k_mimi_attn_1pass<D_, T_>), B * H, 512, 0, s, aa, MimiGroupRows()); \
                             else MMI_LAUNCH((k_mimi_attn<D_, T_>), B * H, 256, attn_smem, s, aa); } while (0)
                if (Dh == 64 && T == 2) MMI_ATT(64, 2);
                else if (Dh == 64 && T == 1) MMI_ATT(64, 1);
                else if (Dh == 32 && T == 2) MMI_ATT(32, 2);
                else if (Dh == 32 && T == 1) MMI_ATT(32, 1);
                else if (Dh == 16 && T == 2) MMI_ATT(16, 2);
                else if (Dh == 16 && T == 1) MMI_ATT(16, 1);
                else return mmi_fail(MMI_ERR_UNSUPPORTED, "Mimi attention: head dim 16/32/64 and 1 or 2 steps per frame are built");
#undef MMI_ATT
                MMI_CHECK_LAUNCH();
                return (int)MMI_OK;
            });
            MimiLinArgs a = lin(L.out_proj, attp, MIMI_LIN_RESID);
            a.outp = x.p; a.outJ = x.J; a.scale = L.ls1;
            if ((rc = add_lin(prog, a, L.out_proj.K))) return rc;
        }
        {   // x = x + ls2 * linear2(gelu(linear1(norm2(x))))
            MimiLinArgs a1 = lin(L.lin1, x.p, MIMI_LIN_GELU);
            a1.ln_w = L.n2w; a1.ln_b = L.n2b;
            a1.outp = hbp; a1.outJ = Jff;
            if ((rc = add_lin(prog, a1, L.lin1.K))) return rc;
            MimiLinArgs a2 = lin(L.lin2, hbp, MIMI_LIN_RESID);
            a2.outp = x.p; a2.outJ = x.J; a2.scale = L.ls2;
            if (l + 1 == layers.size()) { a2.out = xb.p; a2.out_ld = xb.ld; a2.out_off = off; }      // what the convs behind read
            if ((rc = add_lin(prog, a2, L.lin2.K))) return rc;
        }
    }
    if (frames > 1) {
        const int L = (int)layers.size();
        const long n = (long)L * 2 * B * H * (T < cap ? T : cap) * (Dh / 4);
        prog.add([=](hipStream_t s) {
            MMI_LAUNCH(k_mimi_group_ring, (int)mmi_cdiv64(n, 256), 256, 0, s, (const float*)kvn, kv, offsets, L, B, H, T, cap, Dh);
            MMI_CHECK_LAUNCH();
            return (int)MMI_OK;
        });
    }
    return MMI_OK;
}

// the table by value (n = -1: too many descriptors for it); returns the rows of all buffers
int make_hist(std::vector<HistDesc>& h, int B, HistTable* tab) {
    int acc = 0;
    memset(tab, 0, sizeof(*tab));
    for (auto& d : h) {
        if (d.H <= 0) continue;
        d.row_begin = acc;
        acc += B * d.C;
        if (tab->n >= 0 && tab->n < MMI_HIST_MAX) tab->d[tab->n++] = d;
        else tab->n = -1;
    }
    return acc;
}

int upload_hist(mmi_mimi* m, std::vector<HistDesc>& h, int B, HistDesc** dev, int* n, int* rows, HistTable* tab) {
    *rows = make_hist(h, B, tab);
    std::vector<HistDesc> keep;
    for (auto& d : h)
        if (d.H > 0) keep.push_back(d);
    *n = (int)keep.size();
    MMI_HIP_CHECK(m->st.alloc(dev, keep.size() ? keep.size() : 1));
    m->st.own.push_back(*dev);
    if (!keep.empty())
        MMI_HIP_CHECK(hipMemcpy(*dev, keep.data(), keep.size() * sizeof(HistDesc), hipMemcpyHostToDevice));
    return MMI_OK;
}

HistDesc hist_of(const Buf& b, int T) {
    HistDesc d;
    d.p = b.p; d.C = b.C; d.ld = b.ld; d.H = b.H; d.T = T; d.row_begin = 0;
    return d;
}

// the end of a program: histories shifted, transformer offsets advanced, replicate flags cleared
int add_commit(mmi_mimi* m, MmiProgram& prog, std::vector<HistDesc>& hist, int B, const MimiGroup* g, HistDesc** dev, int* n, int* n_rows, HistTable* tab,
               long* counters, int inc, uint8_t* first) {
    int rc, rows;
    if (g) {
        rows = make_hist(hist, B, tab);
        if (tab->n < 0) return mmi_fail(MMI_ERR_UNSUPPORTED, "too many histories for several frames at once");
    } else {
        if ((rc = upload_hist(m, hist, B, dev, n, n_rows, tab))) return rc;
        rows = *n_rows;
    }
    const HistDesc* hd = *dev;
    const int nh = *n;
    const HistTable t = *tab;
    const uint8_t* ex = m->exec;
    const bool one = t.n >= 0 && (g || !getenv("MMI_MIMI_TWO_COMMITS"));
    prog.add([=](hipStream_t s) {
        if (one) {
            MMI_LAUNCH(k_commit_all, mmi_cdiv(rows + B, 256), 256, 0, s, t, rows, ex, counters, 1, inc, first, B);
            MMI_CHECK_LAUNCH();
            return (int)MMI_OK;
        }
        if (rows > 0) MMI_LAUNCH(k_commit_history, mmi_cdiv(rows, 256), 256, 0, s, hd, nh, rows, ex);
        MMI_LAUNCH(k_commit_counters, mmi_cdiv(B, 64), 64, 0, s, counters, 1, inc, first, ex, B);
        MMI_CHECK_LAUNCH();
        return (int)MMI_OK;
    });
    return MMI_OK;
}

// g: null for the frame program, whose buffers and state are the stream's; otherwise `frames` frames at once in the group's own buffers
int build_encoder(mmi_mimi* m, int B, int frames, MimiMem& mem, MimiGroup* g, hipStream_t s0) {
    const mmi_mimi_cfg& c = m->cfg;
    MmiProgram& prog = g ? g->prog : m->enc_prog;
    Buf &ein = g ? g->in : m->enc_in, &lat = g ? g->out : m->latent;
    std::vector<HistDesc> hist;
    int rc;
    int T = c.frame_size * frames;
    size_t ci = 0;
    // input PCM buffer with the first conv's history
    if ((rc = alloc_buf(mem, B, c.channels, c.kernel_size - 1, T, &ein, s0))) return rc;
    hist.push_back(hist_of(ein, T));
    Buf cur = ein;
    int mult = 1;
    // ELU hoisted into the producers (mimi_kernels.h ConvGemmArgs::elu_out / out2): a resblock input is kept raw (residual) AND
    // ELU'd (its first conv reads that, history included); everything else a conv reads through ELU is stored ELU'd only
    {   // conv0: channels -> n_filters, K = kernel_size; consumer = resblock conv (K = residual_kernel_size)
        Buf nxt;
        if ((rc = alloc_buf(mem, B, c.n_filters, c.residual_kernel_size - 1, T, &nxt, s0))) return rc;
        if ((rc = alloc_twin(mem, B, &nxt, s0))) return rc;
        prog.site("enc.conv0");
        if ((rc = add_conv(mem, prog, conv_args(m->enc_convs[ci++], cur, 0, T, nxt, nxt.H, B, false)))) return rc;
        hist.push_back(hist_of_src(nxt, T));
        cur = nxt;
    }
    for (int i = 0; i < c.n_ratios; ++i) {
        const int ratio = c.ratios[c.n_ratios - 1 - i];
        const int ch = mult * c.n_filters;
        // resblock: cur -> (ELU, conv K3 -> hidden) -> (ELU, conv K1 -> ch) + cur ; consumer = strided conv (K=2r, S=r)
        Buf hid, nxt;
        if ((rc = alloc_buf(mem, B, ch / c.compress, 0, T, &hid, s0))) return rc;
        if ((rc = alloc_buf(mem, B, ch, ratio, T, &nxt, s0))) return rc;
        hid.elu = nxt.elu = true;               // read only by the block's second conv / the strided conv, both behind an ELU
        prog.site("enc.res" + std::to_string(i));
        const ConvGemmArgs a1 = conv_args(m->enc_convs[ci++], cur, 0, T, hid, 0, B, true);
        const ConvW& w2 = m->enc_convs[ci++];
        ConvGemmArgs a = conv_args(w2, hid, 0, T, nxt, nxt.H, B, true);
        a.res = cur.p; a.res_ld = cur.ld; a.res_off = cur.H;
        if ((rc = add_resblock(mem, prog, a1, a, w2))) return rc;
        hist.push_back(hist_of(nxt, T));
        cur = nxt;
        // strided conv: ch -> 2ch ; consumer = next resblock conv (K3) or the final conv (last_kernel_size)
        const int Tn = T / ratio;
        const int Hn = (i + 1 < c.n_ratios) ? c.residual_kernel_size - 1 : c.last_kernel_size - 1;
        Buf nx2;
        if ((rc = alloc_buf(mem, B, 2 * ch, Hn, Tn, &nx2, s0))) return rc;
        if (i + 1 < c.n_ratios) { if ((rc = alloc_twin(mem, B, &nx2, s0))) return rc; }   // the next resblock's input
        else nx2.elu = true;                                                                     // read by the final conv only
        prog.site("enc.down" + std::to_string(i));
        if ((rc = add_conv(mem, prog, conv_args(m->enc_convs[ci++], cur, 0, Tn, nx2, nx2.H, B, true)))) return rc;
        hist.push_back(hist_of_src(nx2, Tn));
        cur = nx2;
        T = Tn;
        mult *= 2;
    }
    // final conv -> dimension, written into the downsample conv's input buffer (history = stride)
    const int stride = c.resample_stride;
    Buf dsin;
    if ((rc = alloc_buf(mem, B, c.dimension, 2 * stride - stride, T, &dsin, s0))) return rc;
    TrStream xs;
    if ((rc = alloc_tr_stream(m, mem, B * T, &xs))) return rc;
    prog.site("enc.final");
    {
        ConvGemmArgs a = conv_args(m->enc_convs[ci++], cur, 0, T, dsin, dsin.H, B, true);
        a.outp = xs.p; a.outJ = xs.J;
        if ((rc = add_conv(mem, prog, a))) return rc;
    }
    hist.push_back(hist_of(dsin, T));
    // encoder transformer, its result in dsin[:, :, H:H+T]
    {
        const int Dh = c.tr_d_model / c.tr_num_heads;
        size_t kvn = (size_t)2 * c.tr_num_layers * B * c.tr_num_heads * c.tr_context * Dh;
        if (!g) {
            MMI_HIP_CHECK(m->st.alloc(&m->enc_kv, kvn));
            MMI_HIP_CHECK(mem.zero(m->enc_kv, kvn, s0));
        }
        prog.site("enc.tr");
        if ((rc = add_transformer(m, mem, prog, m->enc_tr, xs, dsin, dsin.H, T, m->enc_kv, m->counters, B, frames, s0))) return rc;
    }
    const int T_tr = T;
    // downsample (ConvDownsample1d learnt, replicate padding on the first frame)
    if (T % stride != 0 || T / stride != frames)
        return mmi_fail(MMI_ERR_UNSUPPORTED, "frame_size must map to exactly one latent column");
    if ((rc = alloc_buf(mem, B, c.dimension, 0, frames, &lat, s0))) return rc;
    const bool latent_packed = (B <= 128 || g) && m->q_in.Q * 8 == c.dimension && !getenv("MMI_MIMI_PACK_LAUNCHES");
    if (g && !latent_packed) return mmi_fail(MMI_ERR_UNSUPPORTED, "quantising several frames needs the packed operand");
    RvqScratch rs = m->rvq;
    if (g) {
        const size_t n = (size_t)B * frames;
        rs.rows = (int)n;
        MMI_HIP_CHECK(mem.alloc(&rs.xq, 2 * n * 2 * c.q_dimension));
        MMI_HIP_CHECK(mem.alloc(&rs.best_d, 4 * m->nchunk * n));
        MMI_HIP_CHECK(mem.alloc(&rs.best_i, 4 * m->nchunk * n));
        MMI_HIP_CHECK(mem.alloc(&rs.codes, n * c.q_n_q));
        MMI_HIP_CHECK(mem.alloc(&rs.qin_bp, (size_t)mmi_cdiv((int)n, 32) * m->q_in.Q * 256));
        MMI_HIP_CHECK(mem.alloc(&rs.qin_part, (size_t)8 * m->q_in.Mt * 32 * mmi_cdiv((int)n, 128) * 128));
        g->codes = rs.codes;
    }
    {
        ConvGemmArgs a = conv_args(m->downsample, dsin, 0, frames, lat, 0, B, false);
        a.first = m->first; a.exec = m->exec;
        if (latent_packed) { a.outp = rs.qin_bp; a.outQ = m->q_in.Q; }   // the latent, also as the RVQ input projection's operand
        prog.site("enc.downsample");
        if ((rc = add_conv(mem, prog, a))) return rc;
    }
    prog.site("enc.rvq");
    if ((rc = add_quantize_ops(m, mem, rs, prog, lat.p, 1, 0, B * frames, latent_packed))) return rc;
    prog.site("enc.commit");
    // commit
    return add_commit(m, prog, hist, B, g, &m->enc_hist, &m->enc_nhist, &m->enc_hist_rows, g ? &g->hist : &m->enc_tab, m->counters, T_tr, m->first);
}

int build_decoder(mmi_mimi* m, int B, int frames, MimiMem& mem, MimiGroup* g, hipStream_t s0) {
    const mmi_mimi_cfg& c = m->cfg;
    MmiProgram& prog = g ? g->prog : m->dec_prog;
    Buf &lat = g ? g->in : m->dec_codes_lat, &pcm = g ? g->out : m->dec_out;
    std::vector<HistDesc> hist;
    int rc;
    const int stride = c.resample_stride;
    size_t np = 0;                                        // the transposed convs' partial sums: the frame program's, in order
    auto partial = [&](long pn, float** out) -> hipError_t {
        if (!g) {
            hipError_t e = m->st.alloc(out, (size_t)B * pn);
            if (e == hipSuccess) e = mem.zero(*out, (size_t)B * pn, s0);
            if (e != hipSuccess) return e;
            m->partials.push_back(*out); m->partial_sizes.push_back(pn);
        }
        *out = m->partials[np++];
        return hipSuccess;
    };
    // dequantised latents [B][dim][frames]
    if ((rc = alloc_buf(mem, B, c.dimension, 0, frames, &lat, s0))) return rc;
    prog.site("dec.dequant");
    DequantScratch ds = m->deq;
    if (g) {
        const size_t n = (size_t)B * frames;
        MMI_HIP_CHECK(mem.alloc(&ds.codes, n * c.q_n_q));
        MMI_HIP_CHECK(mem.alloc(&ds.q2, n * 2 * c.q_dimension));
        MMI_HIP_CHECK(mem.alloc(&ds.qout_bp, (size_t)mmi_cdiv((int)n, 32) * m->q_out.Q * 256));
        MMI_HIP_CHECK(mem.alloc(&ds.qout_part, (size_t)8 * m->q_out.Mt * 32 * mmi_cdiv((int)n, 128) * 128));
        g->codes = ds.codes;
    }
    if ((rc = add_dequant_ops(m, mem, ds, prog, m->n_codebooks, lat, 0, B, frames, /*k_from_device=*/true))) return rc;
    prog.site("dec.upsample");
    // upsample (depthwise transposed conv) into the decoder transformer buffer = input of decoder conv0
    int T = stride * frames;
    Buf din;
    if ((rc = alloc_buf(mem, B, c.dimension, c.kernel_size - 1, T, &din, s0))) return rc;
    hist.push_back(hist_of(din, T));
    TrStream xs;
    if ((rc = alloc_tr_stream(m, mem, B * T, &xs))) return rc;
    {
        float* part = nullptr;
        MMI_HIP_CHECK(partial((long)c.dimension * stride, &part));
        const float* x = lat.p; const float* w = m->upsample_w; const uint8_t* ex = m->exec;
        float* out = din.p; int old = din.ld, ooff = din.H; int C = c.dimension; const int xld = lat.ld;
        prog.add([=](hipStream_t s) {
            MMI_LAUNCH(k_upsample_dw, mmi_cdiv(B * C * stride * frames, 256), 256, 0, s, x, xld, 0, w, part, ex, out, old, ooff, B, C,
                       2 * stride, stride, frames, xs.p, xs.J);
            MMI_CHECK_LAUNCH();
            return (int)MMI_OK;
        });
    }
    {
        const int Dh = c.tr_d_model / c.tr_num_heads;
        size_t kvn = (size_t)2 * c.tr_num_layers * B * c.tr_num_heads * c.tr_context * Dh;
        if (!g) {
            MMI_HIP_CHECK(m->st.alloc(&m->dec_kv, kvn));
            MMI_HIP_CHECK(mem.zero(m->dec_kv, kvn, s0));
        }
        prog.site("dec.tr");
        if ((rc = add_transformer(m, mem, prog, m->dec_tr, xs, din, din.H, T, m->dec_kv, m->counters + B, B, frames, s0))) return rc;
    }
    const int T_tr = T;
    size_t ci = 0;
    int mult = 1 << c.n_ratios;
    Buf cur;
    float* conv0_bp = nullptr;                            // dec.conv0's output in the packed operand order of dec.convtr0's GEMM
    {   // conv0: dimension -> mult*n_filters (no activation before it); consumer = conv-transpose GEMM (no history)
        if ((rc = alloc_buf(mem, B, mult * c.n_filters, 0, T, &cur, s0))) return rc;
        cur.elu = true;
        prog.site("dec.conv0");
        ConvGemmArgs a0 = conv_args(m->dec_convs[ci++], din, 0, T, cur, 0, B, false);
        // its (ELU'd) output is read by the first transposed-conv GEMM only: stored as that GEMM's packed operand as well
        const ConvW& wtr0 = m->dec_convs[ci];
        if ((B * T <= 128 || g) && wtr0.Q * 8 == mult * c.n_filters && !getenv("MMI_MIMI_PACK_LAUNCHES")) {
            MMI_HIP_CHECK(mem.alloc(&conv0_bp, (size_t)mmi_cdiv(B * T, 32) * wtr0.Q * 256));
            MMI_HIP_CHECK(mem.clear_operand(conv0_bp, mmi_cdiv(B * T, 32), wtr0.Q, mult * c.n_filters));
            a0.outp = conv0_bp; a0.outQ = wtr0.Q;
        }
        if ((rc = add_conv(mem, prog, a0))) return rc;
    }
    for (int i = 0; i < c.n_ratios; ++i) {
        const int ratio = c.ratios[i];
        const int cin = mult * c.n_filters, cout = cin / 2, K = 2 * ratio;
        // ELU + ConvTranspose1d: GEMM over channels, then overlap-add with the streaming partial
        Buf tmp, up;
        if ((rc = alloc_buf(mem, B, cout * K, 0, T, &tmp, s0))) return rc;
        const int Tn = T * ratio;
        if ((rc = alloc_buf(mem, B, cout, c.residual_kernel_size - 1, Tn, &up, s0))) return rc;
        if ((rc = alloc_twin(mem, B, &up, s0))) return rc;           // resblock input: raw for the residual, ELU'd for its conv
        const ConvW& wtr = m->dec_convs[ci++];
        prog.site("dec.convtr" + std::to_string(i));
        {
            ConvGemmArgs a = conv_args(wtr, cur, 0, T, tmp, 0, B, true);
            a.bias = nullptr;  // bias is added once, in the combine step
            if (i == 0 && conv0_bp) { a.bp = conv0_bp; a.x_packed = 1; }
            if ((rc = add_conv(mem, prog, a))) return rc;
        }
        {
            float* part = nullptr;
            MMI_HIP_CHECK(partial((long)cout * (K - ratio), &part));
            const float* tp = tmp.p; const float* bias = wtr.bias; const uint8_t* ex = m->exec;
            float* out = up.p; float* out2 = up.pe; int old = up.ld, ooff = up.H; int Tin = T; const int tld = tmp.ld;
            prog.add([=](hipStream_t s) {
                MMI_LAUNCH(k_convtr_combine, (int)mmi_cdiv64((int64_t)B * cout * Tin * ratio, 256), 256, 0, s, tp, bias, part,
                           ex, out, old, ooff, B, cout, K, ratio, Tin, out2, tld, Tin / frames);
                MMI_CHECK_LAUNCH();
                return (int)MMI_OK;
            });
        }
        hist.push_back(hist_of_src(up, Tn));
        T = Tn;
        // resblock; consumer = next conv-transpose GEMM (no history) or the final conv (last_kernel_size)
        Buf hid, nxt;
        const int Hn = (i + 1 < c.n_ratios) ? 0 : c.last_kernel_size - 1;
        if ((rc = alloc_buf(mem, B, cout / c.compress, 0, T, &hid, s0))) return rc;
        if ((rc = alloc_buf(mem, B, cout, Hn, T, &nxt, s0))) return rc;
        hid.elu = nxt.elu = true;               // read only behind an ELU: by the block's second conv / the next layer
        prog.site("dec.res" + std::to_string(i));
        const ConvGemmArgs a1 = conv_args(m->dec_convs[ci++], up, 0, T, hid, 0, B, true);
        const ConvW& w2 = m->dec_convs[ci++];
        ConvGemmArgs a = conv_args(w2, hid, 0, T, nxt, nxt.H, B, true);
        a.res = up.p; a.res_ld = up.ld; a.res_off = up.H;
        if ((rc = add_resblock(mem, prog, a1, a, w2))) return rc;
        if (Hn > 0) hist.push_back(hist_of(nxt, T));
        cur = nxt;
        mult /= 2;
    }
    if (T != c.frame_size * frames) return mmi_fail(MMI_ERR_UNSUPPORTED, "decoder does not reproduce frame_size samples");
    if ((rc = alloc_buf(mem, B, c.channels, 0, T, &pcm, s0))) return rc;
    prog.site("dec.final");
    if ((rc = add_conv(mem, prog, conv_args(m->dec_convs[ci++], cur, 0, T, pcm, 0, B, true)))) return rc;
    prog.site("dec.commit");
    return add_commit(m, prog, hist, B, g, &m->dec_hist, &m->dec_nhist, &m->dec_hist_rows, g ? &g->hist : &m->dec_tab, m->counters + B, T_tr, nullptr);
}

// Is s being captured, or (an error: the null stream, while another one is) not to be asked?  Leaves no error behind.
bool recording(hipStream_t s) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) == hipSuccess) return cap != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

// A call on s changes the exec mask: all_exec becomes `known`, unless the call is only being recorded.
void mask_changes(mmi_mimi* m, int known, hipStream_t s) {
    const bool rec = recording(s);
    m->mask_in_graph = m->mask_in_graph || rec;
    m->all_exec = rec ? -1 : known;
}
// After a mask or a snapshot a call of several frames reads the mask back, waiting for the work on s; once, unless it can change unseen.
bool all_run(mmi_mimi* m, hipStream_t s) {
    if (m->all_exec < 0 || m->mask_in_graph) {
        std::vector<uint8_t> ex(m->batch);
        if (hipMemcpyAsync(ex.data(), m->exec, ex.size(), hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        m->all_exec = std::find(ex.begin(), ex.end(), 0) == ex.end();
    }
    return m->all_exec == 1;
}

// ---- groups of frames ---------------------------------------------------------------------------
// Frames of the next group when `left` frames are to be run (1: frame by frame).  A group takes up to 160 frames over all streams - the 25 Hz
// layers then have 320 columns for weights that they read once, and its buffers 0.6 GB (encoder) or 0.8 GB (decoder) - and what is left is cut into
// equal groups.  Not while the caller's stream is being captured (a group's launch list is not kept for ever), and not under an exec mask
// that leaves streams out (their rows would have to stand still frame by frame).
int group_frames(mmi_mimi* m, const MimiGroup& g, const HistTable& tab, int left, hipStream_t s) {
    const mmi_mimi_cfg& c = m->cfg;
    int most = left;
    if (const char* e = getenv("MMI_MIMI_GROUP")) most = atoi(e);         // test hook: the largest group
    if (left < 2 || most < 2 || g.refused || tab.n < 0 || getenv("MMI_MIMI_PACK_LAUNCHES")) return 1;
    const int tpf = c.resample_stride, B = m->batch;
    most = std::min(most, std::min(std::min(160 / B, 512 / (B * tpf)), ((1 << 19) - 1) / (B * c.frame_size)));
    if (most < 2) return 1;
    return !recording(s) && all_run(m, s) ? mmi_cdiv(left, mmi_cdiv(left, most)) : 1;       // (the larger ones first: a call's slab grows once)
}

// The program of `frames` frames, ready to run on s.  False: this stream goes frame by frame from now on (a shape the plans do not take, no
// memory), with nothing left of the attempt - no buffers, and no error for the next launch check to find.
bool ready_group(mmi_mimi* m, bool enc, int frames, hipStream_t s) {
    MimiGroup& g = enc ? m->enc_grp : m->dec_grp;
    g.earlier = false;
    if (g.frames == frames) return true;
    MimiMem mem;
    mem.slab = &g.slab;
    mem.frames = frames;
    mem.stream = s;
    auto build = [&]() {
        g.frames = 0;
        g.prog.clear();
        g.slab.rewind();
        return enc ? build_encoder(m, m->batch, frames, mem, &g, s) : build_decoder(m, m->batch, frames, mem, &g, s);
    };
    bool ok = build() == MMI_OK;
    if (ok && g.slab.over) {                              // (what runs on s runs in the old reservation)
        ok = hipStreamSynchronize(s) == hipSuccess && g.slab.reserve(g.slab.need) == hipSuccess && build() == MMI_OK && !g.slab.over;
    }
    if (ok) {
        g.frames = frames;
        return true;
    }
    hipStreamSynchronize(s);
    (void)hipGetLastError();
    g.prog.clear();
    g.slab.release();
    g.refused = true;
    return false;
}

// A stream that runs single frames gives back what groups of an earlier one have left here.  (Not at the end of every stream: a file encoded or
// decoded without a stream of its own is one, and hipFree of 100 MB or more takes some 0.3 ms.)
void give_back_group(MimiGroup& g, hipStream_t s) {
    if ((g.frames && !g.earlier) || !g.slab.size || recording(s)) return;
    g.prog.clear();
    g.frames = 0;
    g.slab.release();
}

// The group's launches, and behind them on the host - while the GPU works on them - the capture of the frame program, so that a stream's
// first single frame after a call of several does not wait for it.  (A capture that fails fails there: the group has run.)
int run_group(mmi_mimi* m, bool enc, hipStream_t s) {
    MimiGroup& g = enc ? m->enc_grp : m->dec_grp;
    const HistTable& st = enc ? m->enc_tab : m->dec_tab;
    const int rows = enc ? m->enc_hist_rows : m->dec_hist_rows;
    MMI_LAUNCH(k_move_history, mmi_cdiv(rows, 256), 256, 0, s, st, g.hist, rows);
    int rc = g.prog.run_eager(s);
    if (rc) return rc;
    MMI_LAUNCH(k_move_history, mmi_cdiv(rows, 256), 256, 0, s, g.hist, st, rows);
    MMI_CHECK_LAUNCH();
    if (m->use_graph && (enc ? m->enc_prog : m->dec_prog).capture_full(m->cap_stream)) (void)hipGetLastError();
    return MMI_OK;
}

int check_cfg(const mmi_mimi_cfg& c) {
    if (c.n_ratios < 1 || c.n_ratios > 8) return mmi_fail(MMI_ERR_UNSUPPORTED, "n_ratios out of range");
    int hop = 1;
    for (int i = 0; i < c.n_ratios; ++i) hop *= c.ratios[i];
    if (hop * c.resample_stride != c.frame_size) return mmi_fail(MMI_ERR_UNSUPPORTED, "frame_size != hop*stride");
    if (c.tr_d_model != c.dimension) return mmi_fail(MMI_ERR_UNSUPPORTED, "projected transformer (d_model != dimension)");
    const int Dh = c.tr_d_model / c.tr_num_heads;
    if (Dh * c.tr_num_heads != c.tr_d_model || (Dh & 3) || 256 % Dh != 0)
        return mmi_fail(MMI_ERR_UNSUPPORTED, "head dim must be a multiple of 4 and divide 256");
    if (c.tr_d_model > 1024) return mmi_fail(MMI_ERR_UNSUPPORTED, "transformer width above the LayerNorm kernel's register budget");
    if (c.q_dimension % 4) return mmi_fail(MMI_ERR_UNSUPPORTED, "codebook dimension must be a multiple of 4");
    if (c.compress < 1 || c.q_n_q_semantic < 1 || c.q_n_q < c.q_n_q_semantic)
        return mmi_fail(MMI_ERR_UNSUPPORTED, "bad quantizer/compress config");
    return MMI_OK;
}

int frame_count_ok(const mmi_mimi* m, int batch, int n_frames) {
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    if (!m->streaming) return mmi_fail(MMI_ERR_STATE, "not streaming: call mmi_mimi_streaming_start first");
    if (batch != m->batch) return mmi_fail(MMI_ERR_SHAPE, "batch size does not match the streaming batch");
    if (n_frames <= 0) return mmi_fail(MMI_ERR_SHAPE, "length must be a positive multiple of the frame size");
    return MMI_OK;
}

}  // namespace

// ===============================================================================================
// C ABI
// ===============================================================================================
extern "C" int mmi_mimi_create(const mmi_mimi_cfg* cfg, const mmi_tensor_desc* weights, int32_t n_weights,
                               int32_t max_batch, mmi_mimi** out) {
    if (!cfg || !weights || !out || max_batch <= 0) return mmi_fail(MMI_ERR_INVALID, "mmi_mimi_create: bad argument");
    int rc = check_cfg(*cfg);
    if (rc) return rc;
    mmi_mimi* m = new mmi_mimi();
    if (hipGetDevice(&m->device) != hipSuccess) m->device = -1;
    m->cfg = *cfg;
    m->max_batch = max_batch;
    m->n_codebooks = cfg->q_n_q < 8 ? cfg->q_n_q : 8;
    m->use_graph = mmi_graphs_enabled();
    MmiWeights W{weights, n_weights};
    const mmi_mimi_cfg& c = m->cfg;
    auto fail = [&](int code) { mmi_mimi_destroy(m); return code; };

    // ---- SEANet encoder (seanet.py:169-236): model.{0,3,6,...} strided, model.{1,4,...}.block.{1,3} resblocks
    {
        int idx = 0, mult = 1;
        ConvW cw;
        if ((rc = load_conv(m, W, "encoder.model.0.conv.conv", c.channels, c.n_filters, c.kernel_size, 1, true, &cw))) return fail(rc);
        m->enc_convs.push_back(cw);
        idx = 1;
        for (int i = 0; i < c.n_ratios; ++i) {
            const int ratio = c.ratios[c.n_ratios - 1 - i];
            const int ch = mult * c.n_filters, hid = ch / c.compress;
            std::string rb = "encoder.model." + std::to_string(idx) + ".block.";
            if ((rc = load_conv(m, W, rb + "1.conv.conv", ch, hid, c.residual_kernel_size, 1, true, &cw))) return fail(rc);
            m->enc_convs.push_back(cw);
            if ((rc = load_conv(m, W, rb + "3.conv.conv", hid, ch, 1, 1, true, &cw))) return fail(rc);
            m->enc_convs.push_back(cw);
            idx += 2;  // resblock, ELU
            if ((rc = load_conv(m, W, "encoder.model." + std::to_string(idx) + ".conv.conv", ch, 2 * ch, 2 * ratio, ratio, true, &cw))) return fail(rc);
            m->enc_convs.push_back(cw);
            idx += 1;
            mult *= 2;
        }
        idx += 1;  // ELU
        if ((rc = load_conv(m, W, "encoder.model." + std::to_string(idx) + ".conv.conv", mult * c.n_filters, c.dimension, c.last_kernel_size, 1, true, &cw))) return fail(rc);
        m->enc_convs.push_back(cw);
    }
    // ---- SEANet decoder (seanet.py:315-388)
    {
        int mult = 1 << c.n_ratios;
        ConvW cw;
        if ((rc = load_conv(m, W, "decoder.model.0.conv.conv", c.dimension, mult * c.n_filters, c.kernel_size, 1, true, &cw))) return fail(rc);
        m->dec_convs.push_back(cw);
        int idx = 1;
        for (int i = 0; i < c.n_ratios; ++i) {
            const int ratio = c.ratios[i];
            const int cin = mult * c.n_filters, cout = cin / 2, hid = cout / c.compress;
            idx += 1;  // ELU
            if ((rc = load_convtr(m, W, "decoder.model." + std::to_string(idx) + ".convtr.convtr", cin, cout, 2 * ratio, ratio, &cw))) return fail(rc);
            m->dec_convs.push_back(cw);
            idx += 1;
            std::string rb = "decoder.model." + std::to_string(idx) + ".block.";
            if ((rc = load_conv(m, W, rb + "1.conv.conv", cout, hid, c.residual_kernel_size, 1, true, &cw))) return fail(rc);
            m->dec_convs.push_back(cw);
            if ((rc = load_conv(m, W, rb + "3.conv.conv", hid, cout, 1, 1, true, &cw))) return fail(rc);
            m->dec_convs.push_back(cw);
            idx += 1;
            mult /= 2;
        }
        idx += 1;  // ELU
        if ((rc = load_conv(m, W, "decoder.model." + std::to_string(idx) + ".conv.conv", c.n_filters, c.channels, c.last_kernel_size, 1, true, &cw))) return fail(rc);
        m->dec_convs.push_back(cw);
    }
    if ((rc = load_transformer(m, W, "encoder_transformer", &m->enc_tr))) return fail(rc);
    if ((rc = load_transformer(m, W, "decoder_transformer", &m->dec_tr))) return fail(rc);
    // ---- resampling (resample.py:14-119)
    if ((rc = load_conv(m, W, "downsample.conv.conv.conv", c.dimension, c.dimension, 2 * c.resample_stride, c.resample_stride, false, &m->downsample))) return fail(rc);
    {
        const mmi_tensor_desc* w;
        if ((rc = need(W, "upsample.convtr.convtr.convtr.weight", 3, &w))) return fail(rc);
        if (w->shape[0] != c.dimension || w->shape[1] != 1 || w->shape[2] != 2 * c.resample_stride)
            return fail(mmi_fail(MMI_ERR_SHAPE, "shape mismatch for upsample weight"));
        if ((rc = copy_vec(m, w, c.dimension * 2 * c.resample_stride, &m->upsample_w))) return fail(rc);
    }
    if ((rc = load_rvq(m, W))) return fail(rc);
    // ---- RVQ scratch
    m->nchunk = mmi_cdiv(c.q_bins, MMI_RVQ_CHUNK);
    m->rvq.rows = max_batch;
    if (hipSuccess != m->wts.alloc(&m->rvq.xq, (size_t)2 * max_batch * 2 * c.q_dimension) ||
        hipSuccess != m->wts.alloc(&m->rvq.best_d, (size_t)4 * m->nchunk * max_batch) ||
        hipSuccess != m->wts.alloc(&m->rvq.best_i, (size_t)4 * m->nchunk * max_batch) ||
        hipSuccess != m->wts.alloc(&m->rvq.codes, (size_t)max_batch * c.q_n_q) ||
        hipSuccess != m->wts.alloc(&m->deq.codes, (size_t)max_batch * c.q_n_q) ||
        hipSuccess != m->wts.alloc(&m->deq.q2, (size_t)max_batch * 2 * c.q_dimension) ||
        hipSuccess != m->wts.alloc(&m->rvq.qin_bp, (size_t)mmi_cdiv(max_batch, 32) * m->q_in.Q * 256) ||
        hipSuccess != m->wts.alloc(&m->deq.qout_bp, (size_t)mmi_cdiv(max_batch, 32) * m->q_out.Q * 256) ||
        hipSuccess != m->wts.alloc(&m->rvq.qin_part, (size_t)8 * m->q_in.Mt * 32 * 128) ||
        hipSuccess != m->wts.alloc(&m->deq.qout_part, (size_t)8 * m->q_out.Mt * 32 * 128))
        return fail(mmi_fail(MMI_ERR_HIP, "out of device memory (RVQ scratch)"));
    if (hipDeviceSynchronize() != hipSuccess) return fail(mmi_fail(MMI_ERR_HIP, "weight packing failed"));
    if (m->use_graph && hipStreamCreate(&m->cap_stream) != hipSuccess)
        return fail(mmi_fail(MMI_ERR_HIP, "hipStreamCreate failed"));
    *out = m;
    return MMI_OK;
}

// ---- what handles keep while they do not stream ----
static void stop_stream(mmi_mimi* m) {
    hipDeviceSynchronize();
    m->enc_prog.clear();
    m->dec_prog.clear();
    for (MimiGroup* g : {&m->enc_grp, &m->dec_grp}) {      // their launches name the state that goes now; the slabs stay (give_back_group)
        g->prog.clear();
        g->frames = 0;
        g->refused = false;
    }
    m->st.release();
    m->partials.clear();
    m->partial_sizes.clear();
    m->streaming = m->parked = m->unfinished = false;
    m->batch = 0;
}
static void drop_parked(mmi_mimi* m) {
    if (m->parked) stop_stream(m);
}

// A handle that does not stream may keep the stream of its last file (mmi_mimi_file_stop) and the slabs of its groups of frames.  It is in a list
// of the process then, and an allocation of any thread that finds no memory takes it away (let_go).  A call that starts, stops or ends a
// stream takes its handle out for as long as it lasts.
struct IdleHandles {
    std::mutex mu;
    std::vector<mmi_mimi*> list;
};
static IdleHandles& idle() {                               // (never destroyed: handles may outlive this file's statics)
    static IdleHandles* h = new IdleHandles;
    return *h;
}
struct OutOfIdle {
    mmi_mimi* m;
    explicit OutOfIdle(mmi_mimi* m_) : m(m_) {
        std::lock_guard<std::mutex> g(idle().mu);
        std::vector<mmi_mimi*>& list = idle().list;
        list.erase(std::remove(list.begin(), list.end(), m), list.end());
    }
    ~OutOfIdle() {
        if (!m || m->streaming || m->unfinished || !(m->parked || m->enc_grp.slab.size || m->dec_grp.slab.size)) return;
        std::lock_guard<std::mutex> g(idle().mu);
        idle().list.push_back(m);
    }
    OutOfIdle(const OutOfIdle&) = delete;
    OutOfIdle& operator=(const OutOfIdle&) = delete;
};
static bool let_go(int device) {
    std::lock_guard<std::mutex> g(idle().mu);
    std::vector<mmi_mimi*>& list = idle().list;
    const size_t n = list.size();
    list.erase(std::remove_if(list.begin(), list.end(), [&](mmi_mimi* m) {
        if (m->device != device) return false;
        drop_parked(m);
        return m->enc_grp.slab.release() && m->dec_grp.slab.release();
    }), list.end());
    return list.size() < n;
}
static const bool let_go_set = (mmi_set_let_go(&let_go), true);

extern "C" void mmi_mimi_destroy(mmi_mimi* m) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return;
    { OutOfIdle out(m); out.m = nullptr; }                 // (for good)
    if (m->streaming || m->parked) stop_stream(m);
    m->enc_grp.slab.drop();
    m->dec_grp.slab.drop();
    m->wts.release();
    if (m->cap_stream) hipStreamDestroy(m->cap_stream);
    delete m;
}

extern "C" int mmi_mimi_set_num_codebooks(mmi_mimi* m, int32_t n) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    if (n < 1 || n > m->cfg.q_n_q) return mmi_fail(MMI_ERR_INVALID, "num_codebooks out of range");
    if (m->streaming) return mmi_fail(MMI_ERR_STATE, "set_num_codebooks while streaming");
    m->n_codebooks = n;
    return MMI_OK;
}

extern "C" int mmi_mimi_num_codebooks(const mmi_mimi* m) { return m ? m->n_codebooks : 0; }
extern "C" int mmi_mimi_device(const mmi_mimi* m) { return m ? m->device : -1; }

int64_t mmi_copy_launch_log(const std::vector<std::string>& log, char* buf, int64_t cap);   // api_common.hip

extern "C" int64_t mmi_mimi_launch_list(const mmi_mimi* m, int32_t which, char* buf, int64_t cap) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !m->streaming) return 0;
    const bool enc = which == 0 || which == 2;
    const MmiProgram& p = enc ? m->enc_prog : m->dec_prog;
    const MmiProgram& g = enc ? m->enc_grp.prog : m->dec_grp.prog;
    if (which >= 2 || !p.logged()) return g.logged() ? mmi_copy_launch_log(g.launch_log(), buf, cap) : 0;      // (frames have only been run in groups so far)
    return mmi_copy_launch_log(p.launch_log(), buf, cap);
}

extern "C" int mmi_mimi_get_cfg(const mmi_mimi* m, mmi_mimi_cfg* out) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !out) return mmi_fail(MMI_ERR_INVALID, "null argument");
    *out = m->cfg;
    return MMI_OK;
}

static int start_stream(mmi_mimi* m, int batch, hipStream_t s) {
    m->batch = batch;
    int rc = MMI_OK;
    m->st.chunk = (size_t)32 << 20;
    auto fail = [&](int code) { stop_stream(m); return code; };
    if (hipSuccess != m->st.alloc(&m->exec, (size_t)batch) || hipSuccess != m->st.alloc(&m->first, (size_t)batch) ||
        hipSuccess != m->st.alloc(&m->counters, (size_t)2 * batch) || hipSuccess != m->st.alloc(&m->dec_k_dev, (size_t)1))
        return fail(mmi_fail(MMI_ERR_HIP, "out of device memory (state)"));
    // every failure from here on goes through fail(): what was allocated / appended so far is released again
    m->dec_k_host = m->n_codebooks;
    m->dec_k_cur = m->n_codebooks;
    if (hipMemsetAsync(m->exec, 1, batch, s) != hipSuccess || hipMemsetAsync(m->first, 1, batch, s) != hipSuccess ||
        hipMemsetAsync(m->counters, 0, (size_t)2 * batch * sizeof(long), s) != hipSuccess ||
        hipMemcpyAsync(m->dec_k_dev, &m->dec_k_host, sizeof(int), hipMemcpyHostToDevice, s) != hipSuccess)
        return fail(mmi_fail(MMI_ERR_HIP, "initialising the streaming state failed"));
    MimiMem mem;
    mem.arena = &m->st;
    mem.stream = s;
    if ((rc = build_encoder(m, batch, 1, mem, nullptr, s))) return fail(rc);
    if ((rc = build_decoder(m, batch, 1, mem, nullptr, s))) return fail(rc);
    m->all_exec = 1;
    m->mask_in_graph = false;
    if (hipStreamSynchronize(s) != hipSuccess) return fail(mmi_fail(MMI_ERR_HIP, "hipStreamSynchronize failed"));
    m->streaming = true;
    return MMI_OK;
}

// Work on the device done, for a stream whose own wait has failed
static int finish_parked(mmi_mimi* m) {
    if (!m->unfinished) return MMI_OK;
    MMI_HIP_CHECK(hipDeviceSynchronize());
    m->unfinished = false;
    return MMI_OK;
}

// (the handle is out of the idle ones)
static int start_any_stream(mmi_mimi* m, int32_t batch, mmi_stream stream) {
    if (m->streaming) return mmi_fail(MMI_ERR_STATE, "already streaming");  // streaming.py:113
    if (batch <= 0 || batch > m->max_batch) return mmi_fail(MMI_ERR_SHAPE, "batch exceeds max_batch");
    int rc = finish_parked(m);
    if (rc) return rc;
    drop_parked(m);
    rc = start_stream(m, batch, (hipStream_t)stream);
    if (rc == MMI_ERR_HIP && (m->enc_grp.slab.size || m->dec_grp.slab.size)) {      // without what an earlier stream's groups have left
        m->enc_grp.slab.release();
        m->dec_grp.slab.release();
        rc = start_stream(m, batch, (hipStream_t)stream);
    }
    return rc;
}

extern "C" int mmi_mimi_streaming_start(mmi_mimi* m, int32_t batch, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    OutOfIdle out(m);
    return start_any_stream(m, batch, stream);
}

extern "C" int mmi_mimi_streaming_stop(mmi_mimi* m) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    OutOfIdle out(m);
    if (m->streaming) {
        stop_stream(m);
        return MMI_OK;
    }
    const int rc = finish_parked(m);
    if (rc) return rc;
    drop_parked(m);
    m->enc_grp.slab.release();
    m->dec_grp.slab.release();
    return MMI_OK;
}

// A file is a stream that nobody else sees.  Starting and stopping one takes some 400 us - 32 MB allocated, zeroed and freed, two launch lists built,
// captured and dropped - where 8 frames take the GPU 250; so what it has built stays for the next file of as many streams, which resets the
// state instead.  At most MIMI_PARK bytes of state stay (the full-size codec: four streams), and the groups' slabs as behind every stream: until a
// stream of the caller's own starts, a file of another number of streams or codebooks, an allocation finds no memory, or the handle goes.
// 8 frames of 1, 2, 3, 4 streams encoded and decoded, us: 1755, 1859, 2658, 3318 with a stream's start and stop each, 973, 1085, 1270, 1323 so.
// (More streams would gain as much, 4312 -> 1581 for five, but for memory, 40 MB a stream, that the process's other allocators cannot ask back.)
constexpr size_t MIMI_PARK = (size_t)128 << 20;

// MMI_DEBUG_POISON=1: what the next file may not see - the rings, the buffers with histories, the overlap-adds' partial rows, offsets and flags - is
// NaNs and -1 in front of its reset, whatever the last file has left there.
static int poison_parked(mmi_mimi* m, hipStream_t s) {
    const char* pz = getenv("MMI_DEBUG_POISON");
    if (!pz || pz[0] != '1') return MMI_OK;
    std::vector<const void*> places = {m->enc_kv, m->dec_kv, m->counters, m->first, m->exec};
    places.insert(places.end(), m->partials.begin(), m->partials.end());
    for (const HistTable* t : {&m->enc_tab, &m->dec_tab})
        for (int i = 0; i < t->n; ++i) places.push_back(t->d[i].p);
    for (size_t i = 0; i < m->st.ptrs.size(); ++i) {
        const char* at = (const char*)m->st.ptrs[i];
        if (std::any_of(places.begin(), places.end(), [&](const void* p) { return (const char*)p >= at && (const char*)p < at + m->st.sizes[i]; }))
            MMI_HIP_CHECK(hipMemsetAsync(m->st.ptrs[i], 0xFF, m->st.sizes[i], s));
    }
    return MMI_OK;
}

extern "C" int mmi_mimi_file_start(mmi_mimi* m, int32_t batch, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    OutOfIdle out(m);
    if (!m->parked || m->batch != batch || m->parked_k != m->n_codebooks) return start_any_stream(m, batch, stream);
    // (a stream cannot start there either: it waits for its own state)
    if (recording((hipStream_t)stream)) return mmi_fail(MMI_ERR_HIP, "a file's stream cannot start while its HIP stream is being captured");
    int rc = finish_parked(m);
    if (rc) return rc;
    m->parked = false;
    m->streaming = true;
    m->all_exec = 1;
    m->mask_in_graph = false;
    for (MimiGroup* g : {&m->enc_grp, &m->dec_grp}) {
        g->refused = false;
        g->earlier = true;
    }
    rc = poison_parked(m, (hipStream_t)stream);
    if (!rc) rc = mmi_mimi_reset(m, nullptr, stream);
    if (rc) stop_stream(m);
    return rc;
}

extern "C" int mmi_mimi_file_stop(mmi_mimi* m) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    if (!m->streaming) return MMI_OK;
    OutOfIdle out(m);
    m->streaming = false;
    m->parked = true;
    m->parked_k = m->n_codebooks;
    m->unfinished = true;
    int rc = finish_parked(m);                             // (where it fails nothing goes: work on the device may use it)
    if (!rc && m->st.held() > MIMI_PARK) drop_parked(m);
    return rc;
}

extern "C" int mmi_mimi_streaming_batch(const mmi_mimi* m) { return m && m->streaming ? m->batch : 0; }

extern "C" int64_t mmi_mimi_state_bytes(const mmi_mimi* m) { return m && m->streaming ? (int64_t)m->st.bytes : 0; }

extern "C" int mmi_mimi_state_save(mmi_mimi* m, void* dst, int64_t bytes, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !dst) return mmi_fail(MMI_ERR_INVALID, "null argument");
    if (!m->streaming) return mmi_fail(MMI_ERR_STATE, "not streaming");
    if (bytes != (int64_t)m->st.bytes) return mmi_fail(MMI_ERR_SHAPE, "snapshot buffer has the wrong size");
    MMI_HIP_CHECK(m->st.save(dst, (hipStream_t)stream));
    return MMI_OK;
}

extern "C" int mmi_mimi_state_load(mmi_mimi* m, const void* src, int64_t bytes, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !src) return mmi_fail(MMI_ERR_INVALID, "null argument");
    if (!m->streaming) return mmi_fail(MMI_ERR_STATE, "not streaming");
    if (bytes != (int64_t)m->st.bytes) return mmi_fail(MMI_ERR_SHAPE, "snapshot taken from a different stream (batch)");
    MMI_HIP_CHECK(m->st.load(src, (hipStream_t)stream));
    mask_changes(m, -1, (hipStream_t)stream);      // the snapshot carries its own mask
    m->dec_k_cur = -1;        // the snapshot carries its own device-side K: the next decode re-uploads the caller's
    return MMI_OK;
}

extern "C" int mmi_mimi_set_exec_mask(mmi_mimi* m, const uint8_t* mask, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !mask) return mmi_fail(MMI_ERR_INVALID, "null argument");
    if (!m->streaming) return mmi_fail(MMI_ERR_STATE, "not streaming");
    mask_changes(m, -1, (hipStream_t)stream);
    MMI_LAUNCH(k_set_mask, mmi_cdiv(m->batch, 64), 64, 0, (hipStream_t)stream, m->exec, mask, m->batch);
    MMI_CHECK_LAUNCH();
    return MMI_OK;
}

extern "C" int mmi_mimi_reset(mmi_mimi* m, const uint8_t* mask, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m) return mmi_fail(MMI_ERR_INVALID, "null handle");
    if (!m->streaming) return mmi_fail(MMI_ERR_STATE, "not streaming");
    hipStream_t s = (hipStream_t)stream;
    const int B = m->batch;
    mask_changes(m, !mask || m->all_exec == 1 ? 1 : -1, s);
    if (m->enc_tab.n >= 0 && m->dec_tab.n >= 0 && m->partials.size() <= MMI_PARTIALS_MAX) {
        ResetTable t;
        memset(&t, 0, sizeof(t));
        t.hist[0] = m->enc_tab;
        t.hist[1] = m->dec_tab;
        t.rows[0] = m->enc_hist_rows;
        t.rows[1] = m->dec_hist_rows;
        t.B = B;
        t.counters = m->counters;
        t.first = m->first;
        t.exec = m->exec;
        long n = 0;
        for (size_t i = 0; i < m->partials.size(); ++i) {
            t.part[t.n_part] = m->partials[i];
            t.part_row[t.n_part] = m->partial_sizes[i];
            t.part_end[t.n_part++] = n += (long)B * m->partial_sizes[i];
        }
        MMI_LAUNCH(k_reset_all, (int)mmi_cdiv64(t.rows[0] + t.rows[1] + n + B, 256), 256, 0, s, t, mask);
        MMI_CHECK_LAUNCH();
        return MMI_OK;
    }
    if (m->enc_hist_rows > 0)
        MMI_LAUNCH(k_reset_history, mmi_cdiv(m->enc_hist_rows, 256), 256, 0, s, (const HistDesc*)m->enc_hist, m->enc_nhist, m->enc_hist_rows, mask);
    if (m->dec_hist_rows > 0)
        MMI_LAUNCH(k_reset_history, mmi_cdiv(m->dec_hist_rows, 256), 256, 0, s, (const HistDesc*)m->dec_hist, m->dec_nhist, m->dec_hist_rows, mask);
    for (size_t i = 0; i < m->partials.size(); ++i)
        MMI_LAUNCH(k_reset_rows_f32, (int)mmi_cdiv64((int64_t)B * m->partial_sizes[i], 256), 256, 0, s, m->partials[i], m->partial_sizes[i], B, mask);
    MMI_LAUNCH(k_reset_counters, mmi_cdiv(B, 64), 64, 0, s, m->counters, 2, m->first, m->exec, B, mask);
    MMI_CHECK_LAUNCH();
    return MMI_OK;
}

static int encode_impl(mmi_mimi* m, const float* pcm, int64_t* codes, float* latent, int32_t batch, int32_t n_frames,
                       hipStream_t s) {
    int rc = frame_count_ok(m, batch, n_frames);
    if (rc) return rc;
    if (!pcm) return mmi_fail(MMI_ERR_INVALID, "null pcm");
    const mmi_mimi_cfg& c = m->cfg;
    const int F = c.frame_size, K = m->n_codebooks;
    for (int f = 0, G; f < n_frames; f += G) {
        G = group_frames(m, m->enc_grp, m->enc_tab, n_frames - f, s);
        if (G > 1 && !ready_group(m, true, G, s)) G = 1;
        if (G == 1) give_back_group(m->enc_grp, s);
        const Buf &in = G > 1 ? m->enc_grp.in : m->enc_in, &lat = G > 1 ? m->enc_grp.out : m->latent;
        // stage the samples behind the first conv's history
        MMI_LAUNCH(k_copy2d_f32, (int)mmi_cdiv64((int64_t)batch * c.channels * G * F, 256), 256, 0, s, pcm + (long)f * F,
                   (long)n_frames * F, in.p + in.H, (long)in.ld, batch * c.channels, G * F);
        if ((rc = G > 1 ? run_group(m, true, s) : m->enc_prog.run(s, m->use_graph, m->cap_stream))) return rc;
        if (codes)
            MMI_LAUNCH(k_codes_out, mmi_cdiv(batch * G * K, 256), 256, 0, s, (const int*)(G > 1 ? m->enc_grp.codes : m->rvq.codes), c.q_n_q, (long*)codes,
                       batch, K, n_frames, f, G);
        if (latent)
            MMI_LAUNCH(k_copy2d_f32, mmi_cdiv(batch * c.dimension * G, 256), 256, 0, s, (const float*)lat.p, (long)lat.ld, latent + f,
                       (long)n_frames, batch * c.dimension, G);
        MMI_CHECK_LAUNCH();
    }
    return MMI_OK;
}

extern "C" int mmi_mimi_encode_step(mmi_mimi* m, const float* pcm, int64_t* codes, int32_t batch, int32_t n_frames,
                                    mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!codes) return mmi_fail(MMI_ERR_INVALID, "null codes");
    return encode_impl(m, pcm, codes, nullptr, batch, n_frames, (hipStream_t)stream);
}

extern "C" int mmi_mimi_encode_latent_step(mmi_mimi* m, const float* pcm, float* latent, int32_t batch, int32_t n_frames,
                                           mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!latent) return mmi_fail(MMI_ERR_INVALID, "null latent");
    return encode_impl(m, pcm, nullptr, latent, batch, n_frames, (hipStream_t)stream);
}

extern "C" int mmi_mimi_quantize(mmi_mimi* m, const float* latent, int64_t* codes, int32_t batch, int32_t n_frames,
                                 mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !latent || !codes) return mmi_fail(MMI_ERR_INVALID, "null argument");
    if (batch <= 0 || batch > m->max_batch || n_frames <= 0) return mmi_fail(MMI_ERR_SHAPE, "bad batch / frames");
    hipStream_t s = (hipStream_t)stream;
    const mmi_mimi_cfg& c = m->cfg;
    for (int f = 0; f < n_frames; ++f) {
        MmiProgram prog;
        MimiMem mem;
        mem.arena = &m->st;
        mem.stream = s;
        int rc = add_quantize_ops(m, mem, m->rvq, prog, latent, n_frames, f, batch);
        if (rc) return rc;
        rc = prog.run_eager(s);
        if (rc) return rc;
        MMI_LAUNCH(k_codes_out, mmi_cdiv(batch * m->n_codebooks, 256), 256, 0, s, (const int*)m->rvq.codes, c.q_n_q, (long*)codes, batch,
                   m->n_codebooks, n_frames, f, 1);
        MMI_CHECK_LAUNCH();
    }
    return MMI_OK;
}

extern "C" int mmi_mimi_decode_latent(mmi_mimi* m, const int64_t* codes, float* latent, int32_t batch, int32_t n_codebooks,
                                      int32_t n_frames, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    if (!m || !latent || !codes) return mmi_fail(MMI_ERR_INVALID, "null argument");
    if (batch <= 0 || batch > m->max_batch || n_frames <= 0 || n_codebooks < 1 || n_codebooks > m->cfg.q_n_q)
        return mmi_fail(MMI_ERR_SHAPE, "bad batch / codebooks / frames");
    hipStream_t s = (hipStream_t)stream;
    const mmi_mimi_cfg& c = m->cfg;
    Buf out; out.p = latent; out.C = c.dimension; out.ld = n_frames; out.H = 0;
    for (int f = 0; f < n_frames; ++f) {
        MMI_LAUNCH(k_codes_in, mmi_cdiv(batch * n_codebooks, 256), 256, 0, s, (const long*)codes, (long)n_codebooks * n_frames, m->deq.codes,
                   c.q_n_q, batch, n_codebooks, n_frames, f, 1);
        MmiProgram prog;
        MimiMem mem;
        mem.arena = &m->st;
        mem.stream = s;
        int rc = add_dequant_ops(m, mem, m->deq, prog, n_codebooks, out, f, batch);
        if (rc) return rc;
        rc = prog.run_eager(s);
        if (rc) return rc;
    }
    return MMI_OK;
}

extern "C" int mmi_mimi_decode_step(mmi_mimi* m, const int64_t* codes, float* pcm, int32_t batch, int32_t n_codebooks,
                                    int32_t n_frames, mmi_stream stream) {
    return mmi_mimi_decode_step_strided(m, codes, (int64_t)n_codebooks * n_frames, pcm, batch, n_codebooks, n_frames, stream);
}

extern "C" int mmi_mimi_decode_step_strided(mmi_mimi* m, const int64_t* codes, int64_t batch_stride, float* pcm, int32_t batch,
                                            int32_t n_codebooks, int32_t n_frames, mmi_stream stream) {
    MmiDeviceGuard dev_guard_(m ? m->device : -1);
    int rc = frame_count_ok(m, batch, n_frames);
    if (rc) return rc;
    if (!codes || !pcm) return mmi_fail(MMI_ERR_INVALID, "null argument");
    // any 1 <= K <= n_q: "the split RVQ decodes however many codebooks it is given" (compression.py:406-429, vq.py:281-287)
    if (n_codebooks < 1 || n_codebooks > m->cfg.q_n_q) return mmi_fail(MMI_ERR_SHAPE, "codes must carry between 1 and n_q codebooks");
    if (batch_stride < (int64_t)n_codebooks * n_frames) return mmi_fail(MMI_ERR_SHAPE, "batch stride smaller than one row of codes");
    hipStream_t s = (hipStream_t)stream;
    const mmi_mimi_cfg& c = m->cfg;
    const int F = c.frame_size;
    if (n_codebooks != m->dec_k_cur) {                  // the captured program reads K from device memory
        m->dec_k_host = n_codebooks;
        MMI_HIP_CHECK(hipMemcpyAsync(m->dec_k_dev, &m->dec_k_host, sizeof(int), hipMemcpyHostToDevice, s));
        MMI_HIP_CHECK(hipStreamSynchronize(s));         // the host word is reused; K changes at most once per model in practice
        m->dec_k_cur = n_codebooks;
    }
    for (int f = 0, G; f < n_frames; f += G) {
        G = group_frames(m, m->dec_grp, m->dec_tab, n_frames - f, s);
        if (G > 1 && !ready_group(m, false, G, s)) G = 1;
        if (G == 1) give_back_group(m->dec_grp, s);
        MMI_LAUNCH(k_codes_in, mmi_cdiv(batch * G * n_codebooks, 256), 256, 0, s, (const long*)codes, (long)batch_stride, G > 1 ? m->dec_grp.codes : m->deq.codes,
                   c.q_n_q, batch, n_codebooks, n_frames, f, G);
        MMI_CHECK_LAUNCH();
        if ((rc = G > 1 ? run_group(m, false, s) : m->dec_prog.run(s, m->use_graph, m->cap_stream))) return rc;
        const Buf& out = G > 1 ? m->dec_grp.out : m->dec_out;
        MMI_LAUNCH(k_copy2d_f32, (int)mmi_cdiv64((int64_t)batch * c.channels * G * F, 256), 256, 0, s, (const float*)out.p, (long)out.ld,
                   pcm + (long)f * F, (long)n_frames * F, batch * c.channels, G * F);
        MMI_CHECK_LAUNCH();
    }
    return MMI_OK;
}
