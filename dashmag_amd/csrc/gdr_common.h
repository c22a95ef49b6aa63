// Declarations shared by the gated-delta-rule translation units.
#pragma once

#include "dm_common.h"

namespace dm {

constexpr int kChunk = 64;  // tokens per chunk (chunk/reference.rs:26)

struct GdrArgs {
    int64_t H, Dk, Dv;
    int64_t rows;  // B * T token rows of the inputs
    int g_dt, beta_dt, l2norm;
    float scale;
    const void *q, *k, *v, *g, *beta;
    // element strides of the inputs along their token rows (the flattened b * T + t) and heads:
    // q, k, v, g, beta and the backward's output gradient (o)
    int64_t q_t, q_h, k_t, k_h, v_t, v_h, g_t, g_h, b_t, b_h, o_t, o_h;
};

// Element offsets of token row `tok`, head h of each input.
__host__ __device__ inline int64_t q_at(const GdrArgs &a, int64_t tok, int64_t h) {
    return tok * a.q_t + h * a.q_h;
}
__host__ __device__ inline int64_t k_at(const GdrArgs &a, int64_t tok, int64_t h) {
    return tok * a.k_t + h * a.k_h;
}
__host__ __device__ inline int64_t v_at(const GdrArgs &a, int64_t tok, int64_t h) {
    return tok * a.v_t + h * a.v_h;
}
__host__ __device__ inline int64_t g_at(const GdrArgs &a, int64_t tok, int64_t h) {
    return tok * a.g_t + h * a.g_h;
}
__host__ __device__ inline int64_t b_at(const GdrArgs &a, int64_t tok, int64_t h) {
    return tok * a.b_t + h * a.b_h;
}
__host__ __device__ inline int64_t o_at(const GdrArgs &a, int64_t tok, int64_t h) {
    return tok * a.o_t + h * a.o_h;
}
// Whether the descriptor's strides index tokens as rows b * T + t (b stride = T x t stride, or
// a batch of one), each stride non-negative; `fast16` also asks 16-byte rows (multiples of 8
// elements for the vectors, the MFMA kernels' loads).
bool gdr_strides_ok(const dm_gdr_desc *d, bool step);
bool gdr_strides_16b(const dm_gdr_desc *d);

// Which tokens each chunk holds and which chunks each sequence: the arrays gdr_plan writes for
// packed sequences, or, for a batch of sequences of T tokens, in closed form from its `per` chunks a
// sequence (a launch and its latency less: 6144 tokens forward 143 -> 138 us).
struct GdrPlan {
    int32_t *seq_chunk0, *chunk_tok0, *chunk_len;  // [S + 1], [chunks], [chunks]
    int32_t *seq_order;                            // [S]: the sequences by chunk count, the most first
    int32_t closed, T, per;                        // closed: no arrays
    __device__ __forceinline__ int len(int64_t n) const {
        return closed ? min(kChunk, T - (int32_t)n % per * kChunk) : chunk_len[n];
    }
    __device__ __forceinline__ int64_t tok0(int64_t n) const {
        return closed ? (int64_t)((int32_t)n / per) * T + (int32_t)n % per * kChunk : chunk_tok0[n];
    }
    __device__ __forceinline__ int first(int64_t s) const { return closed ? (int32_t)s * per : seq_chunk0[s]; }
    __device__ __forceinline__ int64_t order(int64_t i) const { return closed ? i : seq_order[i]; }
};

// The f32 kernels' workspace: the plan, then per (chunk, head) f32 intermediates, rows of KP and
// VP columns (Dk and Dv padded with zeros to multiples of 64); names ending in T are transposed.
struct GdrWs {
    int64_t KP, VP, npart;
    GdrPlan plan;
    double *G;  // cumulative log-decay
    float *qn, *kn, *vp, *P, *W, *KT, *UT, *ScT, *VnT;
    // the backward's
    float *inv, *dop, *Tm, *Am, *WT, *dvlT, *F, *dSnT, *dVnT, *DPd, *dae, *gq, *gk, *dw, *dgv, *part;
};

int check_gdr(const dm_gdr_desc *d, const char *op, bool step);
// The longest-first order is kept for at most kOrderMax sequences; the identity beyond.
constexpr int64_t kOrderMax = 4096;
int64_t gdr_nseq(const dm_gdr_desc *d);
int64_t gdr_chunk_bound(const dm_gdr_desc *d);
// The plan's place in a workspace, and its launch (gdr_chunk.hip).
template <class F>
GdrPlan gdr_plan_layout(const dm_gdr_desc *d, F take) {
    const int64_t nc = gdr_chunk_bound(d), S = gdr_nseq(d);
    GdrPlan p{};
    if (!d->cu_seqlens) {
        p.closed = 1;
        p.T = (int32_t)d->t;
        p.per = (int32_t)((d->t + kChunk - 1) / kChunk);
        return p;
    }
    p.seq_chunk0 = (int32_t *)take((S + 1) * 4);
    p.chunk_tok0 = (int32_t *)take(nc * 4);
    p.chunk_len = (int32_t *)take(nc * 4);
    p.seq_order = (int32_t *)take(S * 4);
    return p;
}
int launch_plan(const dm_gdr_desc *d, const GdrPlan &p, hipStream_t st);

// MFMA forward and backward (gdr_chunk_mfma.hip): bf16/f16, Dk and Dv multiples of 8 up to 128
// (the products are 128 wide; columns past a width are held at zero).
bool gdr_mfma_takes(const dm_gdr_desc *d);
size_t gdr_mfma_fwd_workspace(const dm_gdr_desc *d);
int launch_gdr_mfma_fwd(const dm_gdr_desc *d, const void *q, const void *k, const void *v,
                        const void *g, const void *beta, const float *h0, void *out,
                        float *final_state, void *workspace, hipStream_t st);
size_t gdr_mfma_bwd_workspace(const dm_gdr_desc *d);
int launch_gdr_mfma_bwd(const dm_gdr_desc *d, const void *q, const void *k, const void *v,
                        const void *g, const void *beta, const float *h0, const void *d_out,
                        const float *d_final, void *dq, void *dk, void *dv, void *dg,
                        void *dbeta, float *dh0, void *workspace, hipStream_t st);
GdrArgs gdr_args(const dm_gdr_desc *d, const void *q, const void *k, const void *v,
                 const void *g, const void *beta, bool step = false);

}  // namespace dm
