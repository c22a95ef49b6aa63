// Attention forward and backward: the entry points and their contract checks. The 16-bit MFMA
// kernels (attention_fwd.hip, attention_mfma_bwd.hip) run where they take the call, the f32 ones
// (attention_f32.hip) elsewhere.
#include <algorithm>
#include <string>

#include "attention_kernels.h"
#include "dm_common.h"

namespace dm {

// ------------------------------------------------------------------------------------------
// Contract checks (check_shapes, crates/dash-ops/src/attention.rs:551-590)
// ------------------------------------------------------------------------------------------

int check_attention(const dm_attention_desc *d, const char *op) {
    std::string o(op);
    if (!d) return refuse(o + ": null descriptor");
    if (d->b < 0 || d->tq < 0 || d->tk < 0 || d->hq < 0 || d->hkv < 0 || d->d < 0)
        return refuse(o + ": negative dimension");
    if (d->hkv <= 0 || d->hq % d->hkv != 0)
        return refuse(o + ": the query heads (" + std::to_string(d->hq) +
                      ") must be a multiple of the key-value heads (" + std::to_string(d->hkv) +
                      ")");
    if (d->dtype != DM_F32 && d->dtype != DM_BF16 && d->dtype != DM_F16)
        return refuse(o + ": dtype must be f32, bf16 or f16");
    if (d->mask_kind == DM_MASK_KEY_PADDING && !d->key_padding && d->b * d->tk > 0)
        return refuse(o + ": the key padding mask is missing");
    if (d->mask_kind == DM_MASK_PACKED) {
        if (d->b != 1) return refuse(o + ": packed sequences lie along the time, B = 1");
        if (d->nseq < 1 || !d->cu_seqlens_q || !d->cu_seqlens_k)
            return refuse(o + ": cu_seqlens_q and cu_seqlens_k are [S + 1], one S");
    }
    if (d->mask_kind < 0 || d->mask_kind > 2) return refuse(o + ": unknown mask kind");
    if (d->strided) {
        const AttnStrides s = attn_strides(d);
        if (!strides_ok(s.q) || !strides_ok(s.k) || !strides_ok(s.v) || !strides_ok(s.o) ||
            !strides_ok(s.g))
            return refuse(o + ": strides must not be negative");
    }
    if (d->d > 256)
        return refuse(o + ": head dimension " + std::to_string(d->d) +
                      " above 256 is not implemented");
    return DM_OK;
}

}  // namespace dm

using namespace dm;

extern "C" {

size_t dm_attention_fwd_workspace(const dm_attention_desc *desc) {
    return desc ? mfma_fwd_workspace(desc) : 0;
}

int dm_attention_fwd(const dm_attention_desc *desc, const void *q, const void *k, const void *v,
                     void *o, float *lse, void *workspace, size_t workspace_bytes,
                     void *stream) {
    int rc = check_attention(desc, "attention");
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const MaskInfo m = mask_info(desc);
    const float scale = scale_of(desc);
    const int64_t rows = desc->b * desc->tq * desc->hq;
    if (rows == 0) return DM_OK;
    if (desc->tk == 0 || desc->d == 0) {
        // no key at all: zeros and a log-sum-exp of -inf (reference.rs:312-325)
        fill_zero(o, rows * desc->d * dtype_bytes(desc->dtype), st);
        fill_f32(lse, -INFINITY, rows, st);
        DM_LAUNCH_CHECK("attention: fill");
        return DM_OK;
    }
    if (mfma_fwd_takes(desc, q, k, v))
        return launch_attn_fwd_mfma(m, desc, scale, q, k, v, o, lse, workspace, workspace_bytes, st);
    return launch_attn_fwd_f32(m, desc, scale, q, k, v, o, lse, st);
}

size_t dm_attention_bwd_workspace(const dm_attention_desc *desc) {
    if (!desc) return 0;
    const size_t rows = (size_t)(desc->b * desc->tq * desc->hq);
    // the MFMA kernels' delta and the rest of theirs, or the f32 kernels' (which of them runs also
    // depends on the pointers' alignment)
    return std::max(align_up(rows * sizeof(float)) + mfma_bwd_workspace(desc), attn_bwd_f32_workspace(desc));
}

int dm_attention_bwd(const dm_attention_desc *desc, const void *q, const void *k, const void *v,
                     const void *o, const float *lse, const void *d_o, void *dq, void *dk,
                     void *dv, void *workspace, size_t workspace_bytes, void *stream) {
    int rc = check_attention(desc, "attention_backward");
    if (rc) return rc;
    if (workspace_bytes < dm_attention_bwd_workspace(desc))
        return refuse("attention_backward: the workspace is smaller than "
                      "dm_attention_bwd_workspace");
    hipStream_t st = (hipStream_t)stream;
    const MaskInfo m = mask_info(desc);
    const float scale = scale_of(desc);
    const int64_t qrows = desc->b * desc->tq * desc->hq, krows = desc->b * desc->tk * desc->hkv;
    const size_t eb = dtype_bytes(desc->dtype);
    if (qrows == 0 && krows == 0) return DM_OK;
    if (qrows == 0 || krows == 0 || desc->d == 0) {
        fill_zero(dq, qrows * desc->d * eb, st);
        fill_zero(dk, krows * desc->d * eb, st);
        fill_zero(dv, krows * desc->d * eb, st);
        DM_LAUNCH_CHECK("attention_backward: fill");
        return DM_OK;
    }
    float *delta = (float *)workspace;
    char *rest = (char *)workspace + align_up(qrows * sizeof(float));
    if (mfma_bwd_takes(desc, q, k, v, o, d_o))
        return launch_attn_bwd_mfma(m, desc, scale, q, k, v, o, lse, d_o, dq, dk, dv, delta,
                                    rest, st);
    return launch_attn_bwd_f32(m, desc, scale, q, k, v, o, lse, d_o, dq, dk, dv, workspace, st);
}

}  // extern "C"
