// One dense layer over query rows against its context cache (EncoderBaseLayer.forward_test_with_cache,
// src/synthefy_nori/model/layer.py:1915-1967, layer_arch "smf"), its nine launches issued by one call.
//
// For small tables a layer's kernels take a few microseconds each and the Python between them two to
// three times that: the 6m stack over 256 x 9 query tokens spent 4.9 ms of host time on 1.4 ms of
// kernels. The kernels are the ones the module issues one by one -- row norm, q projection, QASS base
// and gate, cached attention, SwiGLU, q|k|v projection, feature attention -- with the projections on
// nori_linear_f16 at every row count and the residual updates and norms inside the output
// projections and the SwiGLU kernel.
#include "nori_common.h"

namespace {

using namespace nori;

int64_t padded(int64_t bytes) { return (bytes + 255) / 256 * 256; }

}  // namespace

extern "C" int64_t nori_dense_apply_scratch_bytes(int64_t tables, int64_t rows, int64_t groups, int32_t embed,
                                                  int32_t heads, int64_t nk) {
    if (tables <= 0 || rows <= 0 || groups <= 0 || embed <= 0 || heads <= 0 || embed % heads || nk <= 0) return 0;
    const int64_t n = tables * rows * groups, d = embed / heads;
    const int64_t seq = nori_icl_attention_workspace_size(tables * groups, rows, heads, (int32_t)d, nk);
    const int64_t feat = nori_icl_attention_workspace_size(tables * rows, groups, heads, (int32_t)d, groups);
    // two [n, embed] operands, one [n, 3 embed] projection, the base scale, the attentions' partials
    return 2 * padded(2 * n * embed) + padded(6 * n * embed) + padded(2 * embed) + padded(seq > feat ? seq : feat);
}

extern "C" int nori_dense_apply(const nori_dense_apply_args* p, void* stream) {
    clear_error();
    if (!p) return fail(NORI_ERR_INVALID, "dense_apply: null arguments");
    const int64_t B = p->tables, R = p->rows, G = p->groups, n = B * R * G;
    const int e = p->embed, h = p->heads;
    if (B <= 0 || R <= 0 || G <= 0 || h <= 0 || e <= 0 || e % h || p->nk <= 1)
        return fail(NORI_ERR_INVALID, "dense_apply: bad shape (%lld x %lld x %lld, %d heads of %d, %lld keys)", (long long)B,
                    (long long)R, (long long)G, h, e, (long long)p->nk);
    if (p->qkv_dtype != NORI_F16 && p->qkv_dtype != NORI_F32)
        return fail(NORI_ERR_UNSUPPORTED, "dense_apply: %s q|k|v weights", dtype_name(p->qkv_dtype));
    if (e != 128 && e != 256) return fail(NORI_ERR_UNSUPPORTED, "dense_apply: width %d is not 128 or 256", e);
    const int d = e / h;
    const int64_t need = nori_dense_apply_scratch_bytes(B, R, G, e, h, p->nk);
    if (!p->scratch || p->scratch_bytes < need)
        return fail(NORI_ERR_INVALID, "dense_apply: %lld scratch bytes given, %lld needed", (long long)p->scratch_bytes,
                    (long long)need);
    char* at = reinterpret_cast<char*>(p->scratch);
    auto take = [&](int64_t bytes) { char* r = at; at += padded(bytes); return (void*)r; };
    void* a0 = take(2 * n * e);
    void* a1 = take(2 * n * e);
    void* qkv = take(6 * n * e);
    void* base = take(2 * e);
    void* ws = at;
    const int64_t ws_bytes = p->scratch_bytes - (at - reinterpret_cast<char*>(p->scratch));
    const float scale = p->logit_scale;
    int st;
#define NORI_STEP(call) do { if ((st = (call)) != NORI_OK) return st; } while (0)
    // sequence attention, in [table, group, row] order
    NORI_STEP(nori_rms_norm_rows(p->x, n, e, G, R, R * G * e, e, G * (int64_t)e, p->eps_seq, a0, NORI_F16, stream));
    NORI_STEP(nori_linear_f16(a0, 1, 1, n, e, 0, 0, e, p->w_q, e, e, a1, 0, 0, e, stream));
    NORI_STEP(nori_qass_base(p->log_n, p->base_w1, p->base_b1, p->base_w2, p->base_b2, p->base_dtype, p->qass_hidden, e,
                             base, stream));
    NORI_STEP(nori_qass_gate(a1, NORI_F16, n, h, d, e, p->gate_w1, p->gate_b1, p->gate_w2, p->gate_b2, p->qass_hidden,
                             base, a0, e, stream));
    NORI_STEP(nori_icl_attention(a0, NORI_F16, B * G, R, h, d, R * e, e, d, p->kv, p->kv_dtype, p->kv_scales, p->nk,
                                 p->kv_heads, p->kv_bg, p->kv_row, p->kv_half, p->sc_bg, p->sc_row, p->sc_half, scale, a1,
                                 NORI_F16, R * e, e, d, nullptr, 0, ws, ws_bytes, stream));
    // x + alpha u into the new stream, then the MLP with its residual, each with the next norm
    NORI_STEP(nori_linear_f16_residual(a1, B, R, G, e, R * G * e, e, R * (int64_t)e, p->w_out, e, NORI_F16, p->alpha, p->x, R * G * e,
                                       G * (int64_t)e, e, p->out, p->eps_mlp, a0, R * G * e, G * (int64_t)e, e, stream));
    NORI_STEP(nori_swiglu_mlp_residual_rms_norm(a0, NORI_F16, n, e, e, p->gate_up, p->down, p->hidden, p->alpha, p->out, e,
                                                e, p->eps_feat, a1, n, 0, e, stream));
    // feature attention over each row's groups
    if (p->qkv_dtype == NORI_F32)
        NORI_STEP(nori_linear_f16_w32(a1, 1, 1, n, e, 0, 0, e, reinterpret_cast<const float*>(p->w_qkv), e, 3 * e, qkv, 0, 0,
                                      3 * e, stream));
    else
        NORI_STEP(nori_linear_f16(a1, 1, 1, n, e, 0, 0, e, p->w_qkv, e, 3 * e, qkv, 0, 0, 3 * e, stream));
    const uint16_t* q3 = reinterpret_cast<const uint16_t*>(qkv);
    NORI_STEP(nori_icl_attention(q3, NORI_F16, B * R, G, h, d, 3 * G * e, 3 * e, d, q3 + e, NORI_F16, nullptr, G, h,
                                 3 * G * e, 3 * e, e, 0, 0, 0, scale, a0, NORI_F16, G * e, e, d, nullptr, 0, ws, ws_bytes,
                                 stream));
    NORI_STEP(nori_linear_f16_residual(a0, 1, 1, n, e, 0, 0, e, p->w_feat_out, e, NORI_F16, p->alpha, p->out, 0, 0, e, p->out, 0.f,
                                       nullptr, 0, 0, 0, stream));
#undef NORI_STEP
    return NORI_OK;
}
