// Entry points the package's own modules call that are not part of the C ABI in nori_hip.h: they
// carry no compatibility promise and change with the modules that bind them. Same conventions:
// device pointers, a nori_status return, the message in nori_last_error().
#pragma once

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

// Moves with every change of a signature or struct below; the package binds one version.
#define NORI_OPS_VERSION 4
int nori_ops_version(void);

// QASS base scale of one key count (QASSMaxScaling.forward's base branch, src/synthefy_nori/model/
// layer.py:316-456, under fp16 autocast): with l = T(log n), T the rounding to fp16,
//     out[o] = T(l * T(1 + T(tanh(T(W2 h + b2)[o])))),  h = T(gelu(T(w1 l + b1))),
// fp32 sums, gelu the erf form. w1, b1 [hidden], w2 [n_out, hidden], b2 [n_out], contiguous, of
// w_dtype (fp32, fp16 or bf16), each rounded by T first; out [n_out] fp16; hidden is 64.
int nori_qass_base(float log_n, const void* w1, const void* b1, const void* w2, const void* b2, int w_dtype,
                   int32_t hidden, int32_t n_out, void* out, void* stream);

// nori_rms_norm_to (no weight) of fp32 rows at three strides, written as contiguous fp16 or bf16
// rows: row r = (i0 * d1 + i1) * d2 + i2 of x starts at element i0 * s0 + i1 * s1 + i2 * s2. Bit for
// bit nori_rms_norm_to of the gathered rows. Rows of more than 1024 elements, cols not a multiple
// of 4, 2^31 rows or more and unaligned operands return NORI_ERR_UNSUPPORTED.
int nori_rms_norm_rows(const float* x, int64_t rows, int32_t cols, int64_t d1, int64_t d2, int64_t s0, int64_t s1,
                       int64_t s2, float eps, void* y, int y_dtype, void* stream);

// nori_linear_f16 of fp32 weights, each rounded to fp16 as it is staged: bit for bit nori_linear_f16 of
// their fp16 cast. weight 16-byte aligned, its row stride a multiple of 4.
int nori_linear_f16_w32(const void* x, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k, int64_t x_outer_stride,
                        int64_t x_mid_stride, int64_t x_row_stride, const float* weight, int64_t w_row_stride, int32_t n,
                        void* y, int64_t y_outer_stride, int64_t y_mid_stride, int64_t y_row_stride, void* stream);

// nori_linear_f16 followed by the per-head RMSNorm of its first norm_cols columns, taken as heads
// of 64 (a multiple of 64): each head row v becomes T(T(v * rsqrt(mean(v^2) + eps)) * gain) with T
// the rounding to fp16 and gain [64] of gain_dtype -- the projection and the q/k norm pass over it
// (MultiheadAttention with qk_norm, layer.py:497-500, 1122-1134), up to the order of the sums.
int nori_linear_f16_head_norm(const void* x, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k,
                              int64_t x_outer_stride, int64_t x_mid_stride, int64_t x_row_stride, const void* weight,
                              int64_t w_row_stride, int32_t n, void* y, int64_t y_outer_stride, int64_t y_mid_stride,
                              int64_t y_row_stride, const void* gain, int gain_dtype, float eps, int32_t norm_cols,
                              void* stream);

// nori_linear_f16_residual_rms_norm with the updated stream written to x_out, at x's strides (x_out may
// be x), with y NULL without the norm, and of fp16 or fp32 weights (w_dtype; fp32 as nori_linear_f16_w32).
int nori_linear_f16_residual(const void* a, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k,
                             int64_t a_outer_stride, int64_t a_mid_stride, int64_t a_row_stride, const void* weight,
                             int64_t w_row_stride, int w_dtype, float alpha, const float* x, int64_t x_outer_stride,
                             int64_t x_mid_stride, int64_t x_row_stride, float* x_out, float eps, void* y,
                             int64_t y_outer_stride, int64_t y_mid_stride, int64_t y_row_stride, void* stream);

// nori_swiglu_mlp_residual_rms_norm without the norm (fp16 x, width 128 or 256).
int nori_swiglu_mlp_residual(const void* x, int64_t rows, int32_t width, int64_t x_row_stride, const void* w_gate_up,
                             const void* w_down, int32_t hidden, float alpha, float* stream_rows,
                             int64_t stream_row_stride, void* stream);

// One dense "smf" layer over query rows against its context cache, every launch from one call
// (dense_layer.hip): x [tables, rows, groups, embed] fp32 contiguous is left as it is, out (the same
// shape) takes the layer's output. Weights fp16 (the QASS base MLP's of base_dtype), contiguous: w_q, w_out,
// w_feat_out [embed, embed], w_qkv [3 embed, embed], the QASS MLPs ([64, 1 | head width], [64],
// [embed | head width, 64], ...), gate_up [2 hidden, embed] and down [embed, hidden] with hidden a
// multiple of 32. The cache as nori_icl_attention takes it; alpha the deep-norm factor as rounded to
// fp16. embed is 128 or 256 (the norm after the MLP is over embed columns); two keys or more.
typedef struct {
    int64_t tables, rows, groups;
    int32_t embed, heads;
    const float* x;
    float* out;
    const void *w_q, *w_out, *w_qkv, *w_feat_out;
    const void *base_w1, *base_b1, *base_w2, *base_b2, *gate_w1, *gate_b1, *gate_w2, *gate_b2;
    int32_t qkv_dtype, base_dtype, qass_hidden;
    const void *gate_up, *down;
    int32_t hidden;
    float eps_seq, eps_mlp, eps_feat, alpha, logit_scale, log_n;
    const void* kv;
    int32_t kv_dtype;
    const float* kv_scales;
    int64_t nk;
    int32_t kv_heads;
    int64_t kv_bg, kv_row, kv_half, sc_bg, sc_row, sc_half;
    void* scratch;
    int64_t scratch_bytes;
} nori_dense_apply_args;

int64_t nori_dense_apply_scratch_bytes(int64_t tables, int64_t rows, int64_t groups, int32_t embed, int32_t heads, int64_t nk);
int nori_dense_apply(const nori_dense_apply_args* args, void* stream);

#ifdef __cplusplus
}
#endif
