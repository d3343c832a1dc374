// QASS "full" query scaling in one pass on the MFMA units: for each query head vector q (d
// wide, fp16),
//     out = q * base_scale[h] * (1 + tanh(W2 gelu(W1 q + b1) + b2))
// as QASSMaxScaling.forward computes it under fp16 autocast (src/synthefy_nori/model/
// layer.py:316-456: the gate MLP Linear(d, 64) -> GELU -> Linear(64, d), then the two
// multiplies), rounded where torch's separate ops round: each linear's fp32 sum with its bias
// rounded to fp16, GELU (erf form) and tanh evaluated in fp32 and rounded, 1 + t rounded, the
// two products rounded in turn. base_scale = log n * (1 + tanh(base_mlp(log n))) is one
// [heads, d] vector per call, formed by the caller. The separate ops make seven passes over
// the queries (two GEMMs, GELU, tanh, add, two multiplies, about 15 GB per 8.4 M vectors of
// 56); this kernel reads each query once and writes it once.
//
// Schedule. A wavefront takes 32 rows of one head at a time. The first GEMM runs transposed,
// H^T [64 hidden x 32 rows] = W1 [64 x d] Q^T, on v_mfma_f32_32x32x16_f16 with W1 (from LDS)
// as the A operand and the query rows (from global) as B. The second also runs transposed,
// G^T [d x 32 rows] = W2 [d x 64] H^T, and its B operand is the first's output registers
// after the bias, GELU and fp16 rounding, with no data movement: both GEMMs enumerate the
// k index of a 16-wide step in the order slot m of lane half hh <-> 4 hh + m % 4 + 8 (m / 4)
// (the rows a lane holds of a 32 x 32 result), the LDS copies of W1 and W2 are stored in that
// order, and the query elements a lane loads for the first GEMM are exactly the ones its
// second-GEMM results belong to. So the epilogue multiplies each result by the query value
// already in the lane's registers and writes 4 consecutive elements per 8-byte store.
//
// What bounds it: VALU work (64 GELUs and up to 64 tanhs a query vector) issues in 55 % of the cycles, MFMAs
// take 7 %, HBM 2.5 TB/s; the rest is the chain of a tile that four wavefronts a SIMD leave uncovered. With the math library's erf and tanh, a conversion for each rounding and 16,384
// workgroups that each staged the weights two bytes at a time for one or two tiles, 153,000 rows of 10
// heads of 56 took 235 us; a GELU of one polynomial and one exponential, packed fp16 products, the
// biases as the accumulators' start, and resident workgroups that walk tiles with the next tile's
// queries in flight take 156 us (0.34 GB; 68 us at the copy rate), 139,264 of 2 of 64 54 -> 32 us.
#include <math.h>

#include <algorithm>

#include "nori_common.h"

// each op rounds separately, as torch's do
#pragma clang fp contract(off)

namespace {

using namespace nori;

constexpr int kWaves = 4;
constexpr int kHid = 64;    // the gate MLP's hidden width (QASSMaxScaling's hidden_dim)
constexpr int kPitch = 72;  // f16 per LDS weight row (144 bytes: rows start on different banks)

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) _Float16 lds_f16;
typedef __attribute__((address_space(3))) f16x8 lds_f16x8;

// k index, within a 16-wide step, of slot m (0..7) of lane half hh: the order both GEMMs use
__host__ __device__ constexpr int kperm(int hh, int m) { return 4 * hh + (m & 3) + 8 * (m >> 2); }

__device__ __forceinline__ float r16(float v) { return round_to<NORI_F16>(v); }

__device__ __forceinline__ f16x8 join(u32x2_t lo, u32x2_t hi) {
    return __builtin_bit_cast(f16x8, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
}

__device__ __forceinline__ f16x2 pair_at(u32x2_t w, int i) {
    const uint32_t x = w[i];
    return __builtin_bit_cast(f16x2, x);
}

// two fp32 values rounded to fp16 (each product rounded to fp32 first)
__device__ __forceinline__ f16x2 pair16(float a, float b) { return f16x2{(_Float16)pin_f32(a), (_Float16)pin_f32(b)}; }

// GELU (the erf form) of an fp16 value in fp32: x Phi(x), with Phi(-|x|) = 2^L(|x|), L a polynomial of
// degree 8 fitted to log2 Phi(-a) over [0, 5.8] (past it the fp16 result is zero; the leading
// coefficient keeps L falling) by least squares reweighted towards the largest error: 1.4e-6. Of the
// 63,488 finite fp16 x, 51 round to another fp16 value than the exact GELU does; x / 2 (1 + erf(x / sqrt
// 2)) in fp32 with a correctly rounded erf misses 331, its sum cancelling for negative x. +-inf and NaN
// give what that expression gives.
__device__ __forceinline__ float gelu(float x) {
    const float a = fabsf(x);
    float p = fmaf(a, -4.04897598e-07f, 6.105983e-06f);
    p = fmaf(p, a, -1.43313975e-06f);
    p = fmaf(p, a, -0.00067129832f);
    p = fmaf(p, a, 0.00792131722f);
    p = fmaf(p, a, -0.0532461218f);
    p = fmaf(p, a, -0.458885486f);
    p = fmaf(p, a, -1.15115821f);
    p = fmaf(p, a, -0.999998548f);
    const float h = __builtin_amdgcn_exp2f(p);
    return x * (x >= 0.0f ? 1.0f - h : h);
}

// tanh in fp32: 1 - 2 / (exp(2 v) + 1), within 2e-7
__device__ __forceinline__ float tanh_f32(float v) {
    return fmaf(-2.0f, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v * 2.885390081777927f) + 1.0f), 1.0f);
}

// the biases of a 32 x 32 result's rows as a lane holds them (rows 8 g + 4 hh + 0..3; p at row 4 hh)
__device__ __forceinline__ f32x16 bias_tile(const float* p) {
    f32x16 r;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(p + 8 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[4 * g + i] = b[i];
    }
    return r;
}

template <int KS1, int NT2>  // k-steps of the first GEMM (ceil(d / 16)), 32-row tiles of the second (ceil(d / 32))
__global__ void __launch_bounds__(64 * kWaves, 4)
qass_gate_kernel(const uint16_t* q, int64_t rows, int heads, int d, int64_t qs, const uint16_t* w1,
                 const uint16_t* b1, const uint16_t* w2, const uint16_t* b2, const uint16_t* bs, uint16_t* out,
                 int64_t os, int64_t ntiles, int vec_w) {
    __shared__ __attribute__((aligned(16))) _Float16 w1s[kHid * kPitch];  // [hidden][k order], zeros past d
    __shared__ __attribute__((aligned(16))) _Float16 w2s[64 * kPitch];    // [output][k order], zero rows past d
    __shared__ __attribute__((aligned(16))) float b1s[kHid];
    __shared__ __attribute__((aligned(16))) float b2s[64];
    const int tid = threadIdx.x;
    // 4 consecutive LDS columns are 4 consecutive source columns (d is a multiple of 4: all in or out)
    if (vec_w) {
#pragma unroll
        for (int k = 0; k < 64 * 16 / (64 * kWaves); ++k) {
            const int i = tid + 64 * kWaves * k, j = i >> 4, p = 4 * (i & 15);
            const int c = 16 * (p >> 4) + kperm((p >> 3) & 1, p & 7);  // source column of LDS column p
            const u32x2_t a = *reinterpret_cast<const u32x2_t*>(w1 + j * d + min(c, d - 4));
            const u32x2_t b = *reinterpret_cast<const u32x2_t*>(w2 + min(j, d - 1) * kHid + c);
            *reinterpret_cast<u32x2_t*>(w1s + j * kPitch + p) = c < d ? a : u32x2_t{0u, 0u};
            *reinterpret_cast<u32x2_t*>(w2s + j * kPitch + p) = j < d ? b : u32x2_t{0u, 0u};
        }
    } else {
        for (int i = tid; i < 64 * 64; i += 64 * kWaves) {
            const int j = i >> 6, p = i & 63;
            const int c = 16 * (p >> 4) + kperm((p >> 3) & 1, p & 7);
            w1s[j * kPitch + p] = __builtin_bit_cast(_Float16, c < d ? w1[j * d + c] : (uint16_t)0);
            w2s[j * kPitch + p] = __builtin_bit_cast(_Float16, j < d ? w2[j * kHid + c] : (uint16_t)0);
        }
    }
    if (tid < 64) {
        b1s[tid] = f16_to_f32(b1[tid]);
        b2s[tid] = tid < d ? f16_to_f32(b2[tid]) : 0.0f;
    }
    __syncthreads();

    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const lds_f16* w1l = (const lds_f16*)w1s + l32 * kPitch + 8 * hh;
    const lds_f16* w2l = (const lds_f16*)w2s + l32 * kPitch + 8 * hh;
    // the lane's query elements of a tile: step s, half e holds q[16 s + 4 hh + 8 e + 0..3] (zeros
    // past d; the address clamped inside the row)
    auto load_q = [&](int64_t tile, u32x2_t (&qw)[KS1][2]) {
        const int64_t block = tile / heads, r = block * 32 + l32;
        const uint16_t* qr = q + min(r, rows - 1) * qs + (tile - block * heads) * d;
#pragma unroll
        for (int s = 0; s < KS1; ++s)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int c = 16 * s + 4 * hh + 8 * e;
                const u32x2_t v = *reinterpret_cast<const u32x2_t*>(qr + min(c, d - 4));
                qw[s][e] = c < d ? v : u32x2_t{0u, 0u};
            }
    };
    int64_t tile = (int64_t)blockIdx.x * kWaves + wave;
    const int64_t step = (int64_t)gridDim.x * kWaves;
    u32x2_t qw[KS1][2];
    if (tile < ntiles) load_q(tile, qw);
    for (; tile < ntiles; tile += step) {
        const int64_t block = tile / heads;
        const int h = (int)(tile - block * heads);
        const int64_t r = block * 32 + l32;  // this lane's row
        const bool live = r < rows;
        u32x2_t qn[KS1][2];  // the next tile's (the last loads its own again, unused)
        load_q(tile + step < ntiles ? tile + step : tile, qn);

        // H^T = W1 Q^T: acc1[t][4 g + i] is hidden unit 32 t + 8 g + 4 hh + i of row l32
        f32x16 acc1[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            acc1[t] = bias_tile(b1s + 32 * t + 4 * hh);
#pragma unroll
            for (int s = 0; s < KS1; ++s) {
                const f16x8 a = *reinterpret_cast<const lds_f16x8*>(w1l + 32 * t * kPitch + 16 * s);
                acc1[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, join(qw[s][0], qw[s][1]), acc1[t], 0, 0, 0);
            }
        }
        // fp16, GELU, fp16: hw[t][g] holds hidden units 32 t + 8 g + 4 hh + 0..3
        u32x2_t hw[2][4];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const f16x2 x = pair16(acc1[t][4 * g + 2 * i], acc1[t][4 * g + 2 * i + 1]);
                    hw[t][g][i] = __builtin_bit_cast(uint32_t, pair16(gelu((float)x[0]), gelu((float)x[1])));
                }

        // G^T = W2 H^T: step s of the hidden units takes hw[s / 2][2 (s % 2) + 0..1] as its B
        // operand; acc2[t][4 g + i] is output 32 t + 8 g + 4 hh + i of row l32
        f32x16 acc2[NT2];
#pragma unroll
        for (int t = 0; t < NT2; ++t) {
            acc2[t] = bias_tile(b2s + 32 * t + 4 * hh);
#pragma unroll
            for (int s = 0; s < kHid / 16; ++s) {
                const f16x8 a = *reinterpret_cast<const lds_f16x8*>(w2l + 32 * t * kPitch + 16 * s);
                acc2[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, join(hw[s >> 1][2 * (s & 1)], hw[s >> 1][2 * (s & 1) + 1]),
                                                                 acc2[t], 0, 0, 0);
            }
        }

        // out = (q * base_scale) * (1 + tanh(g + b2)); output o = 32 t + 8 g + 4 hh + i uses the
        // query element in qw[2 t + g / 2][g % 2], lane slot i. The products and the sum of fp16
        // values are packed fp16: each is rounded once from the exact value, as from fp32.
        const uint16_t* bsr = bs + (int64_t)h * d;
        uint16_t* orow = out + r * os + (int64_t)h * d;
#pragma unroll
        for (int t = 0; t < NT2; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                if (2 * t + (g >> 1) >= KS1) continue;  // past every head width of this kernel
                const int o = 32 * t + 8 * g + 4 * hh;
                const u32x2_t qv = qw[2 * t + (g >> 1)][g & 1];
                const u32x2_t sv = *reinterpret_cast<const u32x2_t*>(bsr + min(o, d - 4));
                u32x2_t ob;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const f16x2 v = pair16(acc2[t][4 * g + 2 * i], acc2[t][4 * g + 2 * i + 1]);
                    const f16x2 gs = pair16(tanh_f32((float)v[0]), tanh_f32((float)v[1])) + f16x2{(_Float16)1.0f, (_Float16)1.0f};
                    ob[i] = __builtin_bit_cast(uint32_t, (pair_at(qv, i) * pair_at(sv, i)) * gs);
                }
                if (live && o < d) *reinterpret_cast<u32x2_t*>(orow + o) = ob;
            }
#pragma unroll
        for (int s = 0; s < KS1; ++s)
#pragma unroll
            for (int e = 0; e < 2; ++e) qw[s][e] = qn[s][e];
    }
}

// The base scale: 64 outputs a workgroup. Every workgroup forms the 64 hidden units anew (a GELU a
// lane) rather than pass them through memory, and takes its 64 rows of w2 through LDS: element loads,
// so that weights of any alignment are taken (a parameter may be a view into a flat buffer), 16 a thread
// in flight at once (the index clamped: under a condition each waits for the last, 19-28 us). Weights are
// rounded to fp16 here, as autocast casts them, so the caller passes the parameters themselves: no cast to
// keep or to launch. As torch ops this vector of a few hundred values took eleven launches a layer (fill,
// two GEMMs with their bias copies, GELU, tanh, add, multiply, weight casts), 37 us of device time and
// three times that on the host; as one kernel about 3 us.
constexpr int kBaseThreads = 256;

template <int WT>
__global__ void __launch_bounds__(kBaseThreads)
qass_base_kernel(float log_n, const void* w1, const void* b1, const void* w2, const void* b2, int n_out, uint16_t* out) {
    __shared__ float hid[kHid];
    __shared__ float wt[64][kHid + 1];
    constexpr int PER = 64 * kHid / kBaseThreads;
    const int tid = threadIdx.x, o0 = blockIdx.x * 64, o = o0 + tid;
    const int64_t first = (int64_t)o0 * kHid;
    const int left = min(64, n_out - o0) * kHid;  // elements of this workgroup's rows
    const int hu = tid % kHid;
    const float u = load_elem<WT>(w1, hu), c = load_elem<WT>(b1, hu), bias = load_elem<WT>(b2, min(o0 + hu, n_out - 1));
    float w[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) w[i] = load_elem<WT>(w2, first + min(kBaseThreads * i + tid, left - 1));
    __builtin_amdgcn_sched_barrier(0);  // every load issued before the first is used
    const float l = r16(log_n);
    if (tid < kHid) hid[tid] = r16(gelu(r16(r16(u) * l + r16(c))));
#pragma unroll
    for (int i = 0; i < PER; ++i) wt[(kBaseThreads * i + tid) / kHid][(kBaseThreads * i + tid) % kHid] = r16(w[i]);
    __syncthreads();
    if (tid >= 64 || o >= n_out) return;
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < kHid; ++j) acc = fmaf(wt[tid][j], hid[j], acc);
    const float delta = r16(acc + r16(bias));
    out[o] = f32_to_f16(l * r16(1.0f + r16(tanh_f32(delta))));
}

template <int KS1, int NT2>
void launch(const uint16_t* q, int64_t rows, int heads, int d, int64_t qs, const uint16_t* w1, const uint16_t* b1,
            const uint16_t* w2, const uint16_t* b2, const uint16_t* bs, uint16_t* out, int64_t os, hipStream_t stream) {
    const int64_t ntiles = (rows + 31) / 32 * heads;
    // resident workgroups (four a CU): each stages the weights once and walks tiles
    const int64_t grid = std::min<int64_t>((ntiles + kWaves - 1) / kWaves, (int64_t)device_cus() * 4);
    hipLaunchKernelGGL((qass_gate_kernel<KS1, NT2>), dim3((unsigned)grid), dim3(64 * kWaves), 0, stream, q, rows,
                       heads, d, qs, w1, b1, w2, b2, bs, out, os, ntiles,
                       (int)((uintptr_t)w1 % 8 == 0 && (uintptr_t)w2 % 8 == 0));
}

}  // namespace

extern "C" int nori_qass_gate(const void* q, int dtype, int64_t rows, int32_t heads, int32_t d, int64_t q_row_stride,
                              const void* w1, const void* b1, const void* w2, const void* b2, int32_t hidden,
                              const void* base_scale, void* out, int64_t out_row_stride, void* stream_v) {
    clear_error();
    if (dtype != NORI_F16) return fail(NORI_ERR_UNSUPPORTED, "qass_gate: %s queries (float16 only)", dtype_name(dtype));
    if (hidden != kHid) return fail(NORI_ERR_UNSUPPORTED, "qass_gate: gate hidden width %d (64 only)", hidden);
    if (rows < 0 || heads <= 0 || d < 4 || d > 64 || d % 4)
        return fail(NORI_ERR_INVALID, "qass_gate: bad shape (%lld rows, %d heads of %d; d a multiple of 4 up to 64)",
                    (long long)rows, heads, d);
    if (q_row_stride < (int64_t)heads * d || out_row_stride < (int64_t)heads * d || q_row_stride % 4 ||
        out_row_stride % 4)
        return fail(NORI_ERR_INVALID, "qass_gate: row strides (%lld, %lld) must be multiples of 4 and at least %d",
                    (long long)q_row_stride, (long long)out_row_stride, heads * d);
    if (rows == 0) return NORI_OK;
    if (!q || !w1 || !b1 || !w2 || !b2 || !base_scale || !out) return fail(NORI_ERR_INVALID, "qass_gate: null pointer");
    if ((uintptr_t)q % 8 || (uintptr_t)out % 8 || (uintptr_t)base_scale % 8)
        return fail(NORI_ERR_INVALID, "qass_gate: q, base_scale and out must be 8-byte aligned");
    if ((rows + 31) / 32 * heads > ((int64_t)1 << 40)) return fail(NORI_ERR_UNSUPPORTED, "qass_gate: too many rows");
    const auto* qh = reinterpret_cast<const uint16_t*>(q);
    const auto* w1h = reinterpret_cast<const uint16_t*>(w1);
    const auto* b1h = reinterpret_cast<const uint16_t*>(b1);
    const auto* w2h = reinterpret_cast<const uint16_t*>(w2);
    const auto* b2h = reinterpret_cast<const uint16_t*>(b2);
    const auto* bsh = reinterpret_cast<const uint16_t*>(base_scale);
    auto* oh = reinterpret_cast<uint16_t*>(out);
    hipStream_t stream = (hipStream_t)stream_v;
    const int ks1 = (d + 15) / 16;
    switch (ks1) {
        case 1: launch<1, 1>(qh, rows, heads, d, q_row_stride, w1h, b1h, w2h, b2h, bsh, oh, out_row_stride, stream); break;
        case 2: launch<2, 1>(qh, rows, heads, d, q_row_stride, w1h, b1h, w2h, b2h, bsh, oh, out_row_stride, stream); break;
        case 3: launch<3, 2>(qh, rows, heads, d, q_row_stride, w1h, b1h, w2h, b2h, bsh, oh, out_row_stride, stream); break;
        default: launch<4, 2>(qh, rows, heads, d, q_row_stride, w1h, b1h, w2h, b2h, bsh, oh, out_row_stride, stream); break;
    }
    return launch_status("qass_gate");
}

extern "C" int nori_qass_base(float log_n, const void* w1, const void* b1, const void* w2, const void* b2, int w_dtype,
                              int32_t hidden, int32_t n_out, void* out, void* stream_v) {
    clear_error();
    if (hidden != kHid) return fail(NORI_ERR_UNSUPPORTED, "qass_base: hidden width %d (64 only)", hidden);
    if (w_dtype != NORI_F32 && w_dtype != NORI_F16 && w_dtype != NORI_BF16)
        return fail(NORI_ERR_UNSUPPORTED, "qass_base: unsupported weight dtype %s", dtype_name(w_dtype));
    if (n_out <= 0) return fail(NORI_ERR_INVALID, "qass_base: %d outputs", n_out);
    if (!w1 || !b1 || !w2 || !b2 || !out) return fail(NORI_ERR_INVALID, "qass_base: null pointer");
    const dim3 grid((unsigned)((n_out + 63) / 64)), block(kBaseThreads);
    hipStream_t stream = (hipStream_t)stream_v;
    auto o = reinterpret_cast<uint16_t*>(out);
    if (w_dtype == NORI_F32)
        hipLaunchKernelGGL((qass_base_kernel<NORI_F32>), grid, block, 0, stream, log_n, w1, b1, w2, b2, n_out, o);
    else if (w_dtype == NORI_F16)
        hipLaunchKernelGGL((qass_base_kernel<NORI_F16>), grid, block, 0, stream, log_n, w1, b1, w2, b2, n_out, o);
    else
        hipLaunchKernelGGL((qass_base_kernel<NORI_BF16>), grid, block, 0, stream, log_n, w1, b1, w2, b2, n_out, o);
    return launch_status("qass_base");
}
