// Fused SwiGLU feed-forward sublayer on the MFMA units:
//     y = (silu(x Wg^T) * (x Wu^T)) Wd^T
// for fp16 rows (SwiGLUMLP.forward, src/synthefy_nori/model/layer.py:261-274, under fp16
// autocast). The unfused sequence writes the [rows, 2h] gate|up projection to HBM, reads it
// back for the gate and writes [rows, h], and the down projection reads that again; here the
// hidden activations of a row tile never leave the CU.
//
// Workgroup: four wavefronts of 32 rows each, two (width 128: three) of them on a CU. Per chunk of
// 16 hidden units:
//   1. up:   G^T, U^T [16 hidden x 32 rows] = W{g,u}[chunk] . X^T on v_mfma_f32_16x16x32_f16 (A:
//            weight rows staged in LDS; B: the wavefront's X fragments, held in registers for the
//            whole kernel);
//   2. gate: a = f16(f16(silu(f16(g))) * f16(u)) in registers; one v_permlane16_swap per word
//            pair turns the C layout into the B operand of step 3;
//   3. down: Y^T [width x 32 rows] += Wd[:, chunk] . a^T on v_mfma_f32_32x32x16_f16, accumulated
//            over every chunk.
// The weight chunks (gate and up rows [32, width], down columns [width, 16]) go global -> LDS
// directly (buffer loads to LDS: no staging registers, no LDS write instructions) into a
// double-buffered ring, the next chunk's loads in flight while the current chunk computes; one
// barrier per chunk.
//
// What bounds it: no one pipe. An LDS read of a weight operand serves one 32-cycle MFMA of one wavefront,
// and the gate and the epilogue are VALU work. Counters, as shares of the kernel's cycles: width 128 (655,360
// rows) MFMA 36 %, VALU issue 52 %, LDS issue 30 %, bank conflicts 14 %, with the residual epilogue 24, 50, 24 and
// 9 % at 3 TB/s; width 256 with it (163,840 rows, hidden 704) 36, 35, 24 and 13 %; width 352, one wavefront per
// SIMD, 19, 13, 11 and 7 %: latency. Chunks of 32 on 32x32x16 MFMAs took 32 registers for G^T and U^T, which left one
// wavefront per SIMD at width 256 (one workgroup of 108 KB), each operand read just before its
// MFMA: 163,840 rows of 256 (hidden 704) 315 us plain and 380 us with the residual epilogue, against
// 210 us (845 TFLOP/s) and 246 us; 655,360 rows of 128 (256) 262 and 362 against 220 and 291 us
// (3.5 TB/s); 33,792 rows of 352 (960) 185 against 151 us. Workgroups of eight wavefronts, which
// stage a chunk for twice the rows: 230, 298, 251 and 355 us.
//
// nori_swiglu_mlp_residual_rms_norm ends the kernel with the deep-norm residual update of an
// fp32 stream and the next sublayer's RMSNorm (no weight) instead of writing y: per row
// x = x + f16(f16(y) * alpha) in place, then f16(x * rsqrt(mean(x^2) + eps)) over norm
// groups of NW columns (the whole row, or 128-column tokens of a wider row) -- bit for bit
// nori_swiglu_mlp followed by nori_residual_add_rms_norm: the sum of squares runs in that
// kernel's order (an fma chain over each 4-column chunk, then pairwise over the chunk index
// bits from the highest).
//
// Rounding: the projections sum in fp32 and round to fp16 as hipBLASLt's fp16 GEMMs do, but in
// their own order, so a value can differ from the unfused sequence's by one fp16 ulp where the
// fp32 sum sits at a rounding boundary. silu(g) = g * rcp(1 + 2^(-g log2 e)) with the hardware
// exp2 and reciprocal, within a few fp32 ulp of torch's g / (1 + exp(-g)) before its rounding
// to fp16; the product of two fp16 values is exact in fp32, so f16(s * u) is one packed fp16
// multiply.
#include "nori_common.h"

// the residual epilogue rounds every op separately, as torch does
#pragma clang fp contract(off)

namespace {

using namespace nori;

// gate | up weights are addressed by 32-bit byte offsets (2 GiB)
constexpr int64_t kMaxWeights = 0x7fffffff / 4;
constexpr float kLog2eF = 1.4426950408889634f;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ uint32_t pack_f16(float a, float b) {
    const f16x2 h = f16x2{(_Float16)pin_f32(a), (_Float16)pin_f32(b)};
    return __builtin_bit_cast(uint32_t, h);
}

// The gate of two hidden units: f16(f16(silu(f16(g))) * f16(u)) as one packed word.
__device__ __forceinline__ uint32_t gate_pair(float g0, float g1, float u0, float u1) {
    const f16x2 gh = f16x2{(_Float16)g0, (_Float16)g1};
    const f16x2 uh = f16x2{(_Float16)u0, (_Float16)u1};
    const float a = (float)gh[0], b = (float)gh[1];
    const float s0 = a * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(a * -kLog2eF));
    const float s1 = b * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(b * -kLog2eF));
    const f16x2 sh = f16x2{(_Float16)s0, (_Float16)s1};
    return __builtin_bit_cast(uint32_t, sh * uh);
}

// The residual epilogue's operands (NW > 0): the fp32 stream (row r at xs + r * xs_row, updated
// in place) and the normalized output, norm group q = r * (E / NW) + k at
// (q / y_group) * y_group_stride + (q % y_group) * y_row_stride elements from y.
struct ResEpi {
    float* xs;
    int64_t xs_row;
    float alpha, eps;
    int64_t y_group, y_group_stride, y_row_stride;
};

// The epilogue's rows: PASSES * 4 rows from rh, their u = f16(y) in LDS at ut (rows E + 8 f16 apart),
// written as y, or into the stream and its norm (NW > 0). A stream row moves in 256-byte pieces (lane
// l takes rows 4p + l/16 at columns 64q + 4 (l % 16)) and an output row whole.
template <int E, int NW, int PASSES>
__device__ __forceinline__ void emit_rows(const _Float16* ut, int64_t rh, int64_t rows, int lane, uint16_t* __restrict__ y,
                                          int64_t ys, const ResEpi& ep) {
    constexpr int UP = E + 8, NCH = (E + 63) / 64, ROWS = 4 * PASSES;
    if constexpr (NW == 0) {
        constexpr int LPR = E / 8;  // 16-byte pieces per row
#pragma unroll
        for (int k = 0; k < (ROWS * LPR + 63) / 64; ++k) {
            const int e = lane + 64 * k, rr = e / LPR, c = 8 * (e % LPR);
            if (rr < ROWS && rh + rr < rows)
                *reinterpret_cast<u32x4*>(y + (rh + rr) * ys + c) = *reinterpret_cast<const u32x4*>(ut + rr * UP + c);
        }
    } else {
        static_assert(NW == 0 || (E % 64 == 0 && NW % 64 == 0), "norm groups of whole 64-column chunks");
        constexpr int GC = NW > 0 ? NW / 64 : 1, GROUPS = NW > 0 ? E / NW : 1;
        const int c4 = 4 * (lane & 15);
        f32x4 v[PASSES][NCH];
        float part[PASSES][NCH];
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int rr = 4 * p + (lane >> 4);
            // (rows past the last, a whole wavefront's in the last workgroup, read the last again)
            const float* xr = ep.xs + (rh + rr < rows ? rh + rr : rows - 1) * ep.xs_row + c4;
#pragma unroll
            for (int q = 0; q < NCH; ++q) v[p][q] = *reinterpret_cast<const f32x4*>(xr + 64 * q);
        }
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int rr = 4 * p + (lane >> 4);
            const bool ok = rh + rr < rows;
            float* xr = ep.xs + (ok ? rh + rr : rows - 1) * ep.xs_row + c4;
#pragma unroll
            for (int q = 0; q < NCH; ++q) {
                const u32x2 uw = *reinterpret_cast<const u32x2*>(ut + rr * UP + 64 * q + c4);
                float s = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float u = f16_to_f32((uint16_t)(uw[e >> 1] >> (16 * (e & 1))));
                    v[p][q][e] = v[p][q][e] + round_to<NORI_F16>(u * ep.alpha);
                    s = fmaf(v[p][q][e], v[p][q][e], s);
                }
                part[p][q] = s;
                if (ok) *reinterpret_cast<f32x4*>(xr + 64 * q) = v[p][q];
            }
        }
        if (y) {  // uniform over the launch (null: no norm)
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
                const int64_t row = rh + 4 * p + (lane >> 4);
#pragma unroll
                for (int k = 0; k < GROUPS; ++k) {
                    // chunk 16 q + l % 16 of the group: pairs over its index bits from the highest, the
                    // q's in the lane, then the 16 lanes
                    float t[GC];
#pragma unroll
                    for (int q = 0; q < GC; ++q) t[q] = part[p][k * GC + q];
#pragma unroll
                    for (int st = GC / 2; st >= 1; st >>= 1) {
#pragma unroll
                        for (int q = 0; q < st; ++q) t[q] = t[q] + t[q + st];
                    }
                    float tot = t[0];
#pragma unroll
                    for (int off = 8; off > 0; off >>= 1) tot = tot + __shfl_xor(tot, off);
                    const float inv = rsqrtf(tot / (float)(NW > 0 ? NW : 1) + ep.eps);
                    if (row < rows) {
                        const int64_t qr = row * GROUPS + k;
                        uint16_t* yr = y + (qr / ep.y_group) * ep.y_group_stride + (qr % ep.y_group) * ep.y_row_stride + c4;
#pragma unroll
                        for (int q = 0; q < GC; ++q) {
                            uint16_t o[4];
#pragma unroll
                            for (int e = 0; e < 4; ++e) o[e] = f32_to_f16(v[p][k * GC + q][e] * inv);
                            *reinterpret_cast<u32x2*>(yr + 64 * q) =
                                u32x2{o[0] | ((uint32_t)o[1] << 16), o[2] | ((uint32_t)o[3] << 16)};
                        }
                    }
                }
            }
        }
    }
}

// u = f16(y) of a lane's tile t (element 4j + i is output 32t + 8j + 4hh + i of its row) into its row at ur
__device__ __forceinline__ void stage_tile(const f32x16& v, _Float16* ur) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
        *reinterpret_cast<u32x2*>(ur + 8 * j) = u32x2{pack_f16(v[4 * j], v[4 * j + 1]), pack_f16(v[4 * j + 2], v[4 * j + 3])};
}

// The epilogue for a wavefront's 32 rows from r0, from its Y^T tiles. u goes through the wavefront's
// LDS slice, 16 rows at a time, into a row layout, where the MFMA layout touched 32 rows in 32-byte
// pieces an instruction. The slice is the wavefront's own: LDS runs its accesses in order.
template <int E, int NW>
__device__ __forceinline__ void write_rows(const f32x16 (&yt)[E / 32], int64_t r0, int64_t rows, int lane, _Float16* ut,
                                           uint16_t* __restrict__ y, int64_t ys, const ResEpi& ep) {
    const int l32 = lane & 31, hh = lane >> 5;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if ((l32 >> 4) == h) {
#pragma unroll
            for (int t = 0; t < E / 32; ++t) stage_tile(yt[t], ut + (l32 & 15) * (E + 8) + 4 * hh + 32 * t);
        }
        asm volatile("" ::: "memory");
        emit_rows<E, NW, 4>(ut, r0 + 16 * h, rows, lane, y, ys, ep);
        asm volatile("" ::: "memory");
    }
}

// Few rows (SPLIT kernels, width 128): up to this many per CU, a workgroup owns 32 rows and its four
// wavefronts take every fourth chunk each, from buffers of their own, so no barrier orders them; their
// partial sums meet in LDS in the order of the wavefronts. With a whole workgroup to 128 rows, 2,304
// rows are 18 workgroups, each one chain of 16 chunks: 17.1 us (hidden 256, with the residual epilogue)
// against 13.6 us here, 13.2 against 10.0 us plain; 9,513 rows are past the line, at 19.6 us.
constexpr int kSplitRowsPerCu = 32;
constexpr int split_width(int e) { return e == 128; }

// Operand reads in flight: each LDS read is issued kAhead reads before its MFMA and the order is
// fenced; left to itself the compiler reads an operand just before its MFMA and waits.
constexpr int kAhead = 4;

// 16 bytes per lane from byte voff + soff of a buffer to LDS at dst + 16 * lane (dst uniform)
__device__ __forceinline__ void buffer_to_lds(__amdgpu_buffer_rsrc_t r, lds_void* dst, uint32_t voff, int soff) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, (int)voff, soff, 0, 0);
#endif
}

template <int E>
struct MlpGeom {
    static constexpr int NWAVES = 4;
    static constexpr int THREADS = 64 * NWAVES;
    static constexpr int HC = 16;         // hidden units per chunk
    static constexpr int S = E / 32;      // k-steps of the up projection
    static constexpr int OT = E / 32;     // 32-row tiles of Y^T
    // 16-byte granules of a chunk in LDS: 16 gate then 16 up rows of E/8 granules and one of padding,
    // then E down rows of 2 granules and one of padding; both parts fill whole wavefront loads
    static constexpr int GROW = E / 8 + 1;
    static constexpr int GLOADS = (2 * HC * GROW + 63) / 64;
    static constexpr int DLOADS = (3 * E + 63) / 64;
    static constexpr int LOADS = GLOADS + DLOADS;
    static constexpr int BUF = LOADS * 64 * 8;  // f16 per ring buffer
    static_assert(NWAVES * 16 * (E + 8) <= 2 * BUF, "the epilogue's rows fit the ring");
};

template <int E, int NW, bool SPLIT>
__global__ void __launch_bounds__(MlpGeom<E>::THREADS)
__attribute__((amdgpu_waves_per_eu(SPLIT ? 1 : (E <= 128 ? 3 : (E <= 256 ? 2 : 1)))))
swiglu_mlp_kernel(const uint16_t* __restrict__ x, int64_t rows, int64_t xs, const uint16_t* __restrict__ wgu,
                    const uint16_t* __restrict__ wd, int hp, uint16_t* __restrict__ y, int64_t ys, const ResEpi ep) {
    using G = MlpGeom<E>;
    constexpr int SHARE = SPLIT ? 1 : G::NWAVES;  // wavefronts that stage and read a buffer together
    constexpr int CSTEP = SPLIT ? G::NWAVES : 1;  // chunks from one of a wavefront's to its next
    constexpr int PER = (G::LOADS + SHARE - 1) / SHARE;
    __shared__ __attribute__((aligned(16))) _Float16 ring[(SPLIT ? G::NWAVES : 1) * 2 * G::BUF];
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5, l16 = lane & 15, g4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t r0 = (int64_t)blockIdx.x * (SHARE * 32) + (SPLIT ? 0 : wave * 32);
    const int nch = hp / G::HC, c0 = SPLIT ? wave : 0;
    const int w0 = SPLIT ? 0 : wave;  // first of the wavefront's loads of a chunk
    _Float16* const bufs = ring + (SPLIT ? wave * 2 * G::BUF : 0);

    // ---- staging: wavefront load i = wave, wave + NWAVES, ... of the chunk; padding granules load a
    // valid weight granule that nothing reads. Byte offsets of the lane's granules in chunk 0.
    const __amdgpu_buffer_rsrc_t rgu = __builtin_amdgcn_make_buffer_rsrc((void*)wgu, 0, 4 * hp * E, 0x00020000);
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void*)wd, 0, 2 * hp * E, 0x00020000);
    uint32_t voff[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int i = w0 + k * SHARE;
        if (i < G::GLOADS) {
            const int q = min(64 * i + lane, 2 * G::HC * G::GROW - 1);
            const int row = q / G::GROW, cp = min(q % G::GROW, E / 8 - 1);
            voff[k] = (uint32_t)((((row / G::HC) * hp + row % G::HC) * E + 8 * cp) * 2);
        } else {
            const int q = min(64 * (i - G::GLOADS) + lane, 3 * E - 1), e = q / 3, cp = min(q % 3, 1);
            voff[k] = (uint32_t)((e * hp + 8 * cp) * 2);
        }
    }
    auto fetch = [&](int c, int b) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int i = w0 + k * SHARE;
            if (i >= G::LOADS) break;  // uniform over the wavefront
            lds_void* dst = (lds_void*)(bufs + b * G::BUF + 512 * i);
            if (i < G::GLOADS) buffer_to_lds(rgu, dst, voff[k], c * G::HC * E * 2);
            else buffer_to_lds(rd, dst, voff[k], c * G::HC * 2);
        }
    };
    if (c0 < nch) fetch(c0, 0);

    // ---- X fragments (B operands): row tile t holds x[r0 + 16t + l16][32s + 8 g4 + 0..7]
    f16x8 xf[2][G::S];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int64_t row = r0 + 16 * t + l16;
        const bool ok = row < rows;
#pragma unroll
        for (int s = 0; s < G::S; ++s) {
            u32x4 v = u32x4{0u, 0u, 0u, 0u};
            if (ok) v = *reinterpret_cast<const u32x4*>(x + row * xs + 32 * s + 8 * g4);
            xf[t][s] = __builtin_bit_cast(f16x8, v);
        }
    }
    f32x16 yt[G::OT];
#pragma unroll
    for (int t = 0; t < G::OT; ++t) yt[t] = f32x16{};
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr (!SPLIT) __syncthreads();

    const int up_lane = 8 * (l16 * G::GROW + g4);                 // gate row l16 (up rows: HC further)
    const int dn_lane = 8 * (64 * G::GLOADS + 3 * l32 + hh);      // down row l32
    for (int c = c0, cur = 0; c < nch; c += CSTEP, cur ^= 1) {
        if (c + CSTEP < nch) fetch(c + CSTEP, cur ^ 1);
        const _Float16* Wc = bufs + cur * G::BUF;
        // operand reads of the chunk in order: gate and up rows of each k-step, then the down tiles
        auto rd_op = [&](int i) {
            const _Float16* p = i < 2 * G::S ? Wc + up_lane + 8 * ((i & 1) * G::HC * G::GROW + 4 * (i >> 1))
                                             : Wc + dn_lane + 8 * 3 * 32 * (i - 2 * G::S);
            return *reinterpret_cast<const f16x8*>(p);
        };
        f16x8 op[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) op[i] = rd_op(i);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 gt[2], ut[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) gt[t] = ut[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < G::S; ++s) {
            const int i = 2 * s;
            const f16x8 ag = op[i % kAhead], au = op[(i + 1) % kAhead];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                gt[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ag, xf[t][s], gt[t], 0, 0, 0);
                ut[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(au, xf[t][s], ut[t], 0, 0, 0);
            }
            op[i % kAhead] = rd_op(i + kAhead);
            op[(i + 1) % kAhead] = rd_op(i + 1 + kAhead);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the gate: word p of row tile t holds hidden 4 g4 + 2p + {0, 1} of row l16; swapping the tiles'
        // words between 16-lane rows gives lane l the hidden units 8 hh + 0..7 of row l32
        uint32_t w[2][2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int p = 0; p < 2; ++p) w[t][p] = gate_pair(gt[t][2 * p], gt[t][2 * p + 1], ut[t][2 * p], ut[t][2 * p + 1]);
        const auto s0 = __builtin_amdgcn_permlane16_swap(w[0][0], w[1][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(w[0][1], w[1][1], false, false);
        const f16x8 af = __builtin_bit_cast(f16x8, u32x4{s0[0], s1[0], s0[1], s1[1]});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < G::OT; ++t) {
            const int i = 2 * G::S + t;
            const f16x8 ad = op[i % kAhead];
            yt[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ad, af, yt[t], 0, 0, 0);
            if (t + kAhead < G::OT) op[i % kAhead] = rd_op(i + kAhead);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (c + CSTEP < nch) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's loads are in LDS
            if constexpr (!SPLIT) __syncthreads();
        }
    }
    __syncthreads();  // the ring's last reads are done: its memory takes the sums or the rows
    if constexpr (SPLIT) {
        // wavefront w sums tile w over the wavefronts' partials, stages its columns of the 32 rows, and
        // after those of all four takes rows 8w..8w+7
        static_assert(G::OT == G::NWAVES, "a tile per wavefront");
        f32x4* red = reinterpret_cast<f32x4*>(ring);  // [wavefront][tile][j][lane]
        _Float16* ut = ring + G::NWAVES * G::OT * 4 * 64 * 8;
        static_assert((G::NWAVES * G::OT * 4 * 64 * 8 + 32 * (E + 8)) <= G::NWAVES * 2 * G::BUF, "sums and rows fit");
#pragma unroll
        for (int t = 0; t < G::OT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                red[((wave * G::OT + t) * 4 + j) * 64 + lane] =
                    f32x4{yt[t][4 * j], yt[t][4 * j + 1], yt[t][4 * j + 2], yt[t][4 * j + 3]};
        __syncthreads();
        f32x16 sum = f32x16{};
#pragma unroll
        for (int w = 0; w < G::NWAVES; ++w)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 v = red[((w * G::OT + wave) * 4 + j) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[4 * j + i] = sum[4 * j + i] + v[i];
            }
        stage_tile(sum, ut + l32 * (E + 8) + 4 * hh + 32 * wave);
        __syncthreads();
        emit_rows<E, NW, 2>(ut + 8 * wave * (E + 8), r0 + 8 * wave, rows, lane, y, ys, ep);
    } else {
        write_rows<E, NW>(yt, r0, rows, lane, ring + wave * 16 * (E + 8), y, ys, ep);
    }
}

template <int E, int NW = 0>
void launch(const uint16_t* x, int64_t rows, int64_t xs, const uint16_t* wgu, const uint16_t* wd, int hp, uint16_t* y,
            int64_t ys, hipStream_t stream, const ResEpi& ep = ResEpi{}) {
    using G = MlpGeom<E>;
    if constexpr (split_width(E)) {
        if (rows <= (int64_t)kSplitRowsPerCu * device_cus()) {
            hipLaunchKernelGGL((swiglu_mlp_kernel<E, NW, true>), dim3((unsigned)((rows + 31) / 32)), dim3(G::THREADS), 0,
                               stream, x, rows, xs, wgu, wd, hp, y, ys, ep);
            return;
        }
    }
    const int64_t per = G::NWAVES * 32;
    const dim3 grid((unsigned)((rows + per - 1) / per));
    hipLaunchKernelGGL((swiglu_mlp_kernel<E, NW, false>), grid, dim3(G::THREADS), 0, stream, x, rows, xs, wgu, wd, hp, y,
                       ys, ep);
}

}  // namespace

extern "C" int nori_swiglu_mlp(const void* x, int dtype, int64_t rows, int32_t width, int64_t x_row_stride,
                               const void* w_gate_up, const void* w_down, int32_t hidden, void* y, int64_t y_row_stride,
                               void* stream_v) {
    clear_error();
    if (dtype != NORI_F16) return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp: unsupported dtype %s (float16 only)", dtype_name(dtype));
    if (width != 128 && width != 256 && width != 352)
        return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp: no kernel for width %d (128, 256 or 352)", width);
    if (rows < 0 || rows > 0x7fffffffLL || hidden <= 0 || hidden % 32 != 0)
        return fail(NORI_ERR_INVALID, "swiglu_mlp: bad shape (%lld rows, hidden %d: a positive multiple of 32)",
                    (long long)rows, hidden);
    if (x_row_stride < width || y_row_stride < width || x_row_stride % 8 != 0 || y_row_stride % 8 != 0)
        return fail(NORI_ERR_INVALID, "swiglu_mlp: row strides (%lld, %lld) must be multiples of 8 and at least %d",
                    (long long)x_row_stride, (long long)y_row_stride, width);
    if (rows == 0) return NORI_OK;
    if (!x || !w_gate_up || !w_down || !y) return fail(NORI_ERR_INVALID, "swiglu_mlp: null pointer");
    if ((uintptr_t)x % 16 || (uintptr_t)w_gate_up % 16 || (uintptr_t)w_down % 16 || (uintptr_t)y % 16)
        return fail(NORI_ERR_INVALID, "swiglu_mlp: x, the weights and y must be 16-byte aligned");
    if ((int64_t)hidden * width > kMaxWeights) return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp: hidden width %d", hidden);
    hipStream_t stream = (hipStream_t)stream_v;
    auto xp = reinterpret_cast<const uint16_t*>(x);
    auto gp = reinterpret_cast<const uint16_t*>(w_gate_up);
    auto dp = reinterpret_cast<const uint16_t*>(w_down);
    auto yp = reinterpret_cast<uint16_t*>(y);
    switch (width) {
        case 128: launch<128>(xp, rows, x_row_stride, gp, dp, hidden, yp, y_row_stride, stream); break;
        case 256: launch<256>(xp, rows, x_row_stride, gp, dp, hidden, yp, y_row_stride, stream); break;
        default: launch<352>(xp, rows, x_row_stride, gp, dp, hidden, yp, y_row_stride, stream); break;
    }
    return launch_status("swiglu_mlp");
}

extern "C" int nori_swiglu_mlp_residual_rms_norm(const void* x, int dtype, int64_t rows, int32_t width,
                                                 int64_t x_row_stride, const void* w_gate_up, const void* w_down,
                                                 int32_t hidden, float alpha, float* stream_rows,
                                                 int64_t stream_row_stride, int32_t norm_width, float eps, void* y,
                                                 int64_t y_group, int64_t y_group_stride, int64_t y_row_stride,
                                                 void* stream_v) {
    clear_error();
    if (dtype != NORI_F16)
        return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp_residual_rms_norm: unsupported dtype %s (float16 only)", dtype_name(dtype));
    if (!((width == 128 && norm_width == 128) || (width == 256 && (norm_width == 128 || norm_width == 256))))
        return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp_residual_rms_norm: width %d with norm width %d (128/128, 256/128 "
                    "and 256/256 are built)", width, norm_width);
    if (rows < 0 || rows > 0x7fffffffLL || hidden <= 0 || hidden % 32 != 0 || y_group <= 0)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual_rms_norm: bad shape (%lld rows, hidden %d, y_group %lld)",
                    (long long)rows, hidden, (long long)y_group);
    if (x_row_stride < width || x_row_stride % 8 || stream_row_stride < width || stream_row_stride % 4 ||
        y_group_stride % 4 || y_row_stride % 4)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual_rms_norm: row strides must be multiples of 8 (x) or 4");
    if (rows == 0) return NORI_OK;
    if (!x || !w_gate_up || !w_down || !stream_rows || !y)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual_rms_norm: null pointer");
    if ((uintptr_t)x % 16 || (uintptr_t)w_gate_up % 16 || (uintptr_t)w_down % 16 || (uintptr_t)stream_rows % 16 ||
        (uintptr_t)y % 8)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual_rms_norm: x, the weights and the stream must be 16-byte "
                    "aligned, y 8-byte aligned");
    if ((int64_t)hidden * width > kMaxWeights)
        return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp_residual_rms_norm: hidden width %d", hidden);
    const ResEpi ep{stream_rows, stream_row_stride, alpha, eps, y_group, y_group_stride, y_row_stride};
    hipStream_t stream = (hipStream_t)stream_v;
    auto xp = reinterpret_cast<const uint16_t*>(x);
    auto gp = reinterpret_cast<const uint16_t*>(w_gate_up);
    auto dp = reinterpret_cast<const uint16_t*>(w_down);
    auto yp = reinterpret_cast<uint16_t*>(y);
    if (width == 128) launch<128, 128>(xp, rows, x_row_stride, gp, dp, hidden, yp, 0, stream, ep);
    else if (norm_width == 128) launch<256, 128>(xp, rows, x_row_stride, gp, dp, hidden, yp, 0, stream, ep);
    else launch<256, 256>(xp, rows, x_row_stride, gp, dp, hidden, yp, 0, stream, ep);
    return launch_status("swiglu_mlp_residual_rms_norm");
}

extern "C" int nori_swiglu_mlp_residual(const void* x, int64_t rows, int32_t width, int64_t x_row_stride,
                                        const void* w_gate_up, const void* w_down, int32_t hidden, float alpha,
                                        float* stream_rows, int64_t stream_row_stride, void* stream_v) {
    clear_error();
    if (width != 128 && width != 256)
        return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp_residual: width %d is not 128 or 256", width);
    if (rows < 0 || rows > 0x7fffffffLL || hidden <= 0 || hidden % 32 != 0)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual: bad shape (%lld rows, hidden %d)", (long long)rows, hidden);
    if (x_row_stride < width || x_row_stride % 8 || stream_row_stride < width || stream_row_stride % 4)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual: row strides must be multiples of 8 (x) or 4");
    if (rows == 0) return NORI_OK;
    if (!x || !w_gate_up || !w_down || !stream_rows) return fail(NORI_ERR_INVALID, "swiglu_mlp_residual: null pointer");
    if ((uintptr_t)x % 16 || (uintptr_t)w_gate_up % 16 || (uintptr_t)w_down % 16 || (uintptr_t)stream_rows % 16)
        return fail(NORI_ERR_INVALID, "swiglu_mlp_residual: x, the weights and the stream must be 16-byte aligned");
    if ((int64_t)hidden * width > kMaxWeights)
        return fail(NORI_ERR_UNSUPPORTED, "swiglu_mlp_residual: hidden width %d", hidden);
    const ResEpi ep{stream_rows, stream_row_stride, alpha, 0.f, 1, 0, 0};
    hipStream_t stream = (hipStream_t)stream_v;
    auto xp = reinterpret_cast<const uint16_t*>(x);
    auto gp = reinterpret_cast<const uint16_t*>(w_gate_up);
    auto dp = reinterpret_cast<const uint16_t*>(w_down);
    if (width == 128) launch<128, 128>(xp, rows, x_row_stride, gp, dp, hidden, nullptr, 0, stream, ep);
    else launch<256, 256>(xp, rows, x_row_stride, gp, dp, hidden, nullptr, 0, stream, ep);
    return launch_status("swiglu_mlp_residual");
}
