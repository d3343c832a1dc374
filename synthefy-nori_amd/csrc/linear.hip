// Tall-skinny fp16 projection y = x W^T for gfx950: the F.linear of the attention projections
// under fp16 autocast (layer.py projections; reference layer.py:651-683, 1114-1160), for row
// counts in the hundreds of thousands and inner widths of 128 or 256.
//
// Semantics. y[r, c] = f16(sum_k f16(x[r, k]) * f16(W[c, k])) with fp32 sums: what the
// library GEMM computes for fp16 operands under autocast, up to the order of the fp32 sums.
//
// Shapes. These GEMMs are HBM-bound (K = 128 or 256: every output element costs 2 bytes of
// write against 2K FLOP), so the kernel is built for bandwidth: each x row is read from HBM
// once and each output row written once.
//   * A workgroup of 8 wavefronts keeps a chunk of 128 output columns of W in LDS as f16 (zero
//     rows past n) and walks blocks of 256 rows; small calls take blocks of 128, and chunks of 64
//     where K is 256 (the rule stands at launch()).
//   * Each wavefront holds its 32 (16) rows of x as v_mfma_f32_16x16x32_f16 B operands (lane
//     n + 16*(k/8) holds row n, elements 8*(k/8)..+8 of every 32-wide step) and computes the
//     transposed product W x^T tile by tile: each lane ends with four consecutive output
//     columns of one row. 64 columns at a time are staged in the wavefront's LDS slice and
//     stored row by row, 16 bytes per lane and 128 contiguous bytes per row (written straight
//     from the MFMA layout, a store instruction touched 16 rows in 32-byte pieces and the
//     kernel ran 10-20 % slower at N = 128-256).
//   * Rows are addressed on a three-level grid, row r = (o * n_mid + j) * n_inner + i (strides
//     x_outer, x_mid, x_row and y_outer, y_mid, y_row), so strided views (a token subset of
//     each row, a slice of a stacked output, the [table, group, row] transpose of a
//     [table, row, group] cell buffer) are read and written in place.
//   * Each XCD takes a contiguous range of the row blocks (the hardware deals workgroup i to XCD
//     i % 8), and its workgroups come in teams of one per column chunk over the same row blocks:
//     an x block is read from HBM once and served to the other chunks by that XCD's L2.
//   * Measured against workgroups of one row block each, which staged W again for every 256 rows
//     and waited out each x load: 655,360 rows 128 -> 640 286 -> 262 us (1.0 GB, 3.8 TB/s).
//   * The head-norm variant also RMS-norms heads of 64 as their rows leave LDS: 8 lanes hold a head
//     row there, so the mean of squares is three DPP adds. As passes of their own the q/k norms of
//     one cell layer (128 x 512 x 10 cells of 128) read and wrote 280 us' worth of projections, and
//     an attention kernel that normed its rows as it loaded them (2,048 columns x 2 heads, 320 x 256)
//     ran 352 us against 282 us on normed operands.
//
// nori_linear_f16_residual_rms_norm fuses the output projection of an attention sublayer with
// the deep-norm residual update of an fp32 stream and the next sublayer's RMSNorm (no weight)
// into the operand dtype (two_phase.py:198, 209, 220-225, 264, 271-272; layer.py:251-253):
//   u = f16(a W^T),  x = x + f16(u * alpha),  y = f16(x * rsqrt(mean(x^2) + eps)),
// each op rounded as torch rounds it. The output width equals the inner width (128 or 256),
// so a wavefront holds whole rows of u in its accumulators: x is read and written once, y
// written once, and u never reaches memory. The mean of squares is summed in the order of
// the separate residual + norm kernel (nori_residual_add_rms_norm: an fma chain over each
// 4-element chunk, then pairwise over the chunk index bits from the highest), so x and y are
// bit for bit what F.linear-equivalent u through that kernel gives.
//   * Persistent workgroups: W is staged in LDS once (128 x 136 or 256 x 264 f16) and each
//     workgroup walks 128-row blocks, 16 rows per wavefront; a wavefront issues a block's
//     stream loads and the next block's operand loads before the block's MFMAs.
//   * The epilogue moves u through LDS into a row layout (16 lanes on 64 consecutive columns
//     of a row), so the stream is read and written in whole 256-byte row pieces.
#include <algorithm>

#include "nori_common.h"

// the residual update and the norm round every op separately, as torch does
#pragma clang fp contract(off)

namespace {

using namespace nori;

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;

struct LinArgs {
    const _Float16* x; int64_t rows, n_mid, n_inner, x_outer, x_mid, x_row;
    const void* w; int64_t w_row;  // fp16, or fp32 (W32 kernels)
    int n;
    _Float16* y; int64_t y_outer, y_mid, y_row;
    int nchunks, teams;  // column chunks; workgroups per XCD and chunk
    int64_t nblocks;     // row blocks
    // head norm (NORM kernels): columns below norm_cols are heads of 64 with gains [64]
    const void* gain; int gain_dtype; float eps; int norm_cols;
};

struct RowIndex { int64_t o, j, i; };

// row r of the three-level grid, r = (o * n_mid + j) * n_inner + i (32-bit divisions when the
// grid fits them: a 64-bit division is about a hundred instructions)
__device__ __forceinline__ RowIndex split_row(int64_t r, int64_t n_mid, int64_t n_inner, bool narrow) {
    if (narrow) {
        const uint32_t r32 = (uint32_t)r, ni = (uint32_t)n_inner, nm = (uint32_t)n_mid;
        const uint32_t oj = r32 / ni, o = oj / nm;
        return {(int64_t)o, (int64_t)(oj - o * nm), (int64_t)(r32 - oj * ni)};
    }
    const int64_t oj = r / n_inner, i = r - oj * n_inner;
    const int64_t o = oj / n_mid, j = oj - o * n_mid;
    return {o, j, i};
}

__device__ __forceinline__ uint32_t pack_f16_rn(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, f16x2{(_Float16)lo, (_Float16)hi});
}

// 8 consecutive weights from element at, as fp16: fp16 as they lie, or fp32 rounded (the values of a cast)
template <bool W32>
__device__ __forceinline__ uint4 weight8(const void* w, int64_t at) {
    if constexpr (W32) {
        const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(w) + at);
        const f32x4 lo = p[0], hi = p[1];
        return uint4{pack_f16_rn(lo[0], lo[1]), pack_f16_rn(lo[2], lo[3]), pack_f16_rn(hi[0], hi[1]),
                     pack_f16_rn(hi[2], hi[3])};
    }
    return *reinterpret_cast<const uint4*>(reinterpret_cast<const _Float16*>(w) + at);
}

// sum over the 8 lanes of a store row (DPP: lane ^ 1, lane ^ 2, the other quad of 8)
__device__ __forceinline__ float sum8(float v) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xb1, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4e, 0xf, 0xf, false));
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xf, 0xf, false));
    return v;
}

// 8 fp16 values of a 64-wide head row whose other values the neighbouring 7 lanes hold:
// T(T(v * rsqrt(mean(v^2) + eps)) * w), T rounding to fp16 (the per-head RMSNorm pass)
__device__ __forceinline__ uint4 head_norm8(uint4 v, const float (&w)[8], float eps) {
    const uint32_t h[4] = {v.x, v.y, v.z, v.w};
    float x[8], ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        x[e] = f16_to_f32((uint16_t)(h[e >> 1] >> (16 * (e & 1))));
        ss = fmaf(x[e], x[e], ss);
    }
    const float inv = rsqrtf(sum8(ss) / 64.0f + eps);
    uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t lo = f32_to_f16(round_to<NORI_F16>(x[2 * k] * inv) * w[2 * k]);
        r[k] = lo | ((uint32_t)f32_to_f16(round_to<NORI_F16>(x[2 * k + 1] * inv) * w[2 * k + 1]) << 16);
    }
    return uint4{r[0], r[1], r[2], r[3]};
}

// NR 16-row tiles per wavefront. A workgroup keeps its column chunk of W in LDS and walks row
// blocks, loading the next block's x rows before it computes the current one's; the workgroups
// of a chunk's row blocks and those of the other chunks over the same rows share an XCD. W32: the
// weights are fp32 and rounded to fp16 as they are staged, the values of a cast; a caller whose
// parameter is fp32 then launches no cast on each call and keeps none (a layer's cast and the gap around
// it are 4-5 us, a third of a short layer's projection and more).
template <int KS, int NC, int NR, bool NORM, bool W32>
__global__ void __launch_bounds__(kThreads, KS == 4 ? 4 : 2) linear_f16_kernel(const LinArgs a) {
    constexpr int PITCH = 32 * KS + 8;  // f16 per staged W row: +16 bytes spreads the 16-row reads over the banks
    constexpr int GC = 64;              // output columns staged per wavefront between stores
    constexpr int SP = GC + 8;          // f16 per staged output row
    constexpr int WROWS = NR * 16, BROWS = kWaves * WROWS;
    extern __shared__ __attribute__((aligned(16))) _Float16 lds[];
    _Float16* wt = lds;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4;

    const int xcd = blockIdx.x % 8, local = blockIdx.x / 8;
    const int chunk = local % a.nchunks, team = local / a.nchunks;
    const int64_t per = a.nblocks / 8, extra = a.nblocks % 8;
    const int64_t first = xcd * per + (xcd < extra ? xcd : extra), last = first + per + (xcd < extra ? 1 : 0);
    int64_t blk = first + team;
    if (blk >= last) return;  // uniform over the workgroup, before its barrier
    const int c0 = chunk * NC;
    const bool narrow = a.rows <= 0x7fffffffLL;

    auto load_x = [&](int64_t rb, f16x8 (&xf)[NR][KS]) {
#pragma unroll
        for (int nt = 0; nt < NR; ++nt) {
            const int64_t row = rb * BROWS + wave * WROWS + nt * 16 + (lane & 15);
            const RowIndex ri = split_row(row < a.rows ? row : a.rows - 1, a.n_mid, a.n_inner, narrow);
            const _Float16* xrow = a.x + ri.o * a.x_outer + ri.j * a.x_mid + ri.i * a.x_row + 8 * g;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) xf[nt][ks] = *reinterpret_cast<const f16x8*>(xrow + 32 * ks);
        }
    };
    f16x8 xf[NR][KS];
    load_x(blk, xf);

    for (int e = tid; e < NC * KS * 4; e += kThreads) {
        const int r = e / (KS * 4), q = e % (KS * 4);
        uint4 v = {0u, 0u, 0u, 0u};
        if (c0 + r < a.n) v = weight8<W32>(a.w, (int64_t)(c0 + r) * a.w_row + 8 * q);
        *reinterpret_cast<uint4*>(wt + r * PITCH + 8 * q) = v;
    }
    float gain[8];
    if constexpr (NORM) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = 8 * (lane & 7) + e;
            gain[e] = a.gain_dtype == NORI_F32   ? load_elem<NORI_F32>(a.gain, c)
                      : a.gain_dtype == NORI_F16 ? load_elem<NORI_F16>(a.gain, c)
                                                 : load_elem<NORI_BF16>(a.gain, c);
        }
    }
    __syncthreads();

    const _Float16* wa = wt + (lane & 15) * PITCH + 8 * g;
    _Float16* my = lds + NC * PITCH + wave * WROWS * SP;
    const int ncols = min(NC, a.n - c0);
    for (; blk < last; blk += a.teams) {
        // the next block's rows
        f16x8 xn[NR][KS];
        const bool more = blk + a.teams < last;  // uniform over the workgroup
        if (more) load_x(blk + a.teams, xn);
        // lane r < WROWS has row r's place in y; the store passes (8 rows each, 8 lanes a row)
        // take it from there
        const int64_t row0 = blk * BROWS + wave * WROWS;
        const int64_t yrow = row0 + (lane & (WROWS - 1));
        const RowIndex ri = split_row(yrow < a.rows ? yrow : a.rows - 1, a.n_mid, a.n_inner, narrow);
        const int64_t yo = ri.o * a.y_outer + ri.j * a.y_mid + ri.i * a.y_row;
        for (int gc = 0; gc < ncols; gc += GC) {
#pragma unroll
            for (int mm = 0; mm < GC / 16; ++mm) {
                const int m = gc / 16 + mm;
                f32x4 acc[NR];
#pragma unroll
                for (int nt = 0; nt < NR; ++nt) acc[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const f16x8 av = *reinterpret_cast<const f16x8*>(wa + 16 * m * PITCH + 32 * ks);
#pragma unroll
                    for (int nt = 0; nt < NR; ++nt) acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, xf[nt][ks], acc[nt], 0, 0, 0);
                }
#pragma unroll
                for (int nt = 0; nt < NR; ++nt)
                    *reinterpret_cast<uint2*>(my + (nt * 16 + (lane & 15)) * SP + 16 * mm + 4 * g) =
                        uint2{pack_f16_rn(acc[nt][0], acc[nt][1]), pack_f16_rn(acc[nt][2], acc[nt][3])};
            }
            // the wavefront's rows x 64 columns, row by row: 16 bytes per lane, 128 per row
            const int col = c0 + gc + 8 * (lane & 7);
#pragma unroll
            for (int p = 0; p < 2 * NR; ++p) {
                const int rr = 8 * p + (lane >> 3);
                uint4 v = *reinterpret_cast<const uint4*>(my + rr * SP + 8 * (lane & 7));
                if constexpr (NORM) {
                    if (c0 + gc < a.norm_cols) v = head_norm8(v, gain, a.eps);
                }
                const int64_t at = __shfl(yo, rr) + col;
                if (row0 + rr < a.rows) {
                    if (col + 8 <= a.n) *reinterpret_cast<uint4*>(a.y + at) = v;
                    else if (col + 4 <= a.n) *reinterpret_cast<uint2*>(a.y + at) = uint2{v.x, v.y};
                }
            }
        }
        if (!more) break;
#pragma unroll
        for (int nt = 0; nt < NR; ++nt)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) xf[nt][ks] = xn[nt][ks];
    }
}

template <int KS, int NC, int NR, bool NORM, bool W32>
int launch_tiles(LinArgs a, int cus, hipStream_t stream) {
    constexpr int BROWS = kWaves * NR * 16;
    constexpr size_t lds = ((size_t)NC * (32 * KS + 8) + (size_t)BROWS * 72) * sizeof(_Float16);
    static_assert(lds <= 160 * 1024, "a chunk of W and the staged rows fit one workgroup's LDS");
    if (hipFuncSetAttribute((const void*)linear_f16_kernel<KS, NC, NR, NORM, W32>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
        return fail(NORI_ERR_RUNTIME, "linear_f16: cannot reserve %zu bytes of LDS", lds);
    a.nchunks = (a.n + NC - 1) / NC;
    a.nblocks = (a.rows + BROWS - 1) / BROWS;
    // resident workgroups (LDS-bound, 16 wavefronts per CU at most), dealt to the XCDs in whole
    // teams: one workgroup per column chunk over the same row blocks
    const int64_t slots = (int64_t)cus * std::max<int64_t>(1, std::min<int64_t>(160 * 1024 / lds, 2)) / 8;
    const int64_t per_xcd = (a.nblocks + 7) / 8, most = std::max<int64_t>(1, std::min<int64_t>(slots / a.nchunks, per_xcd));
    const int64_t rounds = (per_xcd + most - 1) / most;
    a.teams = (int)((per_xcd + rounds - 1) / rounds);  // no more than share the blocks evenly
    const int64_t grid = 8 * (int64_t)a.teams * a.nchunks;
    if (grid > 0x7fffffffLL) return fail(NORI_ERR_UNSUPPORTED, "linear_f16: %d columns exceed one launch", a.n);
    hipLaunchKernelGGL((linear_f16_kernel<KS, NC, NR, NORM, W32>), dim3((unsigned)grid), dim3(kThreads), lds, stream, a);
    return launch_status("linear_f16");
}

// The tile of a call. Workgroups of 256 rows x 128 columns from 0.4 of them a CU: below, twice as many of
// 128 rows are ahead (4,096 rows, K 128: N 768, 96 of them, 7.3 -> 6.3 us), above, W staged twice as often
// costs more (8,192 x 768, 192 of them: 8.5 us against 8.9 in 128 rows; 33,000 x 128, 129: 7.9 against 8.2).
// At K 256 a workgroup stages 64 KB of W, so chunks of 64 are ahead while an XCD's share of the blocks (it
// takes whole ones) leaves no more than one such workgroup a CU: 64 to 4,096 rows, N 256 6.9 - 8.3 -> 4.9 - 6.1
// us; 6,600 to 8,192 rows, N 512 11.4 -> 9.1; past it (2,304 rows, N 1536) they take 15.6 us against 11.5.
// Teams share the blocks evenly: 65,536 x 640, K 128: 27.1 -> 26.7 us, N 384 20.1 -> 19.8; and the last block of
// a workgroup loads no rows after it, which cost calls of about a block each 5 to 10 % (20,000 x 640:
// 13.9 -> 12.7 us).
template <int KS, bool NORM, bool W32>
int launch(LinArgs a, hipStream_t stream) {
    const int cus = device_cus();
    const int64_t chunks = (a.n + 127) / 128, blocks = (a.rows + 255) / 256;
    const bool tall = 5 * blocks * chunks >= 2 * cus;
    if constexpr (KS == 8) {
        auto fits = [&](int64_t nblocks) { return (nblocks + 7) / 8 * 8 * 2 * chunks <= cus; };
        if (tall && fits(blocks)) return launch_tiles<KS, 64, 2, NORM, W32>(a, cus, stream);
        if (!tall && fits((a.rows + 127) / 128)) return launch_tiles<KS, 64, 1, NORM, W32>(a, cus, stream);
    }
    if (tall) return launch_tiles<KS, 128, 2, NORM, W32>(a, cus, stream);
    return launch_tiles<KS, 128, 1, NORM, W32>(a, cus, stream);
}

// ---------------------------------------------------------------- projection + residual + norm

struct ResArgs {
    const _Float16* a; int64_t rows, n_mid, n_inner, a_outer, a_mid, a_row;
    const void* w; int64_t w_row;  // fp16, or fp32 (W32 kernels, rounded as they are staged)
    const float* x; int64_t x_outer, x_mid, x_row;
    float* xo;    // the updated stream, at x's strides (may be x)
    _Float16* y;  // null: no norm
    int64_t y_outer, y_mid, y_row;
    float alpha, eps;
    int64_t nblocks;
};

// K = N = 32 KS; one 16-row tile per wavefront and block; W in dynamic LDS (K rows of K + 8
// f16), then each wavefront's 16 x 72 f16 slice for u. Per block a wavefront issues its
// stream loads and the next block's operand loads before its MFMAs, so both are in flight
// while it computes. The epilogue runs row by row, 64 columns at a time: u of four column
// tiles goes through the wavefront's LDS slice, and 16 lanes take a row's 64 columns (4
// consecutive elements each), so stream rows move 256 contiguous bytes per row and
// instruction and output rows 128. Lane l handles tile rows 4 p + l / 16 (p = 0..3) at
// columns 64 q + 4 (l % 16) for every chunk q: its chunk index in the row is 16 q + l % 16.
template <int KS, int WAVES, bool W32>
__global__ void __launch_bounds__(WAVES * 64, KS == 4 ? 4 : 2) linear_residual_norm_kernel(const ResArgs a) {
    constexpr int K = 32 * KS, PITCH = K + 8;
    constexpr int kBlockRows = WAVES * 16;
    constexpr int NCH = K / 64, UP = 64 + 8;  // 64-column chunks; pitch of a staged u row
    extern __shared__ __attribute__((aligned(16))) _Float16 wt[];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4;
    const int c4 = 4 * (lane & 15);
    const bool narrow = a.rows <= 0x7fffffffLL;

    for (int e = tid; e < K * (K / 8); e += WAVES * 64) {
        const int r = e / (K / 8), q = e % (K / 8);
        *reinterpret_cast<uint4*>(wt + r * PITCH + 8 * q) = weight8<W32>(a.w, (int64_t)r * a.w_row + 8 * q);
    }
    const _Float16* wa = wt + (lane & 15) * PITCH + 8 * g;
    _Float16* ut = wt + K * PITCH + wave * 16 * UP;

    auto operand_row = [&](int64_t blk) {
        const int64_t row = blk * kBlockRows + wave * 16 + (lane & 15);
        const RowIndex ri = split_row(row < a.rows ? row : a.rows - 1, a.n_mid, a.n_inner, narrow);
        return a.a + ri.o * a.a_outer + ri.j * a.a_mid + ri.i * a.a_row + 8 * g;
    };
    f16x8 xf[KS];
    int64_t blk = blockIdx.x;
    {
        const _Float16* ar = operand_row(blk);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) xf[ks] = *reinterpret_cast<const f16x8*>(ar + 32 * ks);
    }
    __syncthreads();

    for (; blk < a.nblocks; blk += gridDim.x) {
        // lane r < 16 computes tile row r's stream and output offsets; the passes take them
        // from there
        const int64_t row0 = blk * kBlockRows + wave * 16;
        const RowIndex ri = split_row(row0 + (lane & 15) < a.rows ? row0 + (lane & 15) : a.rows - 1, a.n_mid,
                                      a.n_inner, narrow);
        const int64_t xo = ri.o * a.x_outer + ri.j * a.x_mid + ri.i * a.x_row;
        const int64_t yo = ri.o * a.y_outer + ri.j * a.y_mid + ri.i * a.y_row;
        f32x4 v[4][NCH];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int rr = 4 * p + (lane >> 4);
            const int64_t xop = __shfl(xo, rr) + c4;
#pragma unroll
            for (int q = 0; q < NCH; ++q)
                v[p][q] = row0 + rr < a.rows ? *reinterpret_cast<const f32x4*>(a.x + xop + 64 * q)
                                             : f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // the next block's operand rows (the last block re-reads its own: in bounds, unused)
        f16x8 xn[KS];
        {
            const int64_t nb = blk + gridDim.x;
            const _Float16* ar = operand_row(nb < a.nblocks ? nb : blk);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) xn[ks] = *reinterpret_cast<const f16x8*>(ar + 32 * ks);
        }
        float part[4][NCH];
#pragma unroll
        for (int q = 0; q < NCH; ++q) {
            f32x4 acc[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const f16x8 av = *reinterpret_cast<const f16x8*>(wa + 16 * (4 * q + m) * PITCH + 32 * ks);
                    acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, xf[ks], acc[m], 0, 0, 0);
                }
            }
            // u = fp16(acc): row lane & 15, columns 16 m + 4 g of this chunk
#pragma unroll
            for (int m = 0; m < 4; ++m)
                *reinterpret_cast<uint2*>(ut + (lane & 15) * UP + 16 * m + 4 * g) =
                    uint2{pack_f16_rn(acc[m][0], acc[m][1]), pack_f16_rn(acc[m][2], acc[m][3])};
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int rr = 4 * p + (lane >> 4);
                const uint2 uw = *reinterpret_cast<const uint2*>(ut + rr * UP + c4);
                const uint32_t hw[2] = {uw.x, uw.y};
                float pp = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float u = f16_to_f32((uint16_t)(hw[e >> 1] >> (16 * (e & 1))));
                    v[p][q][e] = v[p][q][e] + round_to<NORI_F16>(u * a.alpha);
                    pp = fmaf(v[p][q][e], v[p][q][e], pp);
                }
                part[p][q] = pp;
                const int64_t xop = __shfl(xo, rr) + c4 + 64 * q;
                if (row0 + rr < a.rows) *reinterpret_cast<f32x4*>(a.xo + xop) = v[p][q];
            }
        }
        if (a.y) {  // uniform over the launch
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            // pairs over the chunk index bits from the highest: q's in the lane, then l % 16's
#pragma unroll
            for (int st = NCH / 2; st >= 1; st >>= 1) {
#pragma unroll
                for (int q = 0; q < st; ++q) part[p][q] = part[p][q] + part[p][q + st];
            }
            float tot = part[p][0];
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) tot = tot + __shfl_xor(tot, off);
            const float inv = rsqrtf(tot / (float)K + a.eps);
            const int rr = 4 * p + (lane >> 4);
            const int64_t yop = __shfl(yo, rr) + c4;
            if (row0 + rr < a.rows) {
#pragma unroll
                for (int q = 0; q < NCH; ++q) {
                    uint16_t h[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) h[e] = f32_to_f16(v[p][q][e] * inv);
                    *reinterpret_cast<uint2*>(a.y + yop + 64 * q) =
                        uint2{h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16)};
                }
            }
        }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) xf[ks] = xn[ks];
    }
}

template <int KS, int WAVES, bool W32>
int launch_residual(ResArgs a, hipStream_t stream) {
    constexpr int K = 32 * KS;
    constexpr size_t lds = ((size_t)K * (K + 8) + (size_t)WAVES * 16 * 72) * sizeof(_Float16);
    constexpr int kBlockRows = WAVES * 16;
    static_assert(lds <= 160 * 1024, "W must fit one workgroup's LDS");
    if (hipFuncSetAttribute((const void*)linear_residual_norm_kernel<KS, WAVES, W32>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return fail(NORI_ERR_RUNTIME, "linear_f16_residual_rms_norm: cannot reserve %zu bytes of LDS", lds);
    a.nblocks = (a.rows + kBlockRows - 1) / kBlockRows;
    // resident workgroups per CU: LDS-bound, and at most 16 wavefronts per CU
    const int per_cu = std::max(1, (int)std::min<size_t>(160 * 1024 / lds, 16 / WAVES));
    const int64_t grid = std::min<int64_t>(a.nblocks, (int64_t)device_cus() * per_cu);
    hipLaunchKernelGGL((linear_residual_norm_kernel<KS, WAVES, W32>), dim3((unsigned)grid), dim3(WAVES * 64), lds,
                       stream, a);
    return launch_status("linear_f16_residual_rms_norm");
}

}  // namespace

namespace {

int run_linear(const void* x, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k, int64_t x_outer_stride,
               int64_t x_mid_stride, int64_t x_row_stride, const void* weight, int64_t w_row_stride, int32_t n, void* y,
               int64_t y_outer_stride, int64_t y_mid_stride, int64_t y_row_stride, const void* gain, int gain_dtype,
               float eps, int32_t norm_cols, void* stream, bool w32 = false) {
    clear_error();
    if (n_outer < 0 || n_mid < 0 || n_inner < 0 || k <= 0 || n <= 0)
        return fail(NORI_ERR_INVALID, "linear_f16: bad shape n_outer=%lld n_mid=%lld n_inner=%lld k=%d n=%d",
                    (long long)n_outer, (long long)n_mid, (long long)n_inner, k, n);
    if (k != 128 && k != 256) return fail(NORI_ERR_UNSUPPORTED, "linear_f16: inner width %d is not 128 or 256", k);
    if (n % 4) return fail(NORI_ERR_UNSUPPORTED, "linear_f16: output width %d is not a multiple of 4", n);
    if (n_outer == 0 || n_mid == 0 || n_inner == 0) return NORI_OK;
    if (n_inner > INT64_MAX / n_mid || n_mid * n_inner > INT64_MAX / n_outer)
        return fail(NORI_ERR_INVALID, "linear_f16: %lld x %lld x %lld rows overflow", (long long)n_outer,
                    (long long)n_mid, (long long)n_inner);
    if (!x || !weight || !y) return fail(NORI_ERR_INVALID, "linear_f16: null pointer");
    // 16-byte x and W row chunks, 8-byte output pieces
    if ((uintptr_t)x % 16 || x_row_stride % 8 || x_mid_stride % 8 || x_outer_stride % 8 || (uintptr_t)weight % 16 ||
        w_row_stride % (w32 ? 4 : 8) || w_row_stride < k || (uintptr_t)y % 8 || y_row_stride % 4 || y_mid_stride % 4 ||
        y_outer_stride % 4)
        return fail(NORI_ERR_UNSUPPORTED,
                    "linear_f16: x and weight rows must be 16-byte aligned, output rows 8-byte aligned");
    LinArgs a;
    a.x = reinterpret_cast<const _Float16*>(x);
    a.rows = n_outer * n_mid * n_inner;
    a.n_mid = n_mid;
    a.n_inner = n_inner;
    a.x_outer = x_outer_stride;
    a.x_mid = x_mid_stride;
    a.x_row = x_row_stride;
    a.w = weight;
    a.w_row = w_row_stride;
    a.n = n;
    a.y = reinterpret_cast<_Float16*>(y);
    a.y_outer = y_outer_stride;
    a.y_mid = y_mid_stride;
    a.y_row = y_row_stride;
    a.gain = gain;
    a.gain_dtype = gain_dtype;
    a.eps = eps;
    a.norm_cols = norm_cols;
    hipStream_t s = (hipStream_t)stream;
    if (norm_cols > 0) return k == 128 ? launch<4, true, false>(a, s) : launch<8, true, false>(a, s);
    if (w32) return k == 128 ? launch<4, false, true>(a, s) : launch<8, false, true>(a, s);
    return k == 128 ? launch<4, false, false>(a, s) : launch<8, false, false>(a, s);
}

}  // namespace

extern "C" int nori_linear_f16(const void* x, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k,
                               int64_t x_outer_stride, int64_t x_mid_stride, int64_t x_row_stride, const void* weight,
                               int64_t w_row_stride, int32_t n, void* y, int64_t y_outer_stride, int64_t y_mid_stride,
                               int64_t y_row_stride, void* stream) {
    return run_linear(x, n_outer, n_mid, n_inner, k, x_outer_stride, x_mid_stride, x_row_stride, weight, w_row_stride, n,
                      y, y_outer_stride, y_mid_stride, y_row_stride, nullptr, NORI_F32, 0.f, 0, stream);
}

extern "C" int nori_linear_f16_w32(const void* x, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k,
                                   int64_t x_outer_stride, int64_t x_mid_stride, int64_t x_row_stride,
                                   const float* weight, int64_t w_row_stride, int32_t n, void* y, int64_t y_outer_stride,
                                   int64_t y_mid_stride, int64_t y_row_stride, void* stream) {
    return run_linear(x, n_outer, n_mid, n_inner, k, x_outer_stride, x_mid_stride, x_row_stride, weight, w_row_stride, n,
                      y, y_outer_stride, y_mid_stride, y_row_stride, nullptr, NORI_F32, 0.f, 0, stream, true);
}

extern "C" int nori_linear_f16_head_norm(const void* x, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k,
                                         int64_t x_outer_stride, int64_t x_mid_stride, int64_t x_row_stride,
                                         const void* weight, int64_t w_row_stride, int32_t n, void* y,
                                         int64_t y_outer_stride, int64_t y_mid_stride, int64_t y_row_stride,
                                         const void* gain, int gain_dtype, float eps, int32_t norm_cols, void* stream) {
    if (norm_cols <= 0 || norm_cols > n || norm_cols % 64) {
        clear_error();
        return fail(NORI_ERR_INVALID, "linear_f16_head_norm: %d columns of %d are not whole heads of 64", norm_cols, n);
    }
    if (!gain || (gain_dtype != NORI_F32 && gain_dtype != NORI_F16 && gain_dtype != NORI_BF16)) {
        clear_error();
        return fail(NORI_ERR_INVALID, "linear_f16_head_norm: gains must be float32, float16 or bfloat16");
    }
    return run_linear(x, n_outer, n_mid, n_inner, k, x_outer_stride, x_mid_stride, x_row_stride, weight, w_row_stride, n,
                      y, y_outer_stride, y_mid_stride, y_row_stride, gain, gain_dtype, eps, norm_cols, stream);
}


namespace {

int run_residual(const void* a, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k, int64_t a_outer_stride,
                 int64_t a_mid_stride, int64_t a_row_stride, const void* weight, int64_t w_row_stride, bool w32, float alpha,
                 const float* x, int64_t x_outer_stride, int64_t x_mid_stride, int64_t x_row_stride, float* x_out,
                 float eps, void* y, int64_t y_outer_stride, int64_t y_mid_stride, int64_t y_row_stride, void* stream) {
    clear_error();
    if (n_outer < 0 || n_mid < 0 || n_inner < 0 || k <= 0)
        return fail(NORI_ERR_INVALID, "linear_f16_residual_rms_norm: bad shape n_outer=%lld n_mid=%lld n_inner=%lld k=%d",
                    (long long)n_outer, (long long)n_mid, (long long)n_inner, k);
    if (k != 128 && k != 256)
        return fail(NORI_ERR_UNSUPPORTED, "linear_f16_residual_rms_norm: width %d is not 128 or 256", k);
    if (n_outer == 0 || n_mid == 0 || n_inner == 0) return NORI_OK;
    if (n_inner > INT64_MAX / n_mid || n_mid * n_inner > INT64_MAX / n_outer)
        return fail(NORI_ERR_INVALID, "linear_f16_residual_rms_norm: %lld x %lld x %lld rows overflow",
                    (long long)n_outer, (long long)n_mid, (long long)n_inner);
    if (!a || !weight || !x || !x_out) return fail(NORI_ERR_INVALID, "linear_f16_residual_rms_norm: null pointer");
    // 16-byte operand and weight chunks, 16-byte pieces of x, 8-byte pieces of y
    if ((uintptr_t)a % 16 || a_row_stride % 8 || a_mid_stride % 8 || a_outer_stride % 8 || (uintptr_t)weight % 16 ||
        w_row_stride % (w32 ? 4 : 8) || w_row_stride < k || (uintptr_t)x % 16 || (uintptr_t)x_out % 16 || x_row_stride % 4 || x_mid_stride % 4 ||
        x_outer_stride % 4 || (uintptr_t)y % 8 || y_row_stride % 4 || y_mid_stride % 4 || y_outer_stride % 4)
        return fail(NORI_ERR_UNSUPPORTED, "linear_f16_residual_rms_norm: operand and weight rows must be 16-byte "
                    "aligned, stream rows 16-byte aligned, output rows 8-byte aligned");
    ResArgs r;
    r.a = reinterpret_cast<const _Float16*>(a);
    r.rows = n_outer * n_mid * n_inner;
    r.n_mid = n_mid;
    r.n_inner = n_inner;
    r.a_outer = a_outer_stride;
    r.a_mid = a_mid_stride;
    r.a_row = a_row_stride;
    r.w = weight;
    r.w_row = w_row_stride;
    r.x = x;
    r.xo = x_out;
    r.x_outer = x_outer_stride;
    r.x_mid = x_mid_stride;
    r.x_row = x_row_stride;
    r.y = reinterpret_cast<_Float16*>(y);
    r.y_outer = y_outer_stride;
    r.y_mid = y_mid_stride;
    r.y_row = y_row_stride;
    r.alpha = alpha;
    r.eps = eps;
    hipStream_t s = (hipStream_t)stream;
    if (w32) return k == 128 ? launch_residual<4, 8, true>(r, s) : launch_residual<8, 8, true>(r, s);
    return k == 128 ? launch_residual<4, 8, false>(r, s) : launch_residual<8, 8, false>(r, s);
}

}  // namespace

extern "C" int nori_linear_f16_residual_rms_norm(const void* a, int64_t n_outer, int64_t n_mid, int64_t n_inner,
                                                 int32_t k, int64_t a_outer_stride, int64_t a_mid_stride,
                                                 int64_t a_row_stride, const void* weight, int64_t w_row_stride,
                                                 float alpha, float* x, int64_t x_outer_stride, int64_t x_mid_stride,
                                                 int64_t x_row_stride, float eps, void* y, int64_t y_outer_stride,
                                                 int64_t y_mid_stride, int64_t y_row_stride, void* stream) {
    if (!y && n_outer > 0 && n_mid > 0 && n_inner > 0 && (k == 128 || k == 256)) {
        clear_error();
        return fail(NORI_ERR_INVALID, "linear_f16_residual_rms_norm: null pointer");
    }
    return run_residual(a, n_outer, n_mid, n_inner, k, a_outer_stride, a_mid_stride, a_row_stride, weight, w_row_stride,
                        false, alpha, x, x_outer_stride, x_mid_stride, x_row_stride, x, eps, y, y_outer_stride, y_mid_stride,
                        y_row_stride, stream);
}

extern "C" int nori_linear_f16_residual(const void* a, int64_t n_outer, int64_t n_mid, int64_t n_inner, int32_t k,
                                        int64_t a_outer_stride, int64_t a_mid_stride, int64_t a_row_stride,
                                        const void* weight, int64_t w_row_stride, int w_dtype, float alpha, const float* x,
                                        int64_t x_outer_stride, int64_t x_mid_stride, int64_t x_row_stride, float* x_out,
                                        float eps, void* y, int64_t y_outer_stride, int64_t y_mid_stride,
                                        int64_t y_row_stride, void* stream) {
    if (w_dtype != NORI_F16 && w_dtype != NORI_F32) {
        clear_error();
        return fail(NORI_ERR_UNSUPPORTED, "linear_f16_residual: %s weights", dtype_name(w_dtype));
    }
    return run_residual(a, n_outer, n_mid, n_inner, k, a_outer_stride, a_mid_stride, a_row_stride, weight, w_row_stride,
                        w_dtype == NORI_F32, alpha, x, x_outer_stride, x_mid_stride, x_row_stride, x_out, eps, y, y_outer_stride, y_mid_stride,
                        y_row_stride, stream);
}
