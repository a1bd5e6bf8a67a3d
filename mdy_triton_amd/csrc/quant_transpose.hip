// Training-time quantizer: one pass over a bf16 matrix produces
//   (1) the row-wise 1x128 quantization y[PM,PK] with scales s[kb*s_kb_stride + m]      (as the forward quantizer), and
//   (2) the quantized TRANSPOSE y_t[PK,PM], scaled either per 128x1 column group (t_mode 0) or per
//       128x128 block (t_mode 1),
// in the DeepLinear dialect (MODE 1: scale = (min(amax,1e4) + 1e-8) / 448, saturating cast) or, per column group only,
// in the official dialect (MODE 0: scale = amax / 448, no clamp, no eps: act_quant_block(x) and
// act_quant_block(x, transpose=True) of /root/reference/triton_kernels/deepseekv3/fp8_kernel.py:14-87 in one pass).
//
// Restates _quant_grad_output_kernel (/root/reference/triton_kernels/dpsk_fp8linear/fp8.py:13-44;
// t_mode 0: second half at :40-44 quantizes along axis 0 and stores ST[off_n + pid_m*PN]) and the
// training branch of _quant_input_kernel (fp8.py:115-120; t_mode 1: one scale per 128x128 tile, the
// max of the rows' clamped+eps maxima, stored ST[pid_n*num_programs(0) + pid_m]).
//
// One block of 512 threads per 128x128 tile, the tile stays in registers (read once).  Thread t
// owns columns (t%16)*8..+7 of RPT = 4 consecutive rows: row maxima by DPP inside 16-lane rows, column maxima by a per-thread
// max over its rows, row swaps inside the wave and an LDS reduction over the waves.
// What bounds it: memory at the asymptote (6.4 TB/s between 8192 and 16384 rows of 4096), and for the 2 to 8 tiles per CU of an
// ordinary layer the length of one tile's chain, load - maxima - barrier - scales - barrier - quotients - store.  So the loads of
// all rows are in flight together, a row's two divisions are done by one lane instead of 16, and no LDS permutation lies on
// the way: 8192x4096 31.6 -> 27.4 us (4.9 TB/s), 4096x7168 26.6 -> 24.6 us, 4096x2048 11.4 -> 9.2 us, 700x1536 6.1 -> 5.1 us.  Quotients
// use the reciprocal + 2-FMA form (bit-identical to IEEE division for every finite amax in this
// dialect); groups whose amax exceeds the 1e4 clamp or is not finite divide plainly and clamp.
// Because a thread's rows are consecutive, its 4 bytes of one column are 4 consecutive bytes of a row of the
// transposed tile: the transpose goes through a padded LDS tile with 4-byte writes and 8-byte reads, and both
// outputs are written row-contiguously.
#include "swiglu.h"

namespace mdy {

constexpr int RPT = 4;      // consecutive rows per thread (8 rows and 256 threads per tile: 0.5-4 % slower from 4096x2048 to 16384x8192)

// v of lane i of every 16-lane row, for i = 0 .. RPT-1
__device__ __forceinline__ void bcast_rows(float v, float (&out)[RPT]) {
    out[0] = row16_bcast<0>(v);
    out[1] = row16_bcast<1>(v);
    out[2] = row16_bcast<2>(v);
    out[3] = row16_bcast<3>(v);
}

// x / s.  FAST (the group's amax lies where the reciprocal form is proven bit-identical to IEEE division and,
// in the DeepLinear dialect, amax <= 1e4, so |x/s| <= 448 needs no clamp) uses the reciprocal form; otherwise an
// IEEE division, saturated at +-448 in the DeepLinear dialect (NaN kept).
template <int MODE, bool FAST>
__device__ __forceinline__ float qt_quot(float x, float s, float r) {
    if (FAST) return fast_quotient(x, s, r);
    return sat_for_mode<MODE>(x / s);
}

// Scale layouts: row scale of row m, K group kb at s[kb * s_kb_stride + m * s_m_stride]; column-group scale of
// column k, row group a at s_t[a * st_a_stride + k * st_k_stride] (TMODE 0) / block scale at s_t[kb * (PM/128) + a]
// (TMODE 1).  y may be null (MODE 0 callers that only want the transposed copy): the row-wise outputs are skipped.
// XT: input type (0 bf16, 1 fp16, 2 fp32); the reciprocal quotient is proven for bf16 inputs only, other types divide.
// CSUM (with TMODE 0): also the fp32 sums of the tile's columns, to col_sum[row tile * PK + column]: an output gradient's column
// sums are the bias gradient, and here they cost 8 adds per 16 bytes loaded instead of a pass over the matrix.
// y_t_tile: the transposed copy's element (column 0, first row of the tile), rows of yt_stride bytes.  s_t_tile (TMODE 0): the scales of
// the tile's row group, column k at s_t_tile[k * st_k_stride].
constexpr int NRG = 128 / RPT;        // row groups of RPT consecutive rows; 16 threads (8 columns each) per group
constexpr int QT_WAVES = NRG / 4;
template <bool CSUM>
struct QtLds {
    __attribute__((aligned(16))) float col_part[QT_WAVES][128];  // per wave (4 row groups) partial column maxima
    __attribute__((aligned(16))) float sum_part[CSUM ? QT_WAVES : 1][128];       // the same for the column sums
    __attribute__((aligned(16))) float col_amax[128];
    __attribute__((aligned(16))) float col_sc[128];   // per column: scale of the transposed copy ...
    __attribute__((aligned(16))) float col_rc[128];   // ... and its reciprocal, computed once per column
    float row_sc[128];         // the tile's 128 row scales, written out as one contiguous run
    float blk_part[QT_WAVES];
    // [k][m], transposed; the 16-byte pieces of a row are exchanged by tile_at so that the 64 lanes of a write meet 64 banks
    __attribute__((aligned(16))) uint8_t tile[128][128 + 8];
    __device__ __forceinline__ uint8_t* tile_at(int k, int m) { return &tile[k][m ^ (((k >> 5) & 3) << 4)]; }
};

// f: the thread's RPT rows x 8 columns of the tile.  A caller with several tiles puts a barrier between them.
template <int MODE, int TMODE, int XT, bool CSUM>
__device__ __forceinline__ void quant_transpose_regs(QtLds<CSUM>& lds, const float (&f)[RPT][8], int bm, int bk, uint8_t* __restrict__ y,
                                                     float* __restrict__ s, uint8_t* __restrict__ y_t_tile, int yt_stride,
                                                     float* __restrict__ s_t_tile, int PM, int PK, int64_t s_kb_stride, int64_t s_m_stride,
                                                     int64_t st_k_stride, float* __restrict__ col_sum) {
    constexpr int WAVES = QT_WAVES;
    auto& col_part = lds.col_part;
    auto& sum_part = lds.sum_part;
    auto &col_amax = lds.col_amax, &col_sc = lds.col_sc, &col_rc = lds.col_rc, &row_sc = lds.row_sc;
    auto& blk_part = lds.blk_part;
    const int t = threadIdx.x;
    const int lane = t & 63, wave = t >> 6;
    const int cl = (t & 15) * 8;          // first local column of this thread
    const int rg = t >> 4;                // row group 0..NRG-1
    const int c0 = bk * 128 + cl;

    float rmax[RPT];
    float cmax[8], csum[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) cmax[j] = csum[j] = 0.0f;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            m = fmaxf(fmaxf(fabsf(f[i][2 * j]), fabsf(f[i][2 * j + 1])), m);
            cmax[2 * j] = fmaxf(cmax[2 * j], fabsf(f[i][2 * j]));
            cmax[2 * j + 1] = fmaxf(cmax[2 * j + 1], fabsf(f[i][2 * j + 1]));
        }
        if (CSUM) {
#pragma unroll
            for (int j = 0; j < 8; ++j) csum[j] += f[i][j];
        }
        rmax[i] = row16_max(m);
    }

    // ---- (1) row-wise quantization straight from registers.  The 16 lanes of a row hold the same maximum: lane i of them computes
    // the scale and the reciprocal of row i (two divisions per lane instead of two per row) and the others take them from it.
    if (y != nullptr) {
        float am = rmax[0];
#pragma unroll
        for (int i = 1; i < RPT; ++i) am = (t & 15) == i ? rmax[i] : am;
        const float lane_sc = group_scale<MODE>(am), lane_rc = 1.0f / lane_sc;
        if ((t & 15) < RPT) row_sc[rg * RPT + (t & 15)] = lane_sc;
        float rsc[RPT], rrc[RPT];
        bcast_rows(lane_sc, rsc);
        bcast_rows(lane_rc, rrc);
        bool rfast = XT == 0;
#pragma unroll
        for (int i = 0; i < RPT; ++i) rfast = rfast && group_is_fast<MODE>(rmax[i]);
        uint8_t* yp = y + (int64_t)(bm * 128 + rg * RPT) * PK + c0;      // rows < PM
#pragma unroll
        for (int i = 0; i < RPT; ++i)
            store_nt8(yp + (int64_t)i * PK, quantize8_scaled<MODE>(f[i], rsc[i], rrc[i], rfast));      // (slow rows divide, the same bytes)
    }

    // ---- (2) scales of the transposed copy
    float tamax[8];   // amax that scales this thread's 8 columns in the transposed copy
    float tsc[8], tr[8];
    if (TMODE == 0) {
        // the 4 row groups of a wave hold the same columns in lanes 16 apart: fold them before going to LDS
        const int fc = cl + fold_base(lane >> 4);
        *reinterpret_cast<float2*>(&col_part[wave][fc]) = fold_rows8(cmax, [](float a, float b) { return fmaxf(a, b); });
        if (CSUM) *reinterpret_cast<float2*>(&sum_part[CSUM ? wave : 0][fc]) = fold_rows8(csum, [](float a, float b) { return a + b; });
        __syncthreads();
        if (t < 128) {
            float m = 0.0f;
#pragma unroll
            for (int g = 0; g < WAVES; ++g) m = fmaxf(m, col_part[g][t]);
            const float sc = group_scale<MODE>(m);
            col_amax[t] = m;
            col_sc[t] = sc;
            col_rc[t] = 1.0f / sc;
            s_t_tile[(int64_t)(bk * 128 + t) * st_k_stride] = sc;
            if (y != nullptr) s[(int64_t)bk * s_kb_stride + (int64_t)(bm * 128 + t) * s_m_stride] = row_sc[t];
            if (CSUM) {
                float v = 0.0f;
#pragma unroll
                for (int g = 0; g < WAVES; ++g) v += sum_part[CSUM ? g : 0][t];
                col_sum[(int64_t)bm * PK + bk * 128 + t] = v;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            tamax[j] = col_amax[cl + j];
            tsc[j] = col_sc[cl + j];
            tr[j] = col_rc[cl + j];
        }
    } else {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < RPT; ++i) m = fmaxf(m, rmax[i]);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
        if (lane == 0) blk_part[wave] = m;
        __syncthreads();
        float bmax = blk_part[0];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) bmax = fmaxf(bmax, blk_part[w]);
        if (t == 0) s_t_tile[(int64_t)bk * (PM >> 7) + bm] = group_scale<MODE>(bmax);
        if (t < 128 && y != nullptr) s[(int64_t)bk * s_kb_stride + (int64_t)(bm * 128 + t) * s_m_stride] = row_sc[t];
        const float bsc = group_scale<MODE>(bmax), brc = 1.0f / bsc;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            tamax[j] = bmax;
            tsc[j] = bsc;
            tr[j] = brc;
        }
    }
    bool tfast = XT == 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) tfast = tfast && group_is_fast<MODE>(tamax[j]);
    uint32_t qlo[RPT], qhi[RPT];   // row i of the transposed copy's bytes: columns 0..3 | 4..7
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        float q[8];
        if (tfast) {
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = qt_quot<MODE, true>(f[i][j], tsc[j], tr[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = qt_quot<MODE, false>(f[i][j], tsc[j], tr[j]);
        }
        qlo[i] = pack4_fp8<MODE>(q[0], q[1], q[2], q[3]);
        qhi[i] = pack4_fp8<MODE>(q[4], q[5], q[6], q[7]);
    }
    // column j of the thread's RPT x 8 bytes = RPT consecutive bytes of row cl+j of the transposed tile
    const uint32_t rl[4] = {qlo[0], qlo[1], qlo[2], qlo[3]};
    const uint32_t rh[4] = {qhi[0], qhi[1], qhi[2], qhi[3]};
    uint32_t c_lo[4], c_hi[4];
    transpose4x4_bytes(rl, c_lo);
    transpose4x4_bytes(rh, c_hi);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        *reinterpret_cast<uint32_t*>(lds.tile_at(cl + j, rg * 4)) = c_lo[j];
        *reinterpret_cast<uint32_t*>(lds.tile_at(cl + 4 + j, rg * 4)) = c_hi[j];
    }
    __syncthreads();
    // y_t[k][m]: thread owns output columns (t%16)*8..+7 (m) of output rows t/16 + NRG*i (k)
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const int kk = rg + NRG * i;
        const uint2 v = *reinterpret_cast<const uint2*>(lds.tile_at(kk, cl));
        // plain (cached) store: the 128-byte pieces that neighbouring tiles write into the same rows of y_t are merged
        // in L2 before they go to memory (non-temporal stores measured 6-10 % slower here; y keeps them)
        *reinterpret_cast<uint2*>(y_t_tile + (int64_t)(bk * 128 + kk) * yt_stride + cl) = v;
    }
}

template <int MODE, int TMODE, bool VEC, int XT, bool CSUM>
__device__ __forceinline__ void quant_transpose_tile(int bm, int bk, const void* __restrict__ x, uint8_t* __restrict__ y,
                                                     float* __restrict__ s, uint8_t* __restrict__ y_t_tile, int yt_stride,
                                                     float* __restrict__ s_t_tile, int M, int K, int64_t x_row_stride, int64_t x_col_stride,
                                                     int PM, int PK, int64_t s_kb_stride, int64_t s_m_stride, int64_t st_k_stride,
                                                     float* __restrict__ col_sum) {
    __shared__ QtLds<CSUM> lds;
    float f[RPT][8];
    load_rows8_f32<XT, VEC, RPT>(x, bm * 128 + (threadIdx.x >> 4) * RPT, bk * 128 + (threadIdx.x & 15) * 8, M, K, x_row_stride, x_col_stride, f);
    quant_transpose_regs<MODE, TMODE, XT, CSUM>(lds, f, bm, bk, y, s, y_t_tile, yt_stride, s_t_tile, PM, PK, s_kb_stride, s_m_stride, st_k_stride,
                                                col_sum);
}

template <int MODE, int TMODE, bool VEC, int XT, bool CSUM = false>
__global__ __launch_bounds__(2048 / RPT, 32 / RPT) void quant_transpose_kernel(const void* __restrict__ x, uint8_t* __restrict__ y,
                                                               float* __restrict__ s, uint8_t* __restrict__ y_t,
                                                               float* __restrict__ s_t, int M, int K,
                                                               int64_t x_row_stride, int64_t x_col_stride, int PM,
                                                               int PK, int64_t s_kb_stride, int64_t s_m_stride,
                                                               int64_t st_a_stride, int64_t st_k_stride,
                                                               float* __restrict__ col_sum) {
    int bm = block_row(), bk = blockIdx.x;
    if (bm >= (PM >> 7)) return;
    xcd_patch(bm, bk, gridDim.x, PM >> 7);
    quant_transpose_tile<MODE, TMODE, VEC, XT, CSUM>(bm, bk, x, y, s, y_t + (int64_t)bm * 128, PM, TMODE == 0 ? s_t + bm * st_a_stride : s_t, M, K,
                                                     x_row_stride, x_col_stride, PM, PK, s_kb_stride, s_m_stride, st_k_stride, col_sum);
}

// The backward pass of a SwiGLU MLP that kept neither activation: from the up/gate projection x [M, 2I] and the activation's gradient d
// [M, I] (bf16, I % 128 == 0), in one pass, what the three products behind it read:
//   act_t          the transposed copy of act = bf16(silu(gate) * up), for the down projection's weight gradient;
//   y, s, y_t, s_t both copies of the gradient [M, 2I] of x, for the input gradient and the up/gate weight gradient.
// The bytes are those of silu_fwd, silu_bwd and the quantizers in turn, which read and write 24 bytes per element of the
// activation (its value and the gradient of x go to memory as bf16 and come back); here it is 6 in and 5 out.  A workgroup computes all three values of its
// 128x128 elements while it has them, keeps them as bf16 (48 registers) and runs the tile of the quantizer three times.  4096 x 2048
// activations: four kernels of 51 us -> 27 us (3.4 TB/s: 512 workgroups, two per CU, go through their loads, 13 us of arithmetic and
// stores side by side); the training step of that MLP, at the power limit, 824 -> 811 us; 1225 tokens, 5376 -> 2x768: 240 -> 183 us
// with the pass's host side in one native call.
// act_t: [PI][PM]; its scales as the dialect's training quantizers lay them out.
template <int MODE>
__global__ __launch_bounds__(2048 / RPT, 16 / RPT) void swiglu_bwd_quant_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ d, uint8_t* __restrict__ act_t, float* __restrict__ act_ts, uint8_t* __restrict__ y,
    float* __restrict__ s, uint8_t* __restrict__ y_t, float* __restrict__ s_t, int M, int I, int up_off, int gate_off, int PM) {
    constexpr bool DEEP = MODE == 1;
    int bm = block_row(), bi = blockIdx.x;
    if (bm >= (PM >> 7)) return;
    xcd_patch(bm, bi, gridDim.x, PM >> 7);
    __shared__ QtLds<false> lds;
    const int row0 = bm * 128 + (threadIdx.x >> 4) * RPT, c0 = bi * 128 + (threadIdx.x & 15) * 8;
    const bool inside = bi * 128 < I;             // beyond: the zero rows that complete act_t to PI (uniform)
    uint32_t wa[RPT][4], wu[RPT][4], wg[RPT][4];
    {
        uint4 ru[RPT], rg[RPT], rd[RPT];
#pragma unroll
        for (int i = 0; i < RPT; ++i) {           // all loads before the first use; rows beyond M repeat the last and become zeros
            const int64_t row = min(row0 + i, M - 1);
            const int c = inside ? c0 : 0;
            ru[i] = load_nt16(x + row * 2 * I + up_off + c);
            rg[i] = load_nt16(x + row * 2 * I + gate_off + c);
            rd[i] = load_nt16(d + row * I + c);
        }
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            float u[8], g[8], e[8], f[8];
            unpack8(ru[i], u);
            unpack8(rg[i], g);
            unpack8(rd[i], e);
            gated8(u, g, wa[i], f);
            gated8_grad(u, g, e, wu[i], wg[i]);
            if (row0 + i >= M || !inside) {
#pragma unroll
                for (int j = 0; j < 4; ++j) wa[i][j] = wu[i][j] = wg[i][j] = 0u;
            }
        }
    }
    const auto floats = [](const uint32_t (&w)[RPT][4], float (&f)[RPT][8]) {
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[i][2 * j] = bf16_lo(w[i][j]);
                f[i][2 * j + 1] = bf16_hi(w[i][j]);
            }
    };
    const int N = 2 * I, MB = PM >> 7;
    float f[RPT][8];
    floats(wa, f);
    quant_transpose_regs<MODE, DEEP ? 1 : 0, 0, false>(lds, f, bm, bi, nullptr, nullptr, act_t + (int64_t)bm * 128, PM, DEEP ? act_ts : act_ts + bm, PM, I,
                                                       0, 0, MB, nullptr);
    if (!inside) return;
    // row scales: DeepLinear [N/128][PM], official [PM][N/128]; of the transposed copy: [PM/128][N] and [N][PM/128]
    const int64_t s_kb = DEEP ? PM : 1, s_m = DEEP ? 1 : N >> 7, st_k = DEEP ? 1 : MB;
    float* s_t_tile = s_t + (DEEP ? (int64_t)bm * N : bm);
    __syncthreads();
    floats(wu, f);
    quant_transpose_regs<MODE, 0, 0, false>(lds, f, bm, (up_off >> 7) + bi, y, s, y_t + (int64_t)bm * 128, PM, s_t_tile, PM, N, s_kb, s_m, st_k, nullptr);
    __syncthreads();
    floats(wg, f);
    quant_transpose_regs<MODE, 0, 0, false>(lds, f, bm, (gate_off >> 7) + bi, y, s, y_t + (int64_t)bm * 128, PM, s_t_tile, PM, N, s_kb, s_m, st_k, nullptr);
}

int launch_swiglu_bwd_quant(const void* x, const void* d, void* act_t, float* act_ts, void* y, float* s, void* y_t, float* s_t, int64_t M, int64_t I,
                            int gate_first, int64_t PM, int64_t PI, int mode, hipStream_t stream) {
    dim3 grid;
    if (!grid_rows(PI / 128, PM / 128, grid)) return kErrTooManyBlocks;
    const int up_off = gate_first ? (int)I : 0, gate_off = gate_first ? 0 : (int)I;
#define MDY_SBQ(MODE)                                                                                                                         \
    launch_kernel((swiglu_bwd_quant_kernel<MODE>), grid, dim3(2048 / RPT), 0, stream, static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(d), \
                       static_cast<uint8_t*>(act_t), act_ts, static_cast<uint8_t*>(y), s, static_cast<uint8_t*>(y_t), s_t, (int)M, (int)I, up_off, gate_off, \
                       (int)PM)
    if (mode == 0) MDY_SBQ(0); else if (mode == 1) MDY_SBQ(1); else MDY_SBQ(2);
#undef MDY_SBQ
    return (int)hipGetLastError();
}

// Expert groups of m_g rows (multiples of 128) one after the other: the row-wise copy and its scales lie as for one matrix, the
// transposed copy [PK][m_g] of every group and its scales are arrays of their own (a caller drops or changes one without the
// others).  One launch for all groups: 8 ragged groups, 5376 rows x 7168 and x 4096, 16 launches of 8.8 us -> 2 launches, 141 -> 57 us.
constexpr int kMaxQtGroups = 128;      // per launch: the table is a kernel argument of 2.5 KB
struct QtGroups {
    int n;
    int row_start[kMaxQtGroups + 1];
    uint8_t* y_t[kMaxQtGroups];
    float* s_t[kMaxQtGroups];
};
template <bool VEC, int XT>
__global__ __launch_bounds__(2048 / RPT, 32 / RPT) void quant_transpose_grouped_kernel(const void* __restrict__ x, uint8_t* __restrict__ y,
                                                                             float* __restrict__ s, int M, int K, int64_t x_row_stride,
                                                                             int64_t x_col_stride, int64_t s_kb_stride, const QtGroups groups) {
    int bm = block_row(), bk = blockIdx.x;
    if (bm >= (M >> 7)) return;
    xcd_patch(bm, bk, gridDim.x, M >> 7);
    int lo = 0, hi = groups.n - 1;                       // the last group that starts at or before the tile (empty ones skipped)
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (groups.row_start[mid] <= bm * 128) lo = mid; else hi = mid - 1;
    }
    const int r0 = groups.row_start[lo];
    quant_transpose_tile<1, 0, VEC, XT, false>(bm, bk, x, y, s, groups.y_t[lo] + (bm * 128 - r0), groups.row_start[lo + 1] - r0,
                                               groups.s_t[lo] + (int64_t)(bm - (r0 >> 7)) * K, M, K, x_row_stride, x_col_stride, M, K, s_kb_stride, 1, 1,
                                               nullptr);
}

// Shared launcher.  mode: dialect (0 official, column groups only; 1 DeepLinear); t_mode: 0 per column group, 1 per
// 128x128 block.
static int launch_qt(int mode, const void* x, int x_dtype, void* y, float* s, void* y_t, float* s_t, int64_t M, int64_t K,
                     int64_t x_row_stride, int64_t x_col_stride, int64_t PM, int64_t PK, int64_t s_kb_stride,
                     int64_t s_m_stride, int64_t st_a_stride, int64_t st_k_stride, int t_mode, hipStream_t stream) {
    if (PM == 0 || PK == 0) return 0;
    dim3 grid;
    if (!grid_rows(PK / 128, PM / 128, grid)) return kErrTooManyBlocks;
    const dim3 block(2048 / RPT);
    const bool vec = rows_vectorizable(x, K, x_row_stride, x_col_stride, xt_size(x_dtype));
    uint8_t* yp = static_cast<uint8_t*>(y);
    uint8_t* ytp = static_cast<uint8_t*>(y_t);
#define MDY_QT(MODE, TM, VEC, XT)                                                                                        \
    launch_kernel((quant_transpose_kernel<MODE, TM, VEC, XT>), grid, block, 0, stream, x, yp, s, ytp, s_t,          \
                       (int)M, (int)K, x_row_stride, x_col_stride, (int)PM, (int)PK, s_kb_stride, s_m_stride,           \
                       st_a_stride, st_k_stride, static_cast<float*>(nullptr))
#define MDY_QT_V(MODE, TM, XT) do { if (vec) MDY_QT(MODE, TM, true, XT); else MDY_QT(MODE, TM, false, XT); } while (0)
#define MDY_QT_X(MODE, TM) do { if (x_dtype == 0) MDY_QT_V(MODE, TM, 0); else if (x_dtype == 1) MDY_QT_V(MODE, TM, 1); else MDY_QT_V(MODE, TM, 2); } while (0)
    if (mode == 0) MDY_QT_X(0, 0);
    else if (mode == 2) MDY_QT_X(2, 0);
    else if (t_mode == 0) MDY_QT_X(1, 0);
    else MDY_QT_X(1, 1);
#undef MDY_QT_X
#undef MDY_QT_V
#undef MDY_QT
    return (int)hipGetLastError();
}

int launch_quant_transpose(const void* x, int x_dtype, void* y, float* s, void* y_t, float* s_t, int64_t M, int64_t K,
                           int64_t x_row_stride, int64_t x_col_stride, int64_t PM, int64_t PK, int64_t s_kb_stride,
                           int t_mode, hipStream_t stream) {
    // DeepLinear layouts: row scales [PK/128][s_kb_stride >= PM], column-group scales [PM/128][PK]
    return launch_qt(1, x, x_dtype, y, s, y_t, s_t, M, K, x_row_stride, x_col_stride, PM, PK, s_kb_stride, 1, PK, 1, t_mode, stream);
}

int launch_act_quant_transpose(const void* x, int x_dtype, void* y, float* s, void* y_t, float* s_t, int64_t M, int64_t K,
                               int64_t x_row_stride, int64_t x_col_stride, int64_t PM, int64_t PK, int mode, hipStream_t stream) {
    // official layouts, both row-major: s [PM][PK/128], s_t [PK][PM/128]; mode 0 (e4m3fn) or 2 (e5m2)
    return launch_qt(mode == 2 ? 2 : 0, x, x_dtype, y, s, y_t, s_t, M, K, x_row_stride, x_col_stride, PM, PK, 1, PK / 128, 1, PM / 128, 0, stream);
}

// M = sum of m_splits, every one a multiple of 128, K a multiple of 128; y_t, s_t: host arrays of G device pointers
int launch_quant_transpose_grouped(const void* x, int x_dtype, void* y, float* s, void* const* y_t, float* const* s_t, const int64_t* m_splits,
                                   int64_t G, int64_t M, int64_t K, int64_t x_row_stride, int64_t x_col_stride, hipStream_t stream) {
    if (K == 0) return 0;
    const bool vec = rows_vectorizable(x, K, x_row_stride, x_col_stride, xt_size(x_dtype));
    int64_t row0 = 0;
    for (int64_t g0 = 0; g0 < G; g0 += kMaxQtGroups) {
        QtGroups groups = {};
        groups.n = (int)(G - g0 < kMaxQtGroups ? G - g0 : kMaxQtGroups);
        int rows = 0;
        for (int g = 0; g < groups.n; ++g) {
            groups.row_start[g] = rows;
            groups.y_t[g] = static_cast<uint8_t*>(y_t[g0 + g]);
            groups.s_t[g] = s_t[g0 + g];
            rows += (int)m_splits[g0 + g];
        }
        groups.row_start[groups.n] = rows;
        if (rows == 0) continue;
        dim3 grid;
        if (!grid_rows(K / 128, rows / 128, grid)) return kErrTooManyBlocks;
        const void* xg = static_cast<const uint8_t*>(x) + row0 * x_row_stride * xt_size(x_dtype);
        uint8_t* yg = static_cast<uint8_t*>(y) + row0 * K;
        float* sg = s + row0;
#define MDY_QTG(VEC, XT)                                                                                                        \
    launch_kernel((quant_transpose_grouped_kernel<VEC, XT>), grid, dim3(2048 / RPT), 0, stream, xg, yg, sg, rows, (int)K, x_row_stride, \
                       x_col_stride, M, groups)
#define MDY_QTG_V(XT) do { if (vec) MDY_QTG(true, XT); else MDY_QTG(false, XT); } while (0)
        if (x_dtype == 0) MDY_QTG_V(0); else if (x_dtype == 1) MDY_QTG_V(1); else MDY_QTG_V(2);
#undef MDY_QTG_V
#undef MDY_QTG
        const int rc = (int)hipGetLastError();
        if (rc != 0) return rc;
        row0 += rows;
    }
    return 0;
}

// bf16(sum over the row tiles of part[a][k]; zeros without any): 32 columns x 8 interleaved shares of the row tiles per block.  Bound by
// the latency of its loads: eight of a thread are in flight at a time, added in the order of the row tiles (one after the other 16384x512
// 6.3 us, now 4.1, which is what a launch takes; 8192x4096 4.7 -> 4.5).
__global__ __launch_bounds__(256) void col_sum_reduce_kernel(const float* __restrict__ part, uint16_t* __restrict__ out, int A, int K, int PK) {
    __shared__ float share[8][32];
    const int c = threadIdx.x & 31, g = threadIdx.x >> 5, k = blockIdx.x * 32 + c;      // k < PK: PK % 128 == 0
    float v = 0.0f;
    for (int a0 = g; a0 < A; a0 += 64) {
        float p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = part[(int64_t)min(a0 + 8 * u, A - 1) * PK + k];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (a0 + 8 * u < A) v += p[u];
    }
    share[g][c] = v;
    __syncthreads();
    if (g == 0 && k < K) {
#pragma unroll
        for (int h = 1; h < 8; ++h) v += share[h][c];
        out[k] = (uint16_t)(pack2_bf16(v, 0.0f) & 0xFFFFu);
    }
}

int launch_quant_transpose_colsum(const void* x, void* y, float* s, void* y_t, float* s_t, int64_t M, int64_t K, int64_t x_row_stride,
                                  int64_t x_col_stride, int64_t PM, int64_t PK, int64_t s_kb_stride, int mode, float* part, void* col_sum,
                                  hipStream_t stream) {
    if (PK == 0) return 0;
    dim3 grid;
    if (PM > 0 && !grid_rows(PK / 128, PM / 128, grid)) return kErrTooManyBlocks;
    const bool vec = rows_vectorizable(x, K, x_row_stride, x_col_stride, 2);
    const bool deep = mode == 1;
    const int64_t s_kb = deep ? s_kb_stride : 1, s_m = deep ? 1 : PK / 128, st_a = deep ? PK : 1, st_k = deep ? 1 : PM / 128;
#define MDY_QTC(MODE, VEC)                                                                                                        \
    launch_kernel((quant_transpose_kernel<MODE, 0, VEC, 0, true>), grid, dim3(2048 / RPT), 0, stream, x, static_cast<uint8_t*>(y), s, \
                       static_cast<uint8_t*>(y_t), s_t, (int)M, (int)K, x_row_stride, x_col_stride, (int)PM, (int)PK, s_kb, s_m, st_a, st_k, part)
#define MDY_QTC_V(MODE) do { if (vec) MDY_QTC(MODE, true); else MDY_QTC(MODE, false); } while (0)
    if (PM > 0) {
        if (mode == 0) MDY_QTC_V(0); else if (mode == 1) MDY_QTC_V(1); else MDY_QTC_V(2);
    }
#undef MDY_QTC_V
#undef MDY_QTC
    const int rc = (int)hipGetLastError();
    if (rc != 0 || K == 0) return rc;
    launch_kernel(col_sum_reduce_kernel, dim3((unsigned)((K + 31) / 32)), dim3(256), 0, stream, part, static_cast<uint16_t*>(col_sum),
                       (int)(PM / 128), (int)K, (int)PK);
    return (int)hipGetLastError();
}

}  // namespace mdy
