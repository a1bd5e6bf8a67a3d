// The MFMA tile body of the block-scaled FP8 GEMM and the kernel that walks tiles with it (gfx950 only).
// Shared by fp8_gemm.hip (the product kernels) and gemm_probe.hip (the timing probe that switches parts of the
// K loop off); the description of the kernels is at the top of fp8_gemm.hip.  Two bodies: fp8_gemm_tile (every wave
// does everything; the large tiles) and fp8_gemm_tile_ws (producer / consumer waves; 64x128, 128x64, 128x128 and 128x192 tiles).
#pragma once
#include <type_traits>

#include "common.h"

namespace mdy {

// chunk swizzle of an LDS row; depends on row bits 0..3 only so that rows 16 apart share it
__device__ __forceinline__ int swz(int row) { return (row & 7) ^ ((row >> 3) & 1); }

// One 128-deep scale block of a 16x16 sub-tile, from zero: v_mfma_f32_16x16x128_f8f6f4 with e4m3 operands and unit
// hardware scales.  The weight rows go in as the MFMA's rows and the activation rows as its columns, so a lane's
// four results are four consecutive n of one m.
// FMT: byte format of both operands, 0 e4m3fn, 1 e5m2 (the instruction's cbsz / blgp fields).
template <int FMT = 0>
__device__ __forceinline__ floatx4 mfma_block(const intx8& weight_rows, const intx8& act_rows) {
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(weight_rows, act_rows, zero, FMT, FMT, 0, 0, 0, 0);
}

// The promotion of one K block (offical_kernel.py:86): acc += (MFMA result of the block) * (its combined scale).
__device__ __forceinline__ void fold(floatx4& acc, const floatx4& p, float sc) {
    acc[0] = __builtin_fmaf(p[0], sc, acc[0]);
    acc[1] = __builtin_fmaf(p[1], sc, acc[1]);
    acc[2] = __builtin_fmaf(p[2], sc, acc[2]);
    acc[3] = __builtin_fmaf(p[3], sc, acc[3]);
}

// Products of row scales for four sub-tiles at a time, laid out like the results of four mfma_block: v_mfma_f32_16x16x1_4b, each product an
// FMA onto zero and so rounded as v_mul_f32 rounds it.  Lane l holds the scale of row l of four sub-tiles.  ALL_WEIGHTS: the four weight
// sub-tiles against activation sub-tile ONE of its four (blgp 4..7 broadcasts 16 lanes), otherwise weight sub-tile ONE (cbsz / abid) against
// the four activation sub-tiles.  Eight of these per 128x64 wave tile and K block replace 128 multiplies (32 clocks of a SIMD's matrix core, 8 passes, for
// what takes its VALU 64) and 16 to 24 registers of scales; same bits.  4096x7168x512 25.3 -> 24.6 us, x1024 39.7 -> 37.5, x4096 120.6 -> 115.0,
// 2048x2048x2048 15.2 -> 14.0; 200 drawn shapes 3.5 % less time in the mean, none more beyond 2 %.  An MFMA between the products and their
// first use, in place of the wait states there, is slower (4096x7168x1024 37.9).
template <bool ALL_WEIGHTS, int ONE>
__device__ __forceinline__ floatx16 scale_products(float weight_scales, float act_scales) {
    const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(weight_scales, act_scales, zero, ALL_WEIGHTS ? 0 : 2, ALL_WEIGHTS ? 0 : ONE, ALL_WEIGHTS ? 4 + ONE : 0);
}

template <typename OUT>
__device__ __forceinline__ void store4(OUT* c, int64_t ldc, int m, int n, int M, int N, const float (&v)[4], bool vec_ok) {
    if (m >= M || n >= N) return;
    OUT* p = c + (int64_t)m * ldc + n;
    if (vec_ok && n + 3 < N) {
        // plain (cached) stores: the 8-byte pieces of a line written by different instructions are
        // merged in L2; non-temporal stores measured ~5 % slower here
        if (sizeof(OUT) == 2) {
            *reinterpret_cast<uint2*>(p) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        } else {
            *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (n + i < N) {
                if (sizeof(OUT) == 2)
                    reinterpret_cast<uint16_t*>(p)[i] = (uint16_t)(pack2_bf16(v[i], 0.0f) & 0xFFFFu);
                else
                    reinterpret_cast<float*>(p)[i] = v[i];
            }
        }
    }
}

// How a tile kernel writes its results: a template parameter, chosen by the host from N, ldc and the alignment of c (epilogue_kind).
// With all three forms in one kernel the longer code costs every launch 0.15 us and 4096x1544x7168 1 us of 53.
constexpr int kEpiDirect = 0;      // straight from registers, 8 (bf16) or 16 (fp32) bytes per lane, any N and alignment
constexpr int kEpiLines = 1;       // bf16 through LDS in whole rows that start on 128-byte lines, non-temporal
constexpr int kEpiRows = 2;        // through LDS in whole rows, cached: fp32, and bf16 rows that start inside lines

// Between LDS writes of some lanes of a wave and reads of them by others (or the other way round).  The hardware executes a wave's LDS
// accesses in order; this keeps the compiler from moving one across.  No instruction.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Epilogue of one wave's TI x TJ sub-tiles for bf16 results: through the wave's own part of LDS (TI * 16 rows of TJ * 32 bytes,
// free once the K loop is over), so that a store instruction writes whole rows of the wave tile, 16 bytes per lane, instead of
// 8-byte pieces of 16 different rows: a quarter of the cache lines per instruction and half the instructions.  All CUs end
// a round of tiles together, so the stores of a tile are exposed; direct 8-byte stores -> rows through LDS -> the same with
// non-temporal stores (whole lines, never read again by this kernel), operands rotating over three buffers:
// 4096x18432x7168 473 -> 456 -> 451 us, 8192x4096x4096 126 -> 120 -> 117 us, 16384x4096x1024 100 -> 91 -> 84 us, 4096x7168x2048
// 70 -> 63 -> 63 us, with row scales 4096x7168x512 45 -> 36 -> 35 us.  Where rows do not start on 128-byte lines a wave's rows
// end inside lines that its neighbours complete, and the stores stay cached so that L2 joins the parts (3752x15224x768: 82 us direct, 86 through
// LDS non-temporal, 80 through LDS cached).  The 16-byte pieces of a row are XOR-swizzled by
// the row: no bank conflict of the reads; of the writes rows r and r + 8 meet in pairs, 4 cycles a write.  Needs N % 8 == 0 and 16-byte aligned rows of c (the caller checks).
// fp32 results (the slabs of a K split, an fp32 output) go the same way with twice the row length where the pool holds them;
// those stores stay cached: the reduction reads the slabs next.
template <int TI, int TJ, typename OUT, bool NT>
__device__ __forceinline__ void store_rows(const floatx4 (&acc)[TI][TJ], uint8_t* buf, OUT* __restrict__ c, int64_t ldc,
                                           const Bias bias, int m_base, int n_base, int M, int N, int lane) {
    static_assert(TJ % 2 == 0, "a row is a multiple of four 16-byte pieces");
    constexpr bool HALF = sizeof(OUT) == 2;
    constexpr int EPP = 16 / sizeof(OUT);      // elements per 16-byte piece
    constexpr int CH = TJ * 16 / EPP, ROW = CH * 16, MASK = CH % 8 == 0 ? 7 : 3;
    asm volatile("" : "+v"(lane));      // the addresses below belong here and not in registers held across the K loop
    const int frow = lane & 15, fk = lane >> 4;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        const int n = n_base + j * 16 + 4 * fk;
        if (bias.p != nullptr && n < N) {      // N is a multiple of the piece: all four columns are in range
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[e] = bf16_one(bias.p[n + e]);
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            floatx4 v = acc[i][j];
            if (bias.after_rounding) {
                const uint32_t lo = pack2_bf16(v[0], v[1]), hi = pack2_bf16(v[2], v[3]);
                v = floatx4{bf16_lo(lo), bf16_hi(lo), bf16_lo(hi), bf16_hi(hi)};
            }
            uint8_t* row = buf + (i * 16 + frow) * ROW;
            if (HALF)
                *reinterpret_cast<uint2*>(row + (((2 * j + (fk >> 1)) ^ (frow & MASK)) << 4) + (fk & 1) * 8) =
                    make_uint2(pack2_bf16(v[0] + bv[0], v[1] + bv[1]), pack2_bf16(v[2] + bv[2], v[3] + bv[3]));
            else
                *reinterpret_cast<float4*>(row + (((4 * j + fk) ^ (frow & MASK)) << 4)) =
                    make_float4(v[0] + bv[0], v[1] + bv[1], v[2] + bv[2], v[3] + bv[3]);
        }
    }
    wave_lds_fence();
#pragma unroll
    for (int t = 0; t < TI * CH / 4; ++t) {
        const int q = t * 64 + lane, row = q / CH, ch = q % CH;
        const int m = m_base + row, n = n_base + ch * EPP;
        const uint4 v = *reinterpret_cast<const uint4*>(buf + row * ROW + ((ch ^ (row & MASK)) << 4));
        if (m < M && n < N) {
            if (NT) store_nt16(c + (int64_t)m * ldc + n, v);
            else *reinterpret_cast<uint4*>(c + (int64_t)m * ldc + n) = v;
        }
    }
}

// a byte offset beyond every descriptor of these kernels (their ranges stay below 2^31): such a lane accesses nothing
constexpr int kOutOfRange = 0x7ffffff0;

// store_rows for a wave of 64 bf16 columns through 2 KB of LDS, 16 rows at a time, in exactly TI * 2 store instructions: a bounded
// descriptor drops what lies outside, no branch skips one, so a wait can count past them (NEXT of fp8_gemm_tile).
template <int TI, bool NT>
__device__ __forceinline__ void store_rows_beside(const floatx4 (&acc)[TI][4], uint8_t* buf, uint16_t* __restrict__ c, int ldc, const Bias bias,
                                                  int m0, int m_wave, int n_base, int M, int rows, int N, int lane) {
    asm volatile("" : "+v"(lane));      // as in store_rows
    const int frow = lane & 15, fk = lane >> 4, ch = lane & 7;
    float bv[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n_base + j * 16 + 4 * fk;
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[j][e] = 0.0f;
        if (bias.p != nullptr && n < N) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[j][e] = bf16_one(bias.p[n + e]);
        }
    }
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(c + (size_t)m0 * ldc, 0, min(rows, M - m0) * ldc * 2, 0x00020000);
    const int n = n_base + ch * 8;
    const int off = n < N ? ((m_wave + (lane >> 3)) * ldc + n) * 2 : kOutOfRange;
    const int row_step = n < N ? 16 * ldc : 0;      // bytes of 8 rows
    const auto store = [&](auto round_first) __attribute__((always_inline)) {
        uintx4_t v[2][2];      // rows on their way: those of step i - 1 are stored while the ones of step i come back from LDS
#pragma unroll
        for (int i = 0; i <= TI; ++i) {
            if (i < TI) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    floatx4 r = acc[i][j];
                    if (decltype(round_first)::value) {
                        const uint32_t lo = pack2_bf16(r[0], r[1]), hi = pack2_bf16(r[2], r[3]);
                        r = floatx4{bf16_lo(lo), bf16_hi(lo), bf16_lo(hi), bf16_hi(hi)};
                    }
                    *reinterpret_cast<uint2*>(buf + frow * 128 + (((2 * j + (fk >> 1)) ^ (frow & 7)) << 4) + (fk & 1) * 8) =
                        make_uint2(pack2_bf16(r[0] + bv[j][0], r[1] + bv[j][1]), pack2_bf16(r[2] + bv[j][2], r[3] + bv[j][3]));
                }
                wave_lds_fence();
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int row = t * 8 + (lane >> 3);
                    v[i & 1][t] = *reinterpret_cast<const uintx4_t*>(buf + row * 128 + ((ch ^ (row & 7)) << 4));
                }
                wave_lds_fence();      // the next 16 rows are written to the same place
            }
            if (i > 0) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    __builtin_amdgcn_raw_buffer_store_b128(v[(i - 1) & 1][t], rsrc, off + (2 * (i - 1) + t) * row_step, 0, NT ? 2 : 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (bias.after_rounding) store(std::true_type{});
    else store(std::false_type{});
}

// The form of a launch.  Rows that do not start on whole lines go through LDS with 256x256 tiles only (3752x15224x768 83.0 us
// direct -> 81.1; the narrower tiles tie or lose a little), fp32 results wherever the pool holds them (`fits`).
inline int epilogue_kind(const void* c, int64_t ldc, int64_t N, int esz, bool big_tile, bool fits) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(c);
    if (!fits || ((N | ldc) & (16 / esz - 1)) != 0 || (p & 15) != 0 || (big_tile && ldc >= (1 << 21))) return kEpiDirect;      // (256 rows within 2^31 bytes)
    if (esz != 2) return kEpiRows;
    return ((ldc * esz) & 127) == 0 && (p & 127) == 0 ? kEpiLines : big_tile ? kEpiRows : kEpiDirect;
}

// raw buffer descriptor: base, byte range, no stride, no swizzle
__device__ __forceinline__ intx4 make_rsrc(const void* base, uint32_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    intx4 r;
    r[0] = (int)(uint32_t)p;
    r[1] = (int)((uint32_t)(p >> 32) & 0xFFFFu);
    r[2] = (int)bytes;
    r[3] = 0x00020000;
    return r;
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const void*)p);
}
// 64 lanes x 16 bytes, global (descriptor base + voff + soff) -> LDS (lds + lane*16).
// Issued as inline asm so that the copy stays asynchronous: the kernel waits for it
// with an explicit s_waitcnt vmcnt + barrier once per K block, nowhere else.
// rsrc, soff and lds must be wave-uniform.
__device__ __forceinline__ void dma16(const intx4& rsrc, int voff, int soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :: "v"(voff), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
}
__device__ __forceinline__ void dma4(const intx4& rsrc, int voff, int soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds"
                 :: "v"(voff), "s"(rsrc), "s"(soff), "s"(lds) : "memory");
}

// Shares of the panel pre-touches: the A panel of a tile row is cut into 2^a_sh shares among the tiles of
// that row that run side by side, the B panel of a tile column into 2^b_sh shares among its tile rows.
// In the producer/consumer kernel a touch covers kTouchBurst CONSECUTIVE lines (K blocks) of a row at a time: a K
// block's copy needs one 128-byte line from each of a panel's rows, rows that lie K bytes apart - for memory that is
// one isolated line per DRAM page and K block.  Touching 4 lines (512 contiguous bytes) of a row every 4th K block
// instead of one line every K block asks memory for the same bytes in a quarter of the places.  Measured one launch
// after a cache flush (operands cold, caches full of dirty lines), same process, row-major scales: 4096x1536x7168
// 63.5 -> 57.2 us, 2048x2048x7168 52.7 -> 44.2 us, 2048x1024x7168 44.6 -> 34.4 us, 1024x4096x7168 54.0 -> 44.8 us;
// bursts of 2 / 8 / 16 lines are 1.5 / 1.4 / 4.3 us slower than 4 at the first shape; touching single lines further
// ahead (5 or 8 K blocks instead of 2) changes nothing; relaunched back to back (operands in the caches) all tie.
// The one-body kernel (hundreds of tiles, many workgroups on every panel) keeps single-line touches: bursts made
// 4096x18432x7168 472 -> 491 us and 4096x7168x18432 455 -> 468 us back to back.
constexpr int kTouchBurstLog = 2, kTouchBurst = 1 << kTouchBurstLog;
struct Duty {
    int a_duty, a_sh, b_duty, b_sh;
};

// LDS of one tile workgroup, carved out of a pool that the kernel declares: the ring of A and B panels, the ring of activation scales, the tile's weight
// scales for all K blocks, and a dummy area for copies that must go nowhere.
//
// CHUNKED (with BROW): row scales, of the activations and behind them of the weight rows, come in chunks of 4 K blocks, [group of 16 rows][row]
// [K block % 4]: a copy of a wave takes 16 rows x 4 K blocks, which with row-major scales, the official dialect's, is 16 lines; one K block of 64
// rows is 64.  Part r of a chunk (groups r * WAVES ..) goes out with the copies of the K block PARTS - 1 - r in front of the chunk.  With row scales on
// both sides, 16 lines a copy of the 32 that a chunk takes instead of 64 of 32: 8192x4096x4096 row-major 138 -> 129 us; column-major ones lie together
// anyway and lose 1 to 2 % with 256x256 tiles, 2 to 8 % with 128x128 (launch_fp8_gemm_nt_rowscaled says when).  One operand's row scales are copied a
// K block at a time: in chunks 128x256 tiles tie right behind the quantizer and lose otherwise (1500x4096x4096 34.1 -> 35.9 us, 2048x4096x3072
// 27.5 -> 28.1, a weight's rotating copies), 256x256 lose (2048x18432x2048 82.9 -> 85.9), 64x64 tie.
// Without chunks, the weight rows' scales of STAGES K blocks lie where the weight's block scales would.
template <int BM, int BN, int WAVES, int STAGES, bool BROW = false, bool CHUNKED = false>
struct TileLds {
    static constexpr int NBS = (BN + 127) / 128;
    static constexpr int GROUPS = BM / 16 + BN / 16, PARTS = CHUNKED ? (GROUPS + WAVES - 1) / WAVES : 1;
    // Part 0 of chunk c + 1 is copied behind the barrier of K block 4 c + 5 - PARTS - STAGES, when the scales of the next one are read: the chunks
    // from that one's to c + 1 have a buffer each.
    static constexpr int CHUNKS = PARTS + STAGES <= 6 ? 2 : 2 + (PARTS + STAGES - 6 + 3) / 4;
    static constexpr int a_off = 0;
    static constexpr int b_off = a_off + STAGES * BM * 128;
    static constexpr int s_off = b_off + STAGES * BN * 128;
    static constexpr int bs_off = s_off + (CHUNKED ? CHUNKS * GROUPS * 256 : (STAGES * BM * 4 + 255) / 256 * 256);
    static constexpr int dummy_off = bs_off + (!BROW ? NBS * 512 * 4 : CHUNKED ? 0 : STAGES * BN * 4);
    static constexpr int bytes = dummy_off + WAVES * 512;
    // A workgroup that walks its tiles: 16 rows of results of every wave on their way to memory, beside a ring that already
    // receives the next tile.  256x256 tiles with row scales on both sides fill the CU's LDS without a dummy area: a wave's touches go where its
    // rows of results go later.
    static constexpr bool no_dummy = CHUNKED && bytes + WAVES * 2048 > 160 * 1024;
    static constexpr int rows_off = no_dummy ? dummy_off : bytes, walk_bytes = rows_off + WAVES * 2048;
};

// LDS of a wave-specialized tile workgroup: separate ring depths for the a panels and the b panels, and a ring of kScaleChunks chunks of activation
// scales, 4 K blocks each.
constexpr int kScaleChunks = 4;
template <int BM, int BN, int WAVES, int SA, int SB>
struct TileLdsWs {
    static constexpr int NBS = (BN + 127) / 128;
    static constexpr int BSROW = 512;
    static constexpr int a_off = 0;
    static constexpr int b_off = a_off + SA * BM * 128;
    static constexpr int s_off = b_off + SB * BN * 128;
    static constexpr int bs_off = s_off + kScaleChunks * BM * 16;
    static constexpr int dummy_off = bs_off + NBS * BSROW * 4;
    static constexpr int bytes = dummy_off + WAVES * 512;
};
// Ring depths: of the operand that a consumer streams through registers during a K block, and of the one it holds, read a block earlier.  4 K blocks, as the
// K loop is unrolled by 4 and the buffers' addresses are then part of the LDS instructions; 3 where LDS has no room for more (the held operand's buffer is
// free a block earlier).  Deeper rings, 5 K blocks streamed, put one more block in flight and lose (128x128: 0 to 5 % more time, 300x7168x4096 18.0 -> 18.6
// us, 2048x2048x512 6.6 -> 6.9) or tie (128x64, 64x128).
template <int BM, int BN>
struct WsRings {
    static constexpr bool HOLD_A = BM / 2 <= BN / 2;      // 2 x 2 consumers
    static constexpr int STREAM = 4, HOLD = BM * BN > 128 * 128 ? 3 : 4;
    static constexpr int SA = HOLD_A ? HOLD : STREAM, SB = HOLD_A ? STREAM : HOLD;
    using L = TileLdsWs<BM, BN, 8, SA, SB>;
};

// the `next` of a workgroup that computes one tile
struct OneTile {};

// One BM x BN tile of C: WGM x WGN waves, each wave (BM/WGM) x (BN/WGN).
//   rows m0 .. min(m0+BM, m_end) of a (m_end = end of the matrix, or of the expert group the tile belongs to),
//   columns n0 .. of b / b_s / bias (already offset to the group's weight), K % 128 == 0, K <= 65536,
//   K blocks kb0 .. kb1-1 of them (all of them except in the split-K kernel).
// as_bytes = byte size of the addressed part of a_s (host computed, < 2^31); m_total = rows of a_s.
// duty: which share of the A / B panel lines this workgroup pre-touches for the workgroups that copy the same
// panels (those with the same tile row / tile column), and into how many shares the panels are cut.
//
// Schedule of one K block (NT = TI*TJ MFMA slots, each followed DEPTH slots later by its 4 FMAs):
//   slots 0..      the last copies of K block kb+1 (those that did not fit into the tail below), one per GAP
//                  slots, then one "duty touch" load for K block kb+3;
//   slot TB        = first MFMA of the last streamed fragment: every LDS read of this K block has been
//                  consumed, so the wave waits for its copies of kb+1 and meets the others at THE barrier
//                  of the K block; behind it buffer `cur` is free and buffer `cur^1` is complete;
//   slots TB..     while the last MFMAs and FMAs of kb still run: reload the held fragments, the first
//                  streamed fragment and the scales from buffer cur^1, and issue the first copies of kb+2
//                  into buffer cur, one per GAP slots.
// So the LDS latency after the barrier and the issue time of the copies sit in the shadow of the matrix
// pipe instead of in front of the first MFMA of the next K block.
// BROW_: the weight operand carries one scale per ROW and K block (b_s[n * bs_rs + kb * bs_cs], bs_bytes long) instead of
// one per 128x128 block: the scales of the tile's BN rows travel through LDS per K block like the activation scales
// (copied by the waves behind the activation-scale waves), and scale_products multiplies the two for a streamed fragment behind the
// last MFMA of it, when the products of the fragment before have been folded.
//
// NEXT: a workgroup that walks its tiles passes next(m0, n0, duty) -> bool, which moves on to its next tile.  The copies of that
// tile's first two K blocks are then issued BEFORE the results of this one are stored (through LDS beside the ring).  Loads
// and stores complete in order, so with the stores first every wait for a copy was a wait for the stores as well: all CUs end
// a tile together and stood still for the 33 MB of a round.  Now the first two K blocks of a tile run while the stores of the
// last one drain: 4096x7168x512 with row scales 28.4 -> 24.9 us, 8192x8192x512 55 -> 50 us, 3752x15224x768 71 -> 64.5 us,
// 16384x4096x1024 81 -> 76 us, 8192x4096x4096 117.5 -> 116 us; at the power limit of a long K it ties (4096x18432x7168).
// (Those without a bias.  With one its loads complete behind the copies that went out in front of them, and the stores wait for
// both: 0 to 4 us more, 3752x15224x768 64.5 -> 68.6 us, 16384x4096x1024 78.1 -> 79.4, none from K = 4096 on.)
template <int BM, int BN, int WGM, int WGN, int STAGES, typename OUT, int GAP_ = 0, int TD_ = 0, int ABL_ = 0, int FMT_ = 0,
          bool BROW_ = false, int EPI_ = kEpiDirect, bool CHUNKED_ = false, typename NEXT = OneTile>
__device__ __forceinline__ void fp8_gemm_tile(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, OUT* __restrict__ c,
    const Bias bias, int m0, int m_end, int m_total, int n0, int N, int K, int ldc, Duty duty,
    int kb0, int kb1, uint8_t* __restrict__ pool, int bs_rs = 0, int bs_cs = 0, uint32_t bs_bytes = 0, NEXT next = NEXT{}) {
    constexpr bool WALK = !std::is_same<NEXT, OneTile>::value;
    // ABL_ switches parts of the K loop off for the timing probe (mdy_fp8_gemm_probe); the product uses 0.
    //   1: no global->LDS copies in the loop (the ring is filled once and replayed)   2: no LDS fragment / scale reads
    //   4: no FMA fold (the MFMAs accumulate in place, no block scales)                8: no pre-touches
    constexpr bool NO_COPY = (ABL_ & 1) != 0, NO_LDS = (ABL_ & 2) != 0, NO_FOLD = (ABL_ & 4) != 0;
    constexpr bool NO_TOUCH = (ABL_ & 8) != 0 || NO_COPY;
    constexpr int WAVES = WGM * WGN;
    constexpr int WM = BM / WGM, WN = BN / WGN, TI = WM / 16, TJ = WN / 16;
    constexpr int PASS_ROWS = WAVES * 8;  // rows copied by one DMA instruction of every wave
    constexpr int A_PASSES = BM / PASS_ROWS, B_PASSES = BN / PASS_ROWS;
    constexpr int DEPTH = 4;              // MFMAs in flight before their results are folded
    static_assert(BM % PASS_ROWS == 0 && BN % PASS_ROWS == 0 && PASS_ROWS % 16 == 0, "tile/threads mismatch");
    // A wave's WN columns lie in one 128-column weight-scale block when WN divides 128 (tiles then start on multiples
    // of WN); the 192-wide tile (WN = 48, tiles start on multiples of 64) can straddle two: its 16-column sub-tiles never
    // do, so such a wave keeps two combined scales per row and each sub-tile takes the one of its block.
    constexpr bool STRADDLE = (128 % WN) != 0;
    static_assert(WN <= 128 && (!STRADDLE || BN == 192) && WAVES >= 2, "weight-scale blocks per wave column");
    constexpr bool HOLD_A = TI <= TJ;
    constexpr int NH = HOLD_A ? TI : TJ, NS = HOLD_A ? TJ : TI;
    constexpr int NT = TI * TJ;
    constexpr int NDMA = 1 + A_PASSES + B_PASSES;       // copies per K block and wave: scales, A passes, B passes
    constexpr int TB = NT - NH;                         // slot of the barrier
    constexpr int NSLOT = NT + DEPTH;                   // slots of a K block (the last DEPTH hold FMAs only)
    // Copy j of a K block goes out in slot TB+1 + GAP*j, counted on from the barrier of the block two before it
    // and running over into the first slots of the next block.  With 8 waves one copy per slot and wave is
    // twice what the CU's address unit takes (64 lanes x 16 bytes = 16 clocks each, a slot is 64 clocks for
    // the two waves of a SIMD): the waves then queue on the copy instruction and their MFMAs behind it wait.
    // Measured: 256x256 tiles 1-5 % faster with every second slot; 128x256 and 128x192 tiles 2-7 % at 4096x1536x7168.
    constexpr int GAP = GAP_ > 0 ? GAP_ : (WAVES >= 8 && NT >= 12) ? 2 : 1;
    constexpr int TAIL = (NSLOT - TB - 1 + GAP - 1) / GAP;   // copies that still fit behind the barrier
    constexpr int FIRST = TAIL < NDMA ? TAIL : NDMA;         // copies of K block kb+2 issued in the tail of kb
    constexpr int TOUCH = FIRST < NDMA ? TB + 1 + GAP * (NDMA - 1) - NSLOT + 1 : 0;   // slot after the last copy
    constexpr int TD = TD_ > 0 ? TD_ : STAGES + 1;      // duty touches run this many K blocks ahead (in front of the copies)
    // loads younger than the last copy of K block kb+1 when the wave waits for it in K block kb: the copies of
    // blocks kb+2 .. kb+STAGES-1 and one touch per K block since (loads complete in order, so vmcnt(YOUNGER)
    // means "block kb+1 has landed")
    constexpr int YOUNGER = (STAGES - 2) * NDMA + STAGES - 1;
    static_assert(STAGES >= 2 && YOUNGER <= 63, "vmcnt is a 6-bit counter");
    static_assert(!BROW_ || (NH == 4 && DEPTH == 4 && TJ == 4 && WM % 64 == 0), "scale products of four sub-tiles at a time");
    static_assert(NS % 2 == 0 && NS >= 2, "the first streamed fragment of the next K block reuses queue slot 0");
    static_assert(TOUCH < TB, "not enough slots in front of the barrier");

    using L = TileLds<BM, BN, WAVES, STAGES, BROW_, CHUNKED_>;
    constexpr int NBS = L::NBS, PARTS = L::PARTS, PARTS_A = BM / 16 / WAVES, CHUNKS = L::CHUNKS, CHUNK = L::GROUPS * 64;      // (floats)
    // !CHUNKED_: waves that also copy 64 activation scales of the K block each, and behind them those that copy 64 weight rows' scales
    constexpr int S_WAVES = BM / 64, SB_WAVES = BROW_ && !CHUNKED_ ? BN / 64 : 0;
    constexpr bool NO_DUMMY = WALK && L::no_dummy;
    static_assert(CHUNKED_ ? BROW_ && BM / 16 % WAVES == 0 && PARTS <= 4 && BN / 16 % WAVES == 0 : S_WAVES + SB_WAVES <= WAVES,
                  "a part of a chunk is a group of 16 rows for every wave, a K block has one part");
    static_assert(!NO_DUMMY || L::GROUPS == 4 * WAVES, "every scale copy has a part to go to");
    uint8_t(*lds_a)[BM * 128] = reinterpret_cast<uint8_t(*)[BM * 128]>(pool + L::a_off);     // [STAGES]
    uint8_t(*lds_b)[BN * 128] = reinterpret_cast<uint8_t(*)[BN * 128]>(pool + L::b_off);     // [STAGES]
    const float* lds_s = reinterpret_cast<const float*>(pool + L::s_off);                     // [CHUNKS][GROUPS][16][4]; !CHUNKED_: [STAGES][BM]
    float(*lds_bs)[512] = reinterpret_cast<float(*)[512]>(pool + L::bs_off);                  // [NBS] weight scales, all K blocks

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const uint32_t dummy = lds_addr(pool + (NO_DUMMY ? L::rows_off : L::dummy_off)) + wave * (NO_DUMMY ? 2048 : 512);      // target of copies that must go nowhere
    const int M = m_end;
    const int KB = K >> 7;

    // ---- DMA.  What depends on the tile: the descriptors (limited to the rows of the tile, so that the M and N
    // tails read 0), its place, and the share of the panels this workgroup pre-touches.
    struct TileAddr {
        intx4 ra, rb, rt;
        int s_voff, touch_off, m0, n0;
    };
    const int prow = wave * 8 + (lane >> 3);                          // row inside a pass
    const int voff = prow * K + (((lane & 7) ^ swz(prow)) << 4);      // permuted chunk of that row
    // scale copies: lane -> row lane / 4 of the wave's group, K block lane % 4 of the chunk.  Rows beyond the matrix read what lies there, or
    // zeros beyond the array: nothing they scale is stored.
    const bool s_none = !CHUNKED_ && wave >= S_WAVES + SB_WAVES;      // this wave copies no scales: always out of range
    const bool sb_wave = SB_WAVES > 0 && wave >= S_WAVES && !s_none;
    const intx4 rsa = make_rsrc(a_s, s_none ? 0u : as_bytes), rsb = make_rsrc(BROW_ ? b_s : a_s, BROW_ ? bs_bytes : 0u);
    const int srow = wave * 16 + (lane >> 2);
    const auto scale_offset = [](int row, int rs, int kb, int cs) { return (int)(((uint32_t)row * (uint32_t)rs + (uint32_t)kb * (uint32_t)cs) * 4u); };
    const int sa_voff = scale_offset(srow, as_rs, lane & 3, as_cs), sb_voff = BROW_ ? scale_offset(srow, bs_rs, lane & 3, bs_cs) : 0;
    const uint32_t ls_base = s_none ? dummy : sb_wave ? lds_addr(pool + L::bs_off) + (wave - S_WAVES) * 256 : lds_addr(pool + L::s_off) + wave * 256;
    const uint32_t ls_buf = s_none ? 0 : sb_wave ? BN * 4 : BM * 4;
    const intx4 rs = sb_wave ? rsb : rsa;
    const int sc_cs = sb_wave ? bs_cs : as_cs;
    const uint32_t la_base = lds_addr(&lds_a[0][0]) + wave * 1024;
    const uint32_t lb_base = lds_addr(&lds_b[0][0]) + wave * 1024;
    // duty touch: the even waves load one dword of every line of this workgroup's share of the B panel (64
    // rows per wave), the odd waves of the A panel, TD K blocks ahead, into the dummy area: the lines are in L2
    // when this workgroup and its neighbours copy them.  Waves beyond the share run the same instruction on an
    // empty descriptor.
    const bool touch_b = (wave & 1) == 0;
    const int t_idx = (wave >> 1) * 64 + lane;
    auto tile_addr = [&](int tm0, int tn0, const Duty& d) {
        TileAddr t;
        t.ra = make_rsrc(a + (size_t)tm0 * K, (uint32_t)min(BM, M - tm0) * (uint32_t)K);
        t.rb = make_rsrc(b + (size_t)tn0 * K, (uint32_t)min(BN, N - tn0) * (uint32_t)K);
        const int share = touch_b ? (BN >> d.b_sh) : (BM >> d.a_sh);      // rows of the share
        t.rt = touch_b ? t.rb : t.ra;
        // nobody to share with: touching one's own lines ahead of the copy only adds requests (measured)
        if ((wave >> 1) * 64 >= share || (touch_b ? d.b_sh : d.a_sh) == 0) t.rt[2] = 0;
        t.touch_off = ((touch_b ? d.b_duty : d.a_duty) * share + t_idx % share) * K;
        t.s_voff = CHUNKED_ ? 0 : sb_wave ? min(tn0 + (wave - S_WAVES) * 64 + lane, N - 1) * bs_rs * 4
                                          : min(tm0 + (wave % S_WAVES) * 64 + lane, m_total - 1) * as_rs * 4;
        t.m0 = tm0;
        t.n0 = tn0;
        return t;
    };
    TileAddr me = tile_addr(m0, n0, duty);

    // copy i (0: scales, then the A passes, then the B passes) of K block kb into buffer buf.  Past the last K
    // block the offsets run beyond the descriptors: no memory access, zeros into a buffer nobody reads any more.
    auto scale_part = [&](const TileAddr& t, int part, int chunk, bool on) {
        const bool weight = BROW_ && part >= PARTS_A;
        const int rs = weight ? bs_rs : as_rs, cs = weight ? bs_cs : as_cs;
        const int row0 = weight ? t.n0 + (part - PARTS_A) * (WAVES * 16) : t.m0 + part * (WAVES * 16);
        const int slot = CHUNKS == 2 ? chunk & 1 : chunk % CHUNKS;
        dma4(weight ? rsb : rsa, weight ? sb_voff : sa_voff, on ? scale_offset(row0, rs, kb0 + 4 * chunk, cs) : (int)(weight ? bs_bytes : as_bytes),
             on || NO_DUMMY ? ls_base + slot * (CHUNK * 4) + part * (WAVES * 256) : dummy);
    };
    auto issue = [&](const TileAddr& t, int i, int kb, int buf) {
        const bool more = kb < kb1;
        if (i == 0 && !CHUNKED_) {
            dma4(rs, t.s_voff, more ? kb * sc_cs * 4 : (int)(sb_wave ? bs_bytes : as_bytes), ls_base + buf * ls_buf);
        } else if (i == 0) {
            const int u = kb - kb0 + PARTS - 1;
            scale_part(t, u & 3, u >> 2, more && (PARTS == 4 || (u & 3) < PARTS));
        } else if (i <= A_PASSES)
            dma16(t.ra, voff, (i - 1) * PASS_ROWS * K + (more ? kb * 128 : t.ra[2]), la_base + buf * (BM * 128) + (i - 1) * PASS_ROWS * 128);
        else
            dma16(t.rb, voff, (i - 1 - A_PASSES) * PASS_ROWS * K + (more ? kb * 128 : t.rb[2]),
                  lb_base + buf * (BN * 128) + (i - 1 - A_PASSES) * PASS_ROWS * 128);
    };
    // to: where the touch of a tile's start goes without a dummy area, while the last tile's results lie in the rows: a part of the second chunk that
    // this wave itself copies later (loads complete in order)
    const uint32_t touch_to = NO_DUMMY ? dummy : dummy + 256, first_touch_to = NO_DUMMY ? ls_base + CHUNK * 4 + (PARTS - 1) * (WAVES * 256) : touch_to;
    auto touch = [&](const TileAddr& t, int kb, uint32_t to) { dma4(t.rt, t.touch_off, kb < kb1 ? kb * 128 : t.rt[2], to); };
    // The start of a tile: its weight scales, then the copies in the order the K loop keeps up: for every K block its
    // first FIRST copies, the rest, one touch; K blocks 0 .. STAGES-2 whole and the first copies of block STAGES-1.
    auto prologue = [&](const TileAddr& t) {
        if (!BROW_ && wave < NBS) {
            const int nb = min((t.n0 >> 7) + wave, ((N + 127) >> 7) - 1);
            const intx4 rbs = make_rsrc(b_s + (size_t)nb * KB, (uint32_t)KB * 4u);
            for (int cc = 0; cc < KB; cc += 64) dma4(rbs, lane * 4, cc * 4, lds_addr(&lds_bs[wave][cc]));
        }
#pragma unroll
        for (int part = 0; part < (CHUNKED_ ? PARTS - 1 : 0); ++part) scale_part(t, part, 0, true);      // the first chunk; its last part comes with the first K block
#pragma unroll
        for (int blk = 0; blk < STAGES - 1; ++blk) {
#pragma unroll
            for (int i = 0; i < NDMA; ++i) issue(t, i, kb0 + blk, blk);
            if (!NO_TOUCH) touch(t, kb0 + blk + 1 + TD - STAGES, first_touch_to);
            else touch(t, 1 << 20, first_touch_to);      // same load count for the waits below: a copy of nothing
        }
#pragma unroll
        for (int i = 0; i < (WALK ? NDMA : FIRST); ++i) issue(t, i, kb0 + STAGES - 1, STAGES - 1);
        if (NO_COPY) {     // probe: the whole ring up front, nothing is copied later
#pragma unroll
            for (int i = FIRST; i < NDMA; ++i) issue(t, i, kb0 + STAGES - 1, STAGES - 1);
        }
    };

    // ---- fragment reads: lane -> row (lane%16) and the 32-byte K slice (lane/16) of a 16-row sub-tile
    const int frow = lane & 15, fk = lane >> 4;
    const int a_rd0 = (wm * WM + frow) * 128 + (((2 * fk) ^ swz(frow)) << 4);
    const int a_rd1 = (wm * WM + frow) * 128 + (((2 * fk + 1) ^ swz(frow)) << 4);
    const int b_rd0 = (wn * WN + frow) * 128 + (((2 * fk) ^ swz(frow)) << 4);
    const int b_rd1 = (wn * WN + frow) * 128 + (((2 * fk + 1) ^ swz(frow)) << 4);
    const int h0 = HOLD_A ? a_rd0 : b_rd0, h1 = HOLD_A ? a_rd1 : b_rd1;   // held operand
    const int x0 = HOLD_A ? b_rd0 : a_rd0, x1 = HOLD_A ? b_rd1 : a_rd1;   // streamed operand
    const int s_rd = wm * WM + frow;
    constexpr int S_STRIDE = CHUNKED_ ? 4 : 1;
    const int bs_col = (n0 & 127) + wn * WN;                        // first column of the wave inside the tile's first scale block
    const float* my_bs = lds_bs[bs_col >> 7];
    const float* my_bs_hi = lds_bs[(bs_col + WN - 1) >> 7];         // STRADDLE: the block of the wave's last columns
    const int jsplit = STRADDLE ? min(TJ, (128 - (bs_col & 127)) >> 4) : TJ;   // sub-tiles j < jsplit lie in the first block

    floatx4 acc[TI][TJ];

    auto read_frag = [&](const uint8_t* base, int rd0, int rd1, int idx) {
        const intx4 lo = *reinterpret_cast<const intx4*>(base + rd0 + idx * 2048);
        const intx4 hi = *reinterpret_cast<const intx4*>(base + rd1 + idx * 2048);
        return intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    constexpr int STORES = WALK ? TI * 2 : 0;        // store instructions of store_rows_beside
    static_assert(!WALK || (STAGES == 2 && TJ == 4 && sizeof(OUT) == 2 && EPI_ != kEpiDirect && ABL_ == 0 && 2 + NDMA + STORES <= 63),
                  "walking tiles: a ring of two, waves of 64 bf16 columns");
    bool stores_pending = false;                     // WALK: the last tile's stores are younger than this tile's first copies
    prologue(me);
    for (;;) {                                       // WALK: tile by tile; otherwise once
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // ---- wait for block 0, load the registers of step 0
    if (NO_COPY) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if (WALK && stores_pending) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(1 + NDMA + STORES) : "memory");
    else if (WALK) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(1 + NDMA) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 2) * (NDMA + 1) + 1 + FIRST) : "memory");
    __syncthreads();
    intx8 fh[NH], fx[2];
    float sc[TI], sc_hi[STRADDLE ? TI : 1];
    // BROW_: the scales of the wave's 64 weight rows and of its activation rows, one a lane
    constexpr int SAV = BROW_ ? TI / 4 : 1;
    const float* lds_sbr = reinterpret_cast<const float*>(pool + L::bs_off);      // !CHUNKED_: [STAGES][BN]
    const int sbr_lane = CHUNKED_ ? (BM + wn * WN + lane) * 4 : wn * WN + lane, sar_lane = (wm * WM + lane) * S_STRIDE;
    float sb_row = 1.0f, sa_row[SAV];
    if (BROW_) {
        sb_row = CHUNKED_ ? lds_s[sbr_lane] : lds_sbr[sbr_lane];
#pragma unroll
        for (int v = 0; v < SAV; ++v) sa_row[v] = lds_s[sar_lane + v * 64 * S_STRIDE];
    }
#pragma unroll
    for (int h = 0; h < NH; ++h) fh[h] = read_frag(HOLD_A ? lds_a[0] : lds_b[0], h0, h1, h);
    if (!BROW_) {
        const float sb = my_bs[kb0], sb_hi = my_bs_hi[kb0];
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const float sa = lds_s[s_rd + i * 16];
            sc[i] = sa * sb;
            if (STRADDLE) sc_hi[i] = sa * sb_hi;
        }
    }
    fx[0] = read_frag(HOLD_A ? lds_b[0] : lds_a[0], x0, x1, 0);

    int cur = 0;                                             // buffer of K block kb: kb % STAGES
    // FRESH (WALK, a tile's first K block): the copies of block kb+1 are all under way
    auto k_block = [&](int kb, auto fresh) __attribute__((always_inline)) {
        constexpr bool FRESH = decltype(fresh)::value;
        const int nxt = cur + 1 == STAGES ? 0 : cur + 1;     // buffer of K block kb+1
        const int last = cur == 0 ? STAGES - 1 : cur - 1;    // buffer of K block kb+STAGES-1
        const uint8_t* lx = HOLD_A ? lds_b[cur] : lds_a[cur];            // streamed operand of this K block
        const uint8_t* lh_n = HOLD_A ? lds_a[nxt] : lds_b[nxt];          // operands and scales of the next one
        const uint8_t* lx_n = HOLD_A ? lds_b[nxt] : lds_a[nxt];
        const int bn = kb + 1 - kb0, cn = bn >> 2;
        const float* ls_n = CHUNKED_ ? lds_s + (CHUNKS == 2 ? cn & 1 : cn % CHUNKS) * CHUNK + (bn & 3) : lds_s + nxt * BM;
        float sa_n[TI], sb_n = 1.0f, sb_hi_n = 1.0f;         // scales of the next K block
        floatx4 p[DEPTH + 1];
        floatx16 sp;                                         // BROW_: scale products of the streamed fragment that is folded
#pragma unroll
        for (int t = 0; t < NT + DEPTH; ++t) {
            if (t < NT) {
                const int si = t / NH, h = t % NH;
                if (h == 0 && si + 1 < NS) {
                    if (!NO_LDS) fx[(si + 1) & 1] = read_frag(lx, x0, x1, si + 1);
                    else asm volatile("" : "+v"(fx[(si + 1) & 1]));      // probe: keep the operand opaque to the optimizer
                }
                const intx8 fa_ = HOLD_A ? fh[h] : fx[si & 1];
                const intx8 fb_ = HOLD_A ? fx[si & 1] : fh[h];
                if (!NO_FOLD) {
                    p[t % (DEPTH + 1)] = mfma_block<FMT_>(fb_, fa_);
                } else {
                    floatx4& d = acc[HOLD_A ? h : si][HOLD_A ? si : h];
                    d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb_, fa_, d, FMT_, FMT_, 0, 0, 0, 0);
                }
                if (t == TB) {
                    // K block kb+1 has landed once only the younger loads are left in flight
                    if (FRESH && stores_pending) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER + STORES) : "memory");
                    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
                    __syncthreads();
                    if (!NO_LDS) {
                        fx[0] = read_frag(lx_n, x0, x1, 0);      // queue slot 0 was last used by streamed fragment NS-2
                        if (!BROW_) {
                            sb_n = my_bs[min(kb + 1, KB - 1)];
                            sb_hi_n = my_bs_hi[min(kb + 1, KB - 1)];
#pragma unroll
                            for (int i = 0; i < TI; ++i) sa_n[i] = ls_n[s_rd + i * 16];      // combined at the end of the block: nothing waits here
                        }
                    } else {
                        asm volatile("" : "+v"(fx[0]));
                    }
                }
                if (t >= TB) {
                    if (!NO_LDS) fh[h] = read_frag(lh_n, h0, h1, h);   // fh[h] had its last use just above
                    else asm volatile("" : "+v"(fh[h]));
                }
            }
            if (t >= DEPTH && !NO_FOLD) {
                const int u = t - DEPTH, si = u / NH, h = u % NH;
                const int i = HOLD_A ? h : si, j = HOLD_A ? si : h;
                const floatx4 q = p[u % (DEPTH + 1)];
                if (BROW_) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(q[e], sp[h * 4 + e], acc[i][j][e]);
                } else {
                    fold(acc[i][j], q, (STRADDLE && j >= jsplit) ? sc_hi[i] : sc[i]);
                }
                if (FRESH) asm volatile("" : "+v"(acc[i][j]));      // here, not behind the branch around the wait below
            }
            if (BROW_ && t < NT && t % NH == NH - 1) {
                // the fragment before has just been folded: its products make room
                constexpr bool W = !HOLD_A;
                const int si = t / NH;
                const float sa = sa_row[W ? si / 4 : 0];
                sp = si % 4 == 0 ? scale_products<W, 0>(sb_row, sa) : si % 4 == 1 ? scale_products<W, 1>(sb_row, sa)
                     : si % 4 == 2 ? scale_products<W, 2>(sb_row, sa) : scale_products<W, 3>(sb_row, sa);
            }
            if (!NO_COPY) {
#pragma unroll
                for (int j = 0; j < NDMA; ++j) {
                    const int v = TB + 1 + GAP * j;
                    if (v < NSLOT && v == t) issue(me, j, kb + STAGES, cur);                    // behind the barrier: buffer cur is free
                    if (!FRESH && v >= NSLOT && v - NSLOT == t) issue(me, j, kb + STAGES - 1, last);      // the rest of the block started in kb-1
                }
            }
            if (t == TOUCH && !NO_TOUCH) touch(me, kb + TD, touch_to);
            if (BROW_ && t == NT + DEPTH - 1) {
                sb_row = CHUNKED_ ? ls_n[sbr_lane] : lds_sbr[nxt * BN + sbr_lane];      // first used NH - 1 MFMAs from here
#pragma unroll
                for (int v = 0; v < SAV; ++v) sa_row[v] = ls_n[sar_lane + v * 64 * S_STRIDE];
            }
            __builtin_amdgcn_sched_barrier(0);  // keep the MFMA / FMA / ds_read / copy interleaving as written
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            if (NO_LDS || BROW_) continue;
            sc[i] = sa_n[i] * sb_n;
            if (STRADDLE) sc_hi[i] = sa_n[i] * sb_hi_n;
        }
        cur = nxt;
    };
    int kb_first = kb0;
    if constexpr (WALK) k_block(kb_first++, std::true_type{});
    for (int kb = kb_first; kb < kb1; ++kb) k_block(kb, std::false_type{});
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing may still be writing LDS when the wave ends

    // ---- epilogue: lane holds c[m][n..n+3], m = .. + lane%16, n = .. + 4*(lane/16)
    if constexpr (WALK) {
        __syncthreads();                               // every wave has left the ring
        const int m_done = m0, n_done = n0;
        const bool more = next(m0, n0, duty);
        if (more) {
            me = tile_addr(m0, n0, duty);
            prologue(me);
        }
        store_rows_beside<TI, EPI_ == kEpiLines>(acc, pool + L::rows_off + wave * 2048, c, ldc, bias, m_done, wm * WM, n_done + wn * WN, M, BM, N, lane);
        stores_pending = true;
        if (!more) return;
        continue;
    }
    if constexpr (EPI_ != kEpiDirect) {
        static_assert(WAVES * WM * WN * (int)sizeof(OUT) <= L::bytes, "the tile's results fit the pool");
        __syncthreads();                               // every wave's copies have landed: the pool is free
        store_rows<TI, TJ, OUT, EPI_ == kEpiLines>(acc, pool + wave * (WM * WN * (int)sizeof(OUT)), c, ldc, bias, m0 + wm * WM, n0 + wn * WN, M, N,
                                                   lane);
        return;
    }
    const bool vec_ok = (ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(c) & 15) == 0);
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int m = m0 + wm * WM + i * 16 + frow;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int n = n0 + wn * WN + j * 16 + 4 * fk;
            float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if (bias.p != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) v[e] = bias.add(v[e], n + e);
            }
            store4<OUT>(c, ldc, m, n, M, N, v, vec_ok);
        }
    }
    break;
    }
}

// Tile order shared by the kernels below: consecutive workgroup ids land on different XCDs (8 of
// them); give each XCD a contiguous run of tiles, walked in groups of 4 tile rows.  With a tile count that 8 does not divide the
// first XCDs get one tile more (such counts used to run in plain order, every panel pulled into every XCD's L2): 777x2112x7168
// 29.9 -> 28.3 us, 777x7168x7168 62.5 -> 57.2, 250x9000x2048 14.7 -> 13.3, 3752x15224x768 68.8 -> 65.6 (out of the caches 73.2 -> 76.4).  Up to 3
// K blocks it is even (tiles in one launch: 0.94 to 1.07 of the time).
__device__ __forceinline__ int xcd_contiguous(int pid, int ntiles) {
    const int x = pid & 7, rest = ntiles & 7;
    return x * (ntiles >> 3) + min(x, rest) + (pid >> 3);
}
// The same for (slab, tile) pairs of a call cut along K, where a count that 8 does not divide stays in plain order with short slabs: in
// runs, all workgroups of an XCD start on the same few panels, and a slab of few K blocks ends before their sharing pays.
__device__ __forceinline__ int slab_order(int pid, int n, bool runs) { return (n & 7) != 0 && !runs ? pid : xcd_contiguous(pid, n); }
// GM: tile rows per group; the 32 workgroups that an XCD runs at a time then cover a GM x (32 / GM) block of tiles
// (4 x 8 in the product; the probe library also builds 2 x 16 and 8 x 4 to measure their fabric traffic and energy).
template <int GM = 4>
__device__ __forceinline__ Duty tile_of(int local, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int group = local / (GM * tiles_n);
    const int first_m = group * GM;
    const int gsz = min(tiles_m - first_m, GM);
    const int in_group = (local % (GM * tiles_n)) % gsz;
    tm = first_m + in_group;
    tn = (local % (GM * tiles_n)) / gsz;
    // the workgroups of an XCD run a gsz x (up to 32 / GM) block of tiles at a time
    Duty d;
    d.b_sh = gsz >= 8 ? 3 : gsz >= 4 ? 2 : gsz >= 2 ? 1 : 0;
    constexpr int COLS = 32 / GM;
    d.a_sh = (tiles_n >= 16 && COLS >= 16) ? 4 : (tiles_n >= 8 && COLS >= 8) ? 3 : (tiles_n >= 4 && COLS >= 4) ? 2 : tiles_n >= 2 ? 1 : 0;
    d.b_duty = in_group & ((1 << d.b_sh) - 1);
    d.a_duty = tn & ((1 << d.a_sh) - 1);
    return d;
}

// The tile with SPECIALIZED waves and the barrier of a K block EARLY in the block, for small wave tiles.
// In fp8_gemm_tile every wave copies, reads fragments, issues MFMAs and folds, and the one barrier of a K block sits in
// front of its last streamed fragment: behind it every wave reloads the held fragments, the first streamed fragment and the
// scales of the next block from LDS with only NH MFMAs left to cover that latency, and every buffer_load ... lds stays at
// the head of its (in-order) wave until the CU's address unit takes it, holding back the MFMAs queued behind it.  With a
// 256x256 tile both are a small part of a K block; with 64x96 wave tiles on a 128x192 tile, in-kernel clocks at
// 4096x1536x7168 showed 560-730 of ~1700 clocks per K block behind the barrier for 4 of 12 MFMAs, 40 clocks per MFMA slot
// without a copy near it and 60 with one every second slot.  Here:
//   * the first WGM x WGN waves ("consumers") run the MFMAs, the LDS reads and the fold and never touch global memory in the
//     K loop; PW further waves ("producers") do nothing but the global->LDS copies and the pre-touches (small wave tiles
//     leave registers for the second set of waves: all waves of a workgroup get the same allocation);
//   * the barrier of block kb is at slot E, a few MFMAs into the block.  For a consumer it says "I have left block kb-1";
//     a producer first waits for its own copies of block kb+1.  Behind it the consumers read block kb+1's held fragments,
//     first streamed fragment and scales from LDS into a SECOND set of registers, spread over the slots (block kb+1 then
//     starts on registers loaded a dozen slots earlier; an even number of unrolled blocks lets the sets swap without
//     moves), and the producers copy block kb+3 and touch the lines of a later block;
//   * the held operand of block kb is read during block kb-1, the streamed operand during block kb itself: the held
//     operand's buffer is free one block earlier, and a ring of 3 serves it where the streamed operand needs 4 (WsRings);
//   * on the 192-wide tile a wave's columns can straddle two 128-column blocks of weight scales: the combined scale is
//     kept per row and 32-column group (multiplies once per block instead of a select per MFMA);
//   * a consumer alone on its SIMD is bound by the issue of its instructions: an MFMA holds the wave for 16 clocks and any other instruction,
//     scalar ones too, for 4, so with the 4 FMAs of the fold (16 + 16 of the MFMA's 32 clocks) nothing is free.  A K block of 64x64 needs 512 + 64 for
//     its 16 LDS reads; ring positions, addresses and scales used to take 160 more and waits another 100.  Unrolled by 4 K blocks, with rings of 4, the
//     addresses of the buffers are constants in the LDS instructions, and a lane's scales of the next 4 K blocks come as one read per row, 16 bytes:
//     838 -> 690 clocks a K block (64 tiles of 128x128; 861 -> 755 with 256, which also wait for copies).  With the chunks of scales below, rotating
//     operands: 4096x1536x7168 47.7 -> 45.1 us, 2048x2048x16384 74.1 -> 67.7, 900x4096x9216 44.5 -> 40.1, 700x7168x7168 45.4 -> 41.7,
//     1300x4096x4096 29.2 -> 27.1, 200x7168x2048 10.0 -> 9.5, 1000x1090x1664 10.3 -> 9.9, 777x2112x7168 24.6 -> 24.4.
// Swizzle, fragment layout, fold, epilogue and pre-touch shares are fp8_gemm_tile's.
// The activation scales come in chunks of 4 K blocks, 16 rows x 4 K blocks a copy, the first three with the tile's start and one more with every 4th
// K block: with row-major scales, the official dialect's, 64 rows of one K block at a time are 64 lines of 4 bytes for 128 of panels.  What row-major
// scales take over column-major ones, a K block at a time and the longer loop -> now: 1024x4096x7168 41.5 / 37.0 -> 36.6 / 36.2 us, 2048x2048x7168 40.1 / 36.7
// -> 36.2 / 35.6, 300x7168x4096 24.4 / 21.8 -> 21.7 / 21.5, 128x7168x7168 23.4 / 21.7 -> 21.3 / 21.3, 200x7168x2048 11.5 / 10.9 -> 10.5 / 10.4, 4096x1536x7168
// 51.5 / 48.8 -> 49.1 / 48.3 (out of the caches).
template <int BM, int BN, typename OUT, int FMT_ = 0, int EPI_ = kEpiDirect>
__device__ __forceinline__ void fp8_gemm_tile_ws(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, OUT* __restrict__ c,
    const Bias bias, int m0, int m_end, int m_total, int n0, int N, int K, int ldc, const Duty duty,
    int kb0, int kb1, uint8_t* __restrict__ pool) {
    constexpr int WGM = 2, WGN = 2, PW = 4;
    constexpr int CW = WGM * WGN;                       // consumer waves
    constexpr int WM = BM / WGM, WN = BN / WGN, TI = WM / 16, TJ = WN / 16;
    constexpr int PASS_ROWS = PW * 8;                   // rows copied by one instruction of every producer
    constexpr int A_PASSES = BM / PASS_ROWS, B_PASSES = BN / PASS_ROWS;
    constexpr int DEPTH = 4;
    static_assert(BM % PASS_ROWS == 0 && BN % PASS_ROWS == 0 && PASS_ROWS % 16 == 0, "tile/threads mismatch");
    constexpr bool STRADDLE = (128 % WN) != 0;
    static_assert(WN <= 128 && (!STRADDLE || BN == 192), "weight-scale blocks per wave column");
    using R = WsRings<BM, BN>;
    constexpr bool HOLD_A = R::HOLD_A;
    constexpr int NH = HOLD_A ? TI : TJ, NS = HOLD_A ? TJ : TI;
    constexpr int NT = TI * TJ;
    constexpr int NDMA = A_PASSES + B_PASSES;           // panel copies per K block and producer
    constexpr int E = 2;                                // slot of the barrier
    constexpr int TDA = 2;
    constexpr int SA = R::SA, SB = R::SB, STREAM = R::STREAM, HOLD = R::HOLD;
    // A K block's panels go out this many blocks ahead: behind the barrier of a block, the streamed operand of the one before is free and the held
    // operand of the block itself.
    constexpr int AHEAD = 3;
    static_assert(STREAM == 4 && HOLD >= AHEAD && (AHEAD - 1) * (NDMA + 1) + 1 <= 63, "two K blocks in flight; vmcnt is a 6-bit counter");
    // loads younger than the last copy of block kb+1 at the barrier of block kb: the touch behind those copies and the
    // copies + touches of blocks kb+2 .. kb+AHEAD-1 (and chunks of scales, for which a wait may then wait as well)
    constexpr int YOUNGER = (AHEAD - 2) * (NDMA + 1) + 1;
    // streamed fragments are read PF in front of the one in use, at least 4 MFMAs
    constexpr int PF = NH >= 4 ? 1 : 2, FX = NH >= 4 ? 2 : 4;
    static_assert(NS % FX == 0 && NH * (NS - PF) > E && DEPTH <= NT, "the next K block's first fragments are read behind the barrier");
    constexpr int PWIN = NT - 2 - (E + 1);
    static_assert(E >= 0 && E < NT - NH && PWIN >= NH, "barrier slot");

    using L = typename R::L;
    constexpr int RG = BM / 16 / PW;                    // groups of 16 rows per producer in a chunk of scales
    static_assert(L::bytes <= 160 * 1024 && (BM / 16) % PW == 0, "LDS of a CU; groups of 16 rows per producer");
    constexpr int NBS = L::NBS;
    uint8_t(*lds_a)[BM * 128] = reinterpret_cast<uint8_t(*)[BM * 128]>(pool + L::a_off);
    uint8_t(*lds_b)[BN * 128] = reinterpret_cast<uint8_t(*)[BN * 128]>(pool + L::b_off);
    const float* lds_s = reinterpret_cast<const float*>(pool + L::s_off);                       // [chunk % kScaleChunks][row][K block % 4]
    float(*lds_bs)[L::BSROW] = reinterpret_cast<float(*)[L::BSROW]>(pool + L::bs_off);          // of the tile's K blocks, from kb0 on

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = m_end;
    const int KB = K >> 7;

    constexpr bool through_lds = EPI_ != kEpiDirect;
    static_assert(!through_lds || CW * WM * WN * (int)sizeof(OUT) <= L::bytes, "the tile's results fit the pool");
    if (wave >= CW) {
        // ------------------------------------------------------------------ producer
        const int pw = wave - CW;
        const int prow = pw * 8 + (lane >> 3);
        const int voff = prow * K + (((lane & 7) ^ swz(prow)) << 4);
        const uint32_t pool_addr = lds_addr(pool), ld_base = pool_addr + L::dummy_off + wave * 512;
        const uint32_t la_base = pool_addr + L::a_off + pw * 1024;
        const uint32_t lb_base = pool_addr + L::b_off + pw * 1024;
        const intx4 ra = make_rsrc(a + (size_t)m0 * K, (uint32_t)min(BM, M - m0) * (uint32_t)K);
        const intx4 rb = make_rsrc(b + (size_t)n0 * K, (uint32_t)min(BN, N - n0) * (uint32_t)K);
        const bool touch_b = (pw & 1) == 0;
        const int t_idx = (pw >> 1) * 64 + lane;
        const int share = touch_b ? (BN >> duty.b_sh) : (BM >> duty.a_sh);
        intx4 rt = touch_b ? rb : ra;
        if ((touch_b ? duty.b_sh : duty.a_sh) == 0) rt[2] = 0;
        const int touch_row0 = (touch_b ? duty.b_duty : duty.a_duty) * share;
        constexpr int TOUCH_LANES = (PW / 2) * 64;
        auto issue = [&](int i, int kb, int bufa, int bufb) {
            const bool more = kb < kb1;
            if (i < A_PASSES)
                dma16(ra, voff, i * PASS_ROWS * K + (more ? kb * 128 : ra[2]), la_base + bufa * (BM * 128) + i * PASS_ROWS * 128);
            else
                dma16(rb, voff, (i - A_PASSES) * PASS_ROWS * K + (more ? kb * 128 : rb[2]), lb_base + bufb * (BN * 128) + (i - A_PASSES) * PASS_ROWS * 128);
        };
        auto touch = [&](int kbp) {      // kTouchBurst consecutive lines of a row at a time (see kTouchBurst)
            const int j = kbp & (kTouchBurst - 1), base = kbp - j;
            const int q = j * TOUCH_LANES + t_idx, row = q >> kTouchBurstLog, line = q & (kTouchBurst - 1);
            const bool ok = row < share && base + line < kb1;
            dma4(rt, ok ? (touch_row0 + row) * K + (base + line) * 128 : kOutOfRange, 0, ld_base + 256);
        };
        // scales of K blocks kb0 + 4 * chunk ..: rows beyond the matrix read its last one's, K blocks beyond it what lies there or zeros; nothing uses them
        const intx4 rs = make_rsrc(a_s, as_bytes);
        int s_voff[RG];
#pragma unroll
        for (int r = 0; r < RG; ++r) s_voff[r] = (min(m0 + (r * PW + pw) * 16 + (lane >> 2), m_total - 1) * as_rs + (kb0 + (lane & 3)) * as_cs) * 4;
        auto scales = [&](int chunk) {
#pragma unroll
            for (int r = 0; r < RG; ++r)
                dma4(rs, s_voff[r], chunk * 16 * as_cs, pool_addr + L::s_off + (chunk & (kScaleChunks - 1)) * (BM * 16) + (r * PW + pw) * 256);
        };
        const int chunks = (kb1 - kb0 + 3) >> 2;

        if (pw < NBS) {
            const int nb = min((n0 >> 7) + pw, ((N + 127) >> 7) - 1);
            const intx4 rbs = make_rsrc(b_s + (size_t)nb * KB, (uint32_t)KB * 4u);
            for (int cc = 0; cc < kb1 - kb0; cc += 64) dma4(rbs, lane * 4, (kb0 + cc) * 4, pool_addr + L::bs_off + (pw * L::BSROW + cc) * 4);
        }
        for (int q = 0; q < min(chunks, kScaleChunks - 1); ++q) scales(q);
#pragma unroll
        for (int blk = 0; blk < AHEAD; ++blk) {
#pragma unroll
            for (int i = 0; i < NDMA; ++i) issue(i, kb0 + blk, blk % SA, blk % SB);
            touch(kb0 + blk);                  // groups 0 .. AHEAD-1 of the first burst
        }
        // the loop's first touch is of block kb0 + AHEAD + TDA: the blocks in between are touched here, behind the copies,
        // so that the waits below only wait for more than they need (4096x1536x7168 after a cache flush 57.4 -> 56.1 us,
        // 2048x2048x7168 44.0 -> 43.0 us, 2048x1024x7168 34.6 -> 33.5 us)
#pragma unroll
        for (int t = 0; t < TDA; ++t) touch(kb0 + AHEAD + t);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * (NDMA + 1) + 1) : "memory");    // block kb0 has landed
        __syncthreads();
        int fa = AHEAD % SA, fb = AHEAD % SB;      // buffers of block kb + AHEAD
        for (int kb = kb0; kb < kb1; ++kb) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");   // this wave's copies of block kb+1 have landed
            __syncthreads();                                                   // every consumer has left block kb-1
            if (((kb - kb0) & 3) == 0) {      // every consumer has read the chunk before this block's: it makes room
                const int next = ((kb - kb0) >> 2) + kScaleChunks - 1;
                if (next < chunks) scales(next);
            }
#pragma unroll
            for (int i = 0; i < NDMA; ++i) issue(i, kb + AHEAD, fa, fb);
            touch(kb + AHEAD + TDA);
            fa = fa + 1 == SA ? 0 : fa + 1;
            fb = fb + 1 == SB ? 0 : fb + 1;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing may still be writing LDS when the wave ends
        if (through_lds) __syncthreads();                  // the consumers' epilogue goes through the pool
        return;
    }

    // ---------------------------------------------------------------------- consumer
    const int wm = wave / WGN, wn = wave % WGN;
    const int frow = lane & 15, fk = lane >> 4;
    const int a_rd0 = (wm * WM + frow) * 128 + (((2 * fk) ^ swz(frow)) << 4);
    const int a_rd1 = (wm * WM + frow) * 128 + (((2 * fk + 1) ^ swz(frow)) << 4);
    const int b_rd0 = (wn * WN + frow) * 128 + (((2 * fk) ^ swz(frow)) << 4);
    const int b_rd1 = (wn * WN + frow) * 128 + (((2 * fk + 1) ^ swz(frow)) << 4);
    const int h0 = HOLD_A ? a_rd0 : b_rd0, h1 = HOLD_A ? a_rd1 : b_rd1;
    const int x0 = HOLD_A ? b_rd0 : a_rd0, x1 = HOLD_A ? b_rd1 : a_rd1;
    const int bs_col = (n0 & 127) + wn * WN;
    // A wave's columns lie in one 128-column block of weight scales, except on the 192-wide tile (WN = 96): there
    // every group of GW columns does (GW = 32 divides the possible offsets), so the combined scale is kept per row
    // and column group: NG multiplies per row and K block instead of one select per MFMA.
    constexpr int GW = STRADDLE ? ((WN % 32 == 0) ? 32 : 16) : WN, NG = WN / GW, JPG = GW / 16;
    const float* my_bs[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) my_bs[g] = lds_bs[(bs_col + g * GW) >> 7];

    floatx4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto read_frag = [&](const uint8_t* base, int rd0, int rd1, int idx) {
        const intx4 lo = *reinterpret_cast<const intx4*>(base + rd0 + idx * 2048);
        const intx4 hi = *reinterpret_cast<const intx4*>(base + rd1 + idx * 2048);
        return intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    // Scales of the next K block(s): a chunk's in one read per row where registers allow (not with the 24 sub-tiles of 128x192), else a K block's.
    constexpr bool BY_CHUNK = NT <= 16;
    constexpr int SV = BY_CHUNK ? 4 : 1;
    typedef float scale_t __attribute__((ext_vector_type(SV)));
    scale_t sa_n[TI], sb_n[NG];
    auto read_scales = [&](int chunk, int at) {
        const float* p = lds_s + (chunk & (kScaleChunks - 1)) * (BM * 4) + (wm * WM + frow) * 4 + (BY_CHUNK ? 0 : at);
#pragma unroll
        for (int i = 0; i < TI; ++i) sa_n[i] = *reinterpret_cast<const scale_t*>(p + i * 64);
#pragma unroll
        for (int g = 0; g < NG; ++g) sb_n[g] = *reinterpret_cast<const scale_t*>(my_bs[g] + 4 * chunk + (BY_CHUNK ? 0 : at));
    };
    auto combine = [&](float(&sc)[TI][NG], int at) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int g = 0; g < NG; ++g) sc[i][g] = sa_n[i][BY_CHUNK ? at : 0] * sb_n[g][BY_CHUNK ? at : 0];
    };

    __syncthreads();                                     // block kb0, the first scales have landed
    intx8 fh_a[NH], fh_b[NH], fx[FX];
    float sc_a[TI][NG], sc_b[TI][NG];
#pragma unroll
    for (int h = 0; h < NH; ++h) fh_a[h] = read_frag(HOLD_A ? lds_a[0] : lds_b[0], h0, h1, h);
    read_scales(0, 0);
    combine(sc_a, 0);
#pragma unroll
    for (int f = 0; f < PF; ++f) fx[f] = read_frag(HOLD_A ? lds_b[0] : lds_a[0], x0, x1, f);

    // K block kb0 + 4 * chunk + AT, in buffer AT of a ring of 4; ch: its buffer in a held ring of 3
    int ch = 0, chunk = 0;
    auto block = [&](auto at_, intx8(&fh)[NH], intx8(&fhn)[NH], float(&sc)[TI][NG], float(&scn)[TI][NG]) __attribute__((always_inline)) {
        constexpr int AT = decltype(at_)::value, NEXT = (AT + 1) & 3;
        const int nh = HOLD == 4 ? NEXT : ch + 1 == HOLD ? 0 : ch + 1;      // block kb+1, held ring
        const uint8_t* lx = HOLD_A ? lds_b[AT] : lds_a[AT];
        const uint8_t* lh_n = HOLD_A ? lds_a[nh] : lds_b[nh];
        const uint8_t* lx_n = HOLD_A ? lds_b[NEXT] : lds_a[NEXT];
        floatx4 p[DEPTH + 1];
#pragma unroll
        for (int t = 0; t < NT + DEPTH; ++t) {
            if (t < NT) {
                const int si = t / NH, h = t % NH;
                const intx8 fa_ = HOLD_A ? fh[h] : fx[si % FX];
                const intx8 fb_ = HOLD_A ? fx[si % FX] : fh[h];
                p[t % (DEPTH + 1)] = mfma_block<FMT_>(fb_, fa_);
                if (t == E) __syncthreads();
                if (h == 0) fx[(si + PF) % FX] = si + PF < NS ? read_frag(lx, x0, x1, si + PF) : read_frag(lx_n, x0, x1, si + PF - NS);
                if (t == E + 1 && (!BY_CHUNK || AT == 3)) read_scales(AT == 3 ? chunk + 1 : chunk, NEXT);
#pragma unroll
                for (int hh = 0; hh < NH; ++hh)
                    if (t == E + 1 + (hh * PWIN) / NH) fhn[hh] = read_frag(lh_n, h0, h1, hh);
            }
            if (t >= DEPTH) {
                const int u = t - DEPTH, si = u / NH, h = u % NH;
                const int i = HOLD_A ? h : si, j = HOLD_A ? si : h;
                fold(acc[i][j], p[u % (DEPTH + 1)], sc[i][j / JPG]);
            }
            if (t == NT + DEPTH - 1) combine(scn, NEXT);
            __builtin_amdgcn_sched_barrier(0);
        }
        ch = nh;
    };
    {
        constexpr std::integral_constant<int, 0> k0{};
        constexpr std::integral_constant<int, 1> k1{};
        constexpr std::integral_constant<int, 2> k2{};
        constexpr std::integral_constant<int, 3> k3{};
        int left = kb1 - kb0;
        for (; left >= 4; left -= 4) {
            block(k0, fh_a, fh_b, sc_a, sc_b);
            block(k1, fh_b, fh_a, sc_b, sc_a);
            block(k2, fh_a, fh_b, sc_a, sc_b);
            block(k3, fh_b, fh_a, sc_b, sc_a);
            ++chunk;
        }
        if (left > 0) block(k0, fh_a, fh_b, sc_a, sc_b);
        if (left > 1) block(k1, fh_b, fh_a, sc_b, sc_a);
        if (left > 2) block(k2, fh_a, fh_b, sc_a, sc_b);
    }

    if constexpr (through_lds) {
        __syncthreads();                                 // the producers' copies have landed, every consumer has left the K loop
        store_rows<TI, TJ, OUT, EPI_ == kEpiLines>(acc, pool + wave * (WM * WN * (int)sizeof(OUT)), c, ldc, bias, m0 + wm * WM, n0 + wn * WN, M, N, lane);
        return;
    }
    const bool vec_ok = (ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(c) & 15) == 0);
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int m = m0 + wm * WM + i * 16 + frow;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int n = n0 + wn * WN + j * 16 + 4 * fk;
            float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            if (bias.p != nullptr) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) v[e] = bias.add(v[e], n + e);
            }
            store4<OUT>(c, ldc, m, n, M, N, v, vec_ok);
        }
    }
}

// the wave-specialized tile as a kernel: one workgroup of 4 + 4 waves per tile (or per several, walked in turn)
template <int BM, int BN, typename OUT, int FMT_ = 0, int EPI_ = kEpiDirect>
__global__ __launch_bounds__(512) void fp8_gemm_ws_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, OUT* __restrict__ c,
    const Bias bias, int M, int N, int K, int ldc, int tiles_m, int tiles_n, int pretouch) {
    __shared__ __attribute__((aligned(1024))) uint8_t pool[WsRings<BM, BN>::L::bytes];
    const int ntiles = tiles_m * tiles_n;
    for (int pid = blockIdx.x; pid < ntiles; pid += gridDim.x) {
        int tm, tn;
        Duty duty = tile_of(xcd_contiguous(pid, ntiles), tiles_m, tiles_n, tm, tn);
        if (!pretouch) duty.a_sh = duty.b_sh = 0;
        fp8_gemm_tile_ws<BM, BN, OUT, FMT_, EPI_>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, c, bias, tm * BM, M, M, tn * BN, N, K, ldc, duty, 0, K >> 7, pool);
        __syncthreads();
    }
}

// Tiles blockIdx.x, blockIdx.x + gridDim.x, ... of a launch: the `next` of fp8_gemm_tile.
template <int GM = 4>
struct Walk {
    int pid, ntiles, tiles_m, tiles_n, bm, bn, pretouch;
    __device__ __forceinline__ bool operator()(int& m0, int& n0, Duty& duty) {
        if (pid >= ntiles) return false;
        int tm, tn;
        duty = tile_of<GM>(xcd_contiguous(pid, ntiles), tiles_m, tiles_n, tm, tn);
        if (!pretouch) duty.a_sh = duty.b_sh = 0;
        m0 = tm * bm;
        n0 = tn * bn;
        pid += gridDim.x;
        return true;
    }
};
// Kernels whose workgroups walk their tiles with the next tile's copies in front of the results: 256x256 tiles of bf16 results in
// whole rows.
constexpr bool walks(int BM, int BN, int STAGES, int esz, int EPI) { return BM == 256 && BN == 256 && STAGES == 2 && esz == 2 && EPI != kEpiDirect; }

template <int BM, int BN, int WGM, int WGN, int STAGES, typename OUT, int GAP_ = 0, int TD_ = 0, int ABL_ = 0, int FMT_ = 0, int GM_ = 4,
          int EPI_ = kEpiDirect>
__global__ __launch_bounds__(WGM* WGN * 64) void fp8_gemm_mfma_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, OUT* __restrict__ c,
    const Bias bias, int M, int N, int K, int ldc, int tiles_m, int tiles_n, int pretouch) {
    // The grid may be smaller than the number of tiles (one workgroup per CU for the 256x256 tile): a workgroup
    // then walks tiles blockIdx.x, blockIdx.x + gridDim.x, ... itself, which saves the ~4.5 us that pass between
    // the end of a workgroup and the start of its successor on the same CU.  Workgroup ids keep their XCD
    // (id % 8) from tile to tile when gridDim.x is a multiple of 8.
    using L = TileLds<BM, BN, WGM * WGN, STAGES>;
    constexpr bool WALK = walks(BM, BN, STAGES, (int)sizeof(OUT), EPI_) && ABL_ == 0;
    __shared__ __attribute__((aligned(1024))) uint8_t pool[WALK ? L::walk_bytes : L::bytes];
    const int ntiles = tiles_m * tiles_n;
    if constexpr (WALK) {
        Walk<GM_> walk{(int)blockIdx.x, ntiles, tiles_m, tiles_n, BM, BN, pretouch};
        int m0, n0;
        Duty duty;
        if (!walk(m0, n0, duty)) return;
        fp8_gemm_tile<BM, BN, WGM, WGN, STAGES, OUT, GAP_, TD_, ABL_, FMT_, false, EPI_>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, c, bias, m0, M, M, n0,
                                                                                         N, K, ldc, duty, 0, K >> 7, pool, 0, 0, 0, walk);
        return;
    }
    for (int pid = blockIdx.x; pid < ntiles; pid += gridDim.x) {
        int tm, tn;
        Duty duty = tile_of<GM_>(xcd_contiguous(pid, ntiles), tiles_m, tiles_n, tm, tn);
        if (!pretouch) duty.a_sh = duty.b_sh = 0;
        fp8_gemm_tile<BM, BN, WGM, WGN, STAGES, OUT, GAP_, TD_, ABL_, FMT_, false, EPI_>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, c, bias, tm * BM, M,
                                                                            M, tn * BN, N, K, ldc, duty, 0, K >> 7, pool);
        __syncthreads();   // every wave has left the tile's LDS buffers before the next tile's copies land in them
    }
}

}  // namespace mdy
