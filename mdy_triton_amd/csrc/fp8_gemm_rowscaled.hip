// Block-scaled FP8 GEMM, NT layout, with 1x128 scales on BOTH operands:
//   c[m,n] = sum_kb (sum_{k in kb} a[m,k] b[n,k]) * a_s[m,kb] * b_s[n,kb]
//
// Restates the have_w=False branch of _fp8_matmul_kernel
// (/root/reference/triton_kernels/deepseekv3/fp8_kernel.py:190-205; launcher fp8_matmul :214-252), which the
// reference's Fp8Linear uses for its weight gradient dw = dy^T . x with both operands quantized along the token
// dimension (fp8_matmul_bwd, :254-257).
//
// The combined scale differs for each of a lane's four results of an MFMA (four consecutive n of one m).  Multiplied on the VALU the
// fold would be 4 multiplies + 4 FMAs per MFMA instead of 4 FMAs, as much work as the matrix cores have; the scheduled tile body of fp8_gemm_tile.h
// forms the products on the matrix cores instead (scale_products there).  It takes 256x256 tiles where their rounds come out ahead (a
// quarter fewer LDS reads and a third fewer copies per MFMA than 128x256: 4096x7168x4096 154 -> 130 us, 4096x4096x8192 159 -> 136 us; with the
// products on the matrix cores 120.6 -> 115.0 and 129.1 -> 122.9 us = 2.09 and 2.24 PFLOP/s; with row-major scales, copied in chunks of four K
// blocks where K is long, 131 -> 122 us), 128x256 and 128x128 tiles otherwise; a plain
// loop (128x128 tile, four waves of 64x64, the K block's two panels and two scale vectors copied global -> LDS by `buffer_load
// ... lds`, double buffered, one barrier per K block: short ends, but 0.93 us per K block against 0.72) runs what has few K blocks.
// K % 128 == 0 (the callers contract over a padded token count).
#include "../../include/mdy_fp8.h"
#include <algorithm>

#include "fp8_gemm_tile.h"

namespace mdy {

// FMT: byte format of both operands, 0 e4m3fn, 1 e5m2 (the MFMA's cbsz / blgp operand-format fields).
template <typename OUT, int FMT, int EPI>
__global__ __launch_bounds__(256) void fp8_gemm_rowscaled_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, int bs_rs, int bs_cs, uint32_t bs_bytes,
    OUT* __restrict__ c, int M, int N, int K, int tiles_n) {
    constexpr int BM = 128, BN = 128;
    __shared__ __attribute__((aligned(1024))) uint8_t lds_a[2][BM * 128];
    __shared__ __attribute__((aligned(1024))) uint8_t lds_b[2][BN * 128];
    __shared__ __attribute__((aligned(256))) float lds_sa[2][BM];
    __shared__ __attribute__((aligned(256))) float lds_sb[2][BN];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    const int KB = K >> 7;

    // ---- copies: 4 waves x 8 rows per instruction, 4 instructions per panel; rows past M / N read zero
    const intx4 ra = make_rsrc(a + (size_t)m0 * K, (uint32_t)min(BM, M - m0) * (uint32_t)K);
    const intx4 rb = make_rsrc(b + (size_t)n0 * K, (uint32_t)min(BN, N - n0) * (uint32_t)K);
    const intx4 rsa = make_rsrc(a_s, as_bytes), rsb = make_rsrc(b_s, bs_bytes);
    const int prow = wave * 8 + (lane >> 3);
    const int voff = prow * K + (((lane & 7) ^ swz(prow)) << 4);
    // scale vectors: waves 0, 1 copy the 128 activation scales of the K block, waves 2, 3 the 128 weight-row scales
    const bool sc_a = wave < 2;
    const int sc_row = (wave & 1) * 64 + lane;
    const intx4 rsc = sc_a ? rsa : rsb;
    const int sc_voff = sc_a ? min(m0 + sc_row, M - 1) * as_rs * 4 : min(n0 + sc_row, N - 1) * bs_rs * 4;
    const int sc_kstep = (sc_a ? as_cs : bs_cs) * 4;
    const uint32_t la = lds_addr(&lds_a[0][0]) + wave * 1024, lb = lds_addr(&lds_b[0][0]) + wave * 1024;
    const uint32_t lsc = (sc_a ? lds_addr(&lds_sa[0][0]) : lds_addr(&lds_sb[0][0])) + (wave & 1) * 256;
    auto copy_block = [&](int kb, int buf) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            dma16(ra, voff, p * 32 * K + kb * 128, la + buf * (BM * 128) + p * 32 * 128);
            dma16(rb, voff, p * 32 * K + kb * 128, lb + buf * (BN * 128) + p * 32 * 128);
        }
        dma4(rsc, sc_voff, kb * sc_kstep, lsc + buf * 512);
    };

    // ---- fragments: lane -> row lane%16 and the 32-byte K slice lane/16 of a 16-row sub-tile
    const int frow = lane & 15, fk = lane >> 4;
    const int a_rd0 = (wm * 64 + frow) * 128 + (((2 * fk) ^ swz(frow)) << 4);
    const int a_rd1 = (wm * 64 + frow) * 128 + (((2 * fk + 1) ^ swz(frow)) << 4);
    const int b_rd0 = (wn * 64 + frow) * 128 + (((2 * fk) ^ swz(frow)) << 4);
    const int b_rd1 = (wn * 64 + frow) * 128 + (((2 * fk + 1) ^ swz(frow)) << 4);
    auto frag = [&](const uint8_t* base, int rd0, int rd1, int idx) {
        const intx4 lo = *reinterpret_cast<const intx4*>(base + rd0 + idx * 2048);
        const intx4 hi = *reinterpret_cast<const intx4*>(base + rd1 + idx * 2048);
        return intx8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };

    floatx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    copy_block(0, 0);
    for (int kb = 0; kb < KB; ++kb) {
        const int buf = kb & 1;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();     // K block kb is in LDS, and every wave has finished reading the other buffer
        if (kb + 1 < KB) copy_block(kb + 1, buf ^ 1);
        intx8 fb[4];
        floatx4 sbv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            fb[j] = frag(lds_b[buf], b_rd0, b_rd1, j);
            sbv[j] = *reinterpret_cast<const floatx4*>(&lds_sb[buf][wn * 64 + j * 16 + 4 * fk]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const intx8 fa = frag(lds_a[buf], a_rd0, a_rd1, i);
            const float sa = lds_sa[buf][wm * 64 + i * 16 + frow];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
                const floatx4 p = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa, zero, FMT, FMT, 0, 0, 0, 0);
                acc[i][j][0] = __builtin_fmaf(p[0], sa * sbv[j][0], acc[i][j][0]);
                acc[i][j][1] = __builtin_fmaf(p[1], sa * sbv[j][1], acc[i][j][1]);
                acc[i][j][2] = __builtin_fmaf(p[2], sa * sbv[j][2], acc[i][j][2]);
                acc[i][j][3] = __builtin_fmaf(p[3], sa * sbv[j][3], acc[i][j][3]);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    if constexpr (EPI != kEpiDirect) {
        static_assert(sizeof(OUT) == 2, "8 KB of LDS per wave");
        __syncthreads();     // the operand panels are free: 8 KB of results per wave
        store_rows<4, 4, OUT, EPI == kEpiLines>(acc, &lds_a[0][0] + wave * 8192, c, N, Bias{}, m0 + wm * 64, n0 + wn * 64, M, N, lane);
        return;
    }
    const bool vec_ok = (N % 4 == 0) && ((reinterpret_cast<uintptr_t>(c) & 15) == 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + wm * 64 + i * 16 + frow;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + wn * 64 + j * 16 + 4 * fk;
            const float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            store4<OUT>(c, N, m, n, M, N, v, vec_ok);
        }
    }
}

// The scheduled tile body of fp8_gemm_tile.h in its row-scaled-weight form; a grid smaller than the number of tiles walks them.
template <int BM, int BN, int STAGES, typename OUT, int FMT, int EPI, bool CHUNKED>
__global__ __launch_bounds__(512) void fp8_gemm_rowscaled_tile_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, int bs_rs, int bs_cs, uint32_t bs_bytes,
    OUT* __restrict__ c, int M, int N, int K, int tiles_m, int tiles_n) {
    using L = TileLds<BM, BN, 8, STAGES, true, CHUNKED>;
    constexpr bool WALK = walks(BM, BN, STAGES, (int)sizeof(OUT), EPI);
    __shared__ __attribute__((aligned(1024))) uint8_t pool[WALK ? L::walk_bytes : L::bytes];
    const int ntiles = tiles_m * tiles_n;
    if constexpr (WALK) {
        Walk<> walk{(int)blockIdx.x, ntiles, tiles_m, tiles_n, BM, BN, 1};
        int m0, n0;
        Duty duty;
        if (!walk(m0, n0, duty)) return;
        fp8_gemm_tile<BM, BN, 2, 4, STAGES, OUT, 0, 0, 0, FMT, true, EPI, CHUNKED>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, c, Bias{}, m0, M, M, n0, N, K, N,
                                                                          duty, 0, K >> 7, pool, bs_rs, bs_cs, bs_bytes, walk);
        return;
    }
    for (int pid = blockIdx.x; pid < ntiles; pid += gridDim.x) {
        int tm, tn;
        const Duty duty = tile_of(xcd_contiguous(pid, ntiles), tiles_m, tiles_n, tm, tn);
        fp8_gemm_tile<BM, BN, 2, 4, STAGES, OUT, 0, 0, 0, FMT, true, EPI, CHUNKED>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, c, Bias{}, tm * BM, M, M,
                                                                     tn * BN, N, K, N, duty, 0, K >> 7, pool, bs_rs, bs_cs, bs_bytes);
        __syncthreads();
    }
}

// 128x128 tiles of the same body, four waves of 64x64, one tile per workgroup: for outputs that leave CUs idle with larger tiles, on a
// ring of 3 K blocks (one workgroup per CU) or of 2 (two per CU).  It took these from the plain loop and from 128x256 tiles that ran one
// to a CU and left others empty: 896x3712x3072 33.2 -> 22.9 us, 1536x1024x2304 20.5 -> 16.5, two per CU 2304x1280x640
// 10.2 -> 8.2, 2560x3200x1024 20.1 -> 15.3, 7296x2176x1792 56.7 -> 44.1.
template <int STAGES, typename OUT, int FMT, int EPI>
__global__ __launch_bounds__(256) void fp8_gemm_rowscaled_small_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, int bs_rs, int bs_cs, uint32_t bs_bytes,
    OUT* __restrict__ c, int M, int N, int K, int tiles_m, int tiles_n) {
    __shared__ __attribute__((aligned(1024))) uint8_t pool[TileLds<128, 128, 4, STAGES, true>::bytes];
    int tm, tn;
    const Duty duty = tile_of(xcd_contiguous(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    fp8_gemm_tile<128, 128, 2, 2, STAGES, OUT, 0, 0, 0, FMT, true, EPI>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, c, Bias{}, tm * 128, M, M, tn * 128, N,
                                                                K, N, duty, 0, K >> 7, pool, bs_rs, bs_cs, bs_bytes);
}

// The 128x256 tiles cut along K: workgroup (slab, tile) writes the fp32 partial sums of K blocks slab * kb_per .. of its tile into a
// workspace [slabs][M][N]; splitk_reduce_kernel adds the slabs in order.
template <int FMT, int EPI, bool CHUNKED>
__global__ __launch_bounds__(512) void fp8_gemm_rowscaled_split_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ a_s, int as_rs, int as_cs, uint32_t as_bytes,
    const uint8_t* __restrict__ b, const float* __restrict__ b_s, int bs_rs, int bs_cs, uint32_t bs_bytes,
    float* __restrict__ ws, int M, int N, int K, int tiles_m, int tiles_n, int slabs, int kb_per) {
    __shared__ __attribute__((aligned(1024))) uint8_t pool[TileLds<128, 256, 8, 3, true, CHUNKED>::bytes];
    const int ntiles = tiles_m * tiles_n;
    // runs per XCD from 13 K blocks per slab on, against K > 8192 from 10 (runs against plain order, warm / cold: 768x512x11648, slabs of 7,
    // 21.9 -> 23.5 / 23.7 -> 26.2 us, 512x1152x10368 (9) 24.0 -> 24.8 / 26.0 -> 27.1, 2304x512x3712 (10) 22.0 -> 23.5 / 24.8 -> 27.0; 640x768x15232
    // (10) 1.08 / 1.06 times as fast, 1408x768x13440 (15) 1.08 / 1.10)
    const int pid = slab_order(blockIdx.x, ntiles * slabs, kb_per >= 13 || (kb_per >= 10 && K > 8192));
    const int ks = __builtin_amdgcn_readfirstlane(pid / ntiles);
    int tm, tn;
    const Duty duty = tile_of(pid - ks * ntiles, tiles_m, tiles_n, tm, tn);
    const int kb0 = ks * kb_per, kb1 = min(K >> 7, kb0 + kb_per);
    fp8_gemm_tile<128, 256, 2, 4, 3, float, 0, 0, 0, FMT, true, EPI, CHUNKED>(a, a_s, as_rs, as_cs, as_bytes, b, b_s, ws + (size_t)ks * M * N, Bias{},
                                                                tm * 128, M, M, tn * 256, N, K, N, duty, kb0, kb1, pool, bs_rs, bs_cs,
                                                                bs_bytes);
}

// Which kernel, and into how many slabs of K.  The time of every form is estimated, in us, and the smallest wins:
//   128x128 tiles, ring of 3, one per CU; two per CU, a tile alone on its CU or a pair of them per K block; 128x256 and 256x256 tiles
//   in rounds of the CUs (a round takes its time whether it is full or not); slabs of 128x256 tiles and their reduction.  Every
//   form writes the output, M x N.
// Fits to 150 shapes of 512..8192 rows and columns and 1 to 128 K blocks, rms error 3-6 % (slabs 9 %).  Against lines between sizes, 250 other
// shapes: 6 % less time in the mean, up to 1.38 times as fast, one of them more than 5 % behind, out of the
// caches alone (3328x512x3456 23.7 -> 23.7 / 25.3 -> 28.1 us).  They were made with the scale products on the VALU; since then every form takes 7
// to 13 % less (200 shapes, 180 others for the forms), too evenly to choose by: refitted constants move one call in fifteen, 0.3 % in the mean.  4096x7168 and 4096x4096 from 2 K blocks on stay on 256x256 tiles.  Up to 2 K blocks, and up to 4 where 128x128 tiles need two workgroups per
// CU, the plain loop's shorter ends win (640x7680x256 5.8 us against 7.1, 1792x3072x384 7.4 / 8.4, 2816x768x256 5.0 / 5.3).  With one K
// block they do so for any number of tiles (against 256x256: 6400x8064 23.9 us / 28.6, 4224x4096 11.6 / 14.5, 5504x2048 8.2 / 8.9; two
// 128x128 per CU are never ahead, 6656x3456 12.7 / 14.3), but where its rounds of two workgroups per CU are twice as many as those of
// 256x256 tiles and the last is hardly begun (5504x4736 15.3 / 14.8, 5248x4992 15.2 / 14.7, 5504x5504 16.0 / 16.9).
enum { kPlainLoop = 0, kTiles128x256 = 1, kTiles256x256 = 2, kTiles128Ring3 = 3, kTiles128Two = 4 };
struct RowscaledPlan {
    int config, slabs, kb_per;
};
static RowscaledPlan plan_rowscaled(int64_t M, int64_t N, int64_t K, bool slabs) {
    const int64_t cus = cu_count(), KB = K / 128, rows = (M + 127) / 128, small = rows * ((N + 127) / 128), wide = rows * ((N + 255) / 256),
                  big = ((M + 255) / 256) * ((N + 255) / 256);
    RowscaledPlan p{kPlainLoop, 1, (int)KB};
    if (K > (1 << 16) || (small <= 2 * cus && (KB <= 2 || (KB <= 4 && small > cus)))) return p;
    if (KB == 1) {
        if (2 * ((big + cus - 1) / cus) <= (small + 2 * cus - 1) / (2 * cus) && (small - 1) % (2 * cus) < cus * 3 / 4) p.config = kTiles256x256;
        return p;
    }
    const double kb = (double)KB, out = (double)M * (double)N * 1e-6;
    const int64_t per_cu = (small + cus - 1) / cus;
    double best = 2.96 + kb * (double)(per_cu / 2) * 1.284 + kb * (double)(per_cu % 2) * 0.82 + 0.283 * out;
    p.config = kTiles128Two;
    auto consider = [&](int config, int64_t n, int64_t per, double us) {
        if (us < best) {
            best = us;
            p = RowscaledPlan{config, (int)n, (int)per};
        }
    };
    if (small <= cus) consider(kTiles128Ring3, 1, KB, 3.84 + kb * (0.671 + 0.071 * (double)small / (double)cus) + 0.155 * out);
    consider(kTiles128x256, 1, KB, 1.66 + (double)((wide + cus - 1) / cus) * (1.015 * kb + 2.09) + 0.262 * out);
    consider(kTiles256x256, 1, KB, 1.46 + (double)((big + cus - 1) / cus) * (1.703 * kb + 2.16) + 0.227 * out);
    best *= 1.05;      // ties go to slabs
    // how many slabs: a K block takes a workgroup 1.0 us, a slab's traffic 1.333 us per million results.  The counts of the estimate that says
    // whether to cut promise up to 5 % less, which is within its error: over 65 shapes that it cut into fewer slabs 1.1 % less time with operands
    // in the caches, 1.1 % more without, up to 17 % (768x640x8192 22.7 us with 11, 26.5 with 8)
    double slabs_us = best, least = 1e30;
    RowscaledPlan cut = p;
    for (int64_t want = 2; slabs && want <= 16 && wide * want <= cus && KB / want >= 4; ++want) {
        const int64_t per = (KB + want - 1) / want, n = (KB + per - 1) / per;
        slabs_us = std::min(slabs_us, 8.22 + (double)per * (0.98 - 0.187 * (double)(wide * n) / (double)cus) + 1.857 * (double)n * out);
        const double cost = (double)per + 1.333 * (double)want * out;
        if (cost < least) {
            least = cost;
            cut = RowscaledPlan{kTiles128x256, (int)n, (int)per};
        }
    }
    return slabs_us < best ? cut : p;
}
int64_t fp8_gemm_rowscaled_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    const RowscaledPlan p = plan_rowscaled(M, N, K, true);
    return p.slabs > 1 ? (int64_t)p.slabs * M * N * 4 : 0;
}

// the form of a call whose operands qualify, and its slabs of K in the bits above
int fp8_gemm_rowscaled_form(int64_t M, int64_t N, int64_t K, int with_workspace) {
    constexpr int kForm[5] = {MDY_FORM_PLAIN_LOOP, MDY_FORM_128X256, MDY_FORM_256X256, MDY_FORM_128X128, MDY_FORM_128X128_TWO};
    const RowscaledPlan p = plan_rowscaled(M, N, K, with_workspace != 0);
    return kForm[p.config] | (p.slabs > 1 ? p.slabs << 8 : 0);
}

// returns hipError_t, or -1 when the operands do not qualify (K % 128 != 0, misaligned, scale extents >= 2^31 bytes)
int launch_fp8_gemm_nt_rowscaled(const void* a, const float* a_s, int64_t as_rs, int64_t as_cs, const void* b,
                                 const float* b_s, int64_t bs_rs, int64_t bs_cs, void* c, int64_t M, int64_t N, int64_t K,
                                 int fmt, int out_dtype, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
    if (M == 0 || N == 0) return 0;
    const int64_t KB = K / 128;
    const int64_t a_ext = ((M - 1) * as_rs + (KB - 1) * as_cs + 1) * 4, b_ext = ((N - 1) * bs_rs + (KB - 1) * bs_cs + 1) * 4;
    if (K % 128 != 0 || K > (1 << 20) || as_rs < 0 || as_cs < 0 || bs_rs < 0 || bs_cs < 0 || a_ext >= ((int64_t)1 << 31) ||
        b_ext >= ((int64_t)1 << 31) || ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & 15) != 0 ||
        128 * K >= ((int64_t)1 << 31))
        return -1;
    RowscaledPlan sp = plan_rowscaled(M, N, K, true);
    // Scales that lie K block after K block (row-major) in chunks of four of them (CHUNKED of TileLds), with tiles of 256 columns, from 12 K blocks on.
    // A K block at a time -> in chunks, row-major: 8192x4096x4096 137 -> 131 us, 7168x2048x4096 67.6 -> 62.9, 1792x4096x4096 39.7 -> 36.9, 4096x7168 with
    // 12 / 16 blocks 52.5 -> 50.7 / 65.2 -> 64.5, but with 2 to 8 blocks +1 % (the first chunk comes before the first K block), 128x128 tiles +2 to 5 % (2048x2048x2048 14.9 ->
    // 15.3); column-major +1 % (4096x7168x1024 38.8 -> 39.4), 128x128 tiles +4 to 8 % (1024x3072x2048 13.5 -> 14.6).  It is all of K that counts, not a slab's
    // part: row-major slabs gain down to 4 blocks, in the caches / out of them 512x512x4096 (8 slabs of 4) 15.7 -> 15.5 / 18.3 -> 17.8, 256x1280x6400 (5) 19.8 ->
    // 19.2 / 21.6 -> 20.6, 2305x512x3712 (6) 20.7 -> 19.9 / 22.0 -> 21.0, 1530x640x4736 (8) 22.7 -> 20.9 / 23.6 -> 21.8; the shortest, 4 slabs of 5,
    // 384x576x2176 13.0 -> 13.5 / 15.9 -> 15.3.  One operand row-major is enough: a weight's 3 % less in the mean of 43 shapes in the caches and 4.5 % out
    // of them, the activations' even (in one launch -7.5 to +3.6 %) and 1 to 3 % less.
    const bool chunked = KB >= 12 && (as_cs < as_rs || bs_cs < bs_rs);
    if (sp.slabs > 1 && workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && workspace_bytes >= (int64_t)sp.slabs * M * N * 4) {
        const int tm = (int)((M + 127) / 128), tn = (int)((N + 255) / 256);
        float* ws = static_cast<float*>(workspace);
#define MDY_RSS(FMT, EPI) do { if (chunked) MDY_RSS_C(FMT, EPI, true); else MDY_RSS_C(FMT, EPI, false); } while (0)
#define MDY_RSS_C(FMT, EPI, CHUNKED)                                                                                     \
    launch_kernel((fp8_gemm_rowscaled_split_kernel<FMT, EPI, CHUNKED>), dim3((unsigned)(tm * tn * sp.slabs)), dim3(512), 0, stream, \
                       static_cast<const uint8_t*>(a), a_s, (int)as_rs, (int)as_cs, (uint32_t)a_ext, static_cast<const uint8_t*>(b), b_s, \
                       (int)bs_rs, (int)bs_cs, (uint32_t)b_ext, ws, (int)M, (int)N, (int)K, tm, tn, sp.slabs, sp.kb_per)
        if (epilogue_kind(ws, N, N, 4, false, true) == kEpiRows) {
            if (fmt == 0) MDY_RSS(0, kEpiRows); else MDY_RSS(1, kEpiRows);
        } else {
            if (fmt == 0) MDY_RSS(0, kEpiDirect); else MDY_RSS(1, kEpiDirect);
        }
#undef MDY_RSS
#undef MDY_RSS_C
        const int rc = (int)hipGetLastError();
        return rc != 0 ? rc : launch_splitk_reduce(ws, c, out_dtype, Bias{}, M, N, sp.slabs, stream);
    }
    if (sp.slabs > 1) sp = plan_rowscaled(M, N, K, false);
    const int cfg = sp.config;
    if (cfg == kTiles128x256 || cfg == kTiles256x256) {
        const int bm = cfg == kTiles256x256 ? 256 : 128;
        const int64_t tm = (M + bm - 1) / bm, tn = (N + 255) / 256, cus = cu_count();
        if (tm * tn > 0x7FFFFFFF) return kErrTooManyBlocks;
        const dim3 grid((unsigned)(cfg == kTiles256x256 && tm * tn > cus ? cus : tm * tn));      // 256x256: a workgroup per CU walks its tiles
#define MDY_RST(BM, ST, OUT_T, FMT, EPI) do { if (chunked) MDY_RST_K(BM, ST, OUT_T, FMT, EPI, true); else MDY_RST_K(BM, ST, OUT_T, FMT, EPI, false); } while (0)
#define MDY_RST_K(BM, ST, OUT_T, FMT, EPI, CHUNKED)                                                                      \
    launch_kernel((fp8_gemm_rowscaled_tile_kernel<BM, 256, ST, OUT_T, FMT, EPI, CHUNKED>), grid, dim3(512), 0, stream,            \
                       static_cast<const uint8_t*>(a), a_s, (int)as_rs, (int)as_cs, (uint32_t)a_ext,                      \
                       static_cast<const uint8_t*>(b), b_s, (int)bs_rs, (int)bs_cs, (uint32_t)b_ext, static_cast<OUT_T*>(c), \
                       (int)M, (int)N, (int)K, (int)tm, (int)tn)
#define MDY_RST_C(OUT_T, FMT, EPI) do { if (cfg == kTiles256x256) MDY_RST(256, 2, OUT_T, FMT, EPI); else MDY_RST(128, 3, OUT_T, FMT, EPI); } while (0)
        const int epi = epilogue_kind(c, N, N, out_dtype == 0 ? 2 : 4, cfg == kTiles256x256, out_dtype == 0);
        if (out_dtype != 0) { if (fmt == 0) MDY_RST_C(float, 0, kEpiDirect); else MDY_RST_C(float, 1, kEpiDirect); }
        else if (epi == kEpiLines) { if (fmt == 0) MDY_RST_C(uint16_t, 0, kEpiLines); else MDY_RST_C(uint16_t, 1, kEpiLines); }
        else if (epi == kEpiRows) { if (fmt == 0) MDY_RST(256, 2, uint16_t, 0, kEpiRows); else MDY_RST(256, 2, uint16_t, 1, kEpiRows); }
        else { if (fmt == 0) MDY_RST_C(uint16_t, 0, kEpiDirect); else MDY_RST_C(uint16_t, 1, kEpiDirect); }
#undef MDY_RST_C
#undef MDY_RST_K
#undef MDY_RST
        return (int)hipGetLastError();
    }
    const int tiles_m = (int)((M + 127) / 128), tiles_n = (int)((N + 127) / 128);
    if ((int64_t)tiles_m * tiles_n > 0x7FFFFFFF) return kErrTooManyBlocks;
    dim3 grid((unsigned)(tiles_m * tiles_n)), block(256);
#define MDY_RS_ARGS(OUT_T)                                                                                                  \
    grid, block, 0, stream, static_cast<const uint8_t*>(a), a_s, (int)as_rs, (int)as_cs, (uint32_t)a_ext, static_cast<const uint8_t*>(b), b_s, \
        (int)bs_rs, (int)bs_cs, (uint32_t)b_ext, static_cast<OUT_T*>(c), (int)M, (int)N, (int)K
#define MDY_RS(OUT_T, FMT, EPI)                                                                                                                     \
    do {                                                                                                                                            \
        if (cfg == kTiles128Ring3) launch_kernel((fp8_gemm_rowscaled_small_kernel<3, OUT_T, FMT, EPI>), MDY_RS_ARGS(OUT_T), tiles_m, tiles_n); \
        else if (cfg == kTiles128Two) launch_kernel((fp8_gemm_rowscaled_small_kernel<2, OUT_T, FMT, EPI>), MDY_RS_ARGS(OUT_T), tiles_m, tiles_n); \
        else launch_kernel((fp8_gemm_rowscaled_kernel<OUT_T, FMT, EPI>), MDY_RS_ARGS(OUT_T), tiles_n);                                          \
    } while (0)
    const int epi = epilogue_kind(c, N, N, out_dtype == 0 ? 2 : 4, false, out_dtype == 0);
    if (out_dtype != 0) { if (fmt == 0) MDY_RS(float, 0, kEpiDirect); else MDY_RS(float, 1, kEpiDirect); }
    else if (epi == kEpiLines) { if (fmt == 0) MDY_RS(uint16_t, 0, kEpiLines); else MDY_RS(uint16_t, 1, kEpiLines); }
    else { if (fmt == 0) MDY_RS(uint16_t, 0, kEpiDirect); else MDY_RS(uint16_t, 1, kEpiDirect); }
#undef MDY_RS
#undef MDY_RS_ARGS
    return (int)hipGetLastError();
}

}  // namespace mdy
