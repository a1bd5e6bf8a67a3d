// Row padding / unpadding of grouped (mixture-of-experts) activations.
//
// The rows of x are G consecutive groups of m_splits[g] rows; padding copies group g to a slot of
// pad(m_splits[g]) rows (the next multiple of `multiple`) and fills the slot's remaining rows with zeros,
// unpadding copies the first m_splits[g] rows of every slot back.  Restates what Fp8Padding / Fp8Unpadding
// (/root/reference/triton_kernels/megatron_patchs/dpsk_grouped_linear.py:690-902) do with TransformerEngine's
// multi_padding_fused and with torch.split / torch.cat: the padded layout is what the grouped quantizer with
// the transposed copy needs (group sizes that are multiples of 256,
// /root/reference/triton_kernels/megatron_patchs/fp8_matmul.py:227).
//
// One launch per 128 groups: the table of first rows (unpadded and padded) travels as a kernel
// argument and a wave finds the group of its destination row by binary search.  Streaming copy, 16 bytes per
// lane, non-temporal (every byte is touched once).
#include "common.h"

namespace mdy {

constexpr int kPadGroups = 128;     // the table is a kernel argument: 3 KB of the 4 KB a launch may carry
struct PadTable {
    int n_groups;
    int64_t src_start[kPadGroups + 1];   // first row of group g in the source (its [n_groups] = all source rows)
    int64_t dst_start[kPadGroups + 1];   // first row of group g in the destination
    int64_t rows[kPadGroups];            // rows of group g that hold data (the smaller of its two slot sizes)
};

// Pieces of a row that a lane moves: their loads are in flight together and share one search of the table (with one piece per lane,
// 4000 rows of 14336 bytes to 5376: 28 us).  Unpadding takes four; padding, which writes a third more rows than it reads, two: the
// blocks of zeros are gone at once and leave their slots to the others (four -> two pieces: 25.2 -> 23.3 us there, 4000 rows of 8192 bytes
// 16.1 -> 14.5, 12000 rows of 14336 66.4 -> 62.2; unpadding 22.3 = 22.3, 12.6 -> 13.5, 60.7 -> 58.7, 4000 rows of 4096 bytes 7.4 -> 8.1).
constexpr int kPadPieces = 2, kUnpadPieces = 4;

// grid.x: chunks of 64 lanes x PIECES pieces of a row, grid.y/z: destination rows (block_row()), 4 rows per block
template <int VEC, int PIECES>
__global__ __launch_bounds__(256) void group_pad_kernel(const uint8_t* __restrict__ x, uint8_t* __restrict__ y,
                                                         int64_t row_bytes, int64_t dst_rows, const PadTable tbl) {
    const int64_t row = (int64_t)block_row() * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t col = ((int64_t)blockIdx.x * (64 * PIECES) + (threadIdx.x & 63)) * VEC;
    if (row >= dst_rows) return;
    int lo = 0, hi = tbl.n_groups - 1;     // last group whose destination slot starts at or before this row
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tbl.dst_start[mid] <= row) lo = mid; else hi = mid - 1;
    }
    const int64_t r = row - tbl.dst_start[lo];
    const bool data = r < tbl.rows[lo];
    const uint8_t* src = x + (tbl.src_start[lo] + r) * row_bytes + col;
    uint8_t* dst = y + row * row_bytes + col;
    if (VEC == 16) {
        uint4 v[PIECES];
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            v[p] = make_uint4(0u, 0u, 0u, 0u);
            if (data && col + p * 64 * VEC < row_bytes) v[p] = load_nt16(src + p * 64 * VEC);
        }
#pragma unroll
        for (int p = 0; p < PIECES; ++p)
            if (col + p * 64 * VEC < row_bytes) store_nt16(dst + p * 64 * VEC, v[p]);
        return;
    }
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        if (col + p * 64 * VEC >= row_bytes) break;
        if (VEC == 2)
            *reinterpret_cast<uint16_t*>(dst + p * 64 * VEC) = data ? *reinterpret_cast<const uint16_t*>(src + p * 64 * VEC) : (uint16_t)0;
        else
            dst[p * 64 * VEC] = data ? src[p * 64 * VEC] : (uint8_t)0;
    }
}

// unpad == 0: x [sum m, row_bytes] -> y [sum pad(m), row_bytes]; unpad != 0: the reverse.
int launch_group_pad(const void* x, void* y, const int64_t* m_splits, int64_t G, int64_t row_bytes, int64_t multiple,
                     int unpad, hipStream_t stream) {
    const bool a16 = row_bytes % 16 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
    const bool a2 = row_bytes % 2 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 1) == 0;
    const int vec = a16 ? 16 : a2 ? 2 : 1, pieces = unpad ? kUnpadPieces : kPadPieces;
    int64_t src_row = 0, dst_row = 0;
    for (int64_t g0 = 0; g0 < G; g0 += kPadGroups) {
        PadTable tbl;
        const int n = (int)(G - g0 < kPadGroups ? G - g0 : kPadGroups);
        tbl.n_groups = n;
        const int64_t src0 = src_row, dst0 = dst_row;
        for (int g = 0; g < n; ++g) {
            const int64_t m = m_splits[g0 + g], pm = (m + multiple - 1) / multiple * multiple;
            tbl.src_start[g] = src_row - src0;
            tbl.dst_start[g] = dst_row - dst0;
            tbl.rows[g] = m;
            src_row += unpad ? pm : m;
            dst_row += unpad ? m : pm;
        }
        for (int g = n; g <= kPadGroups; ++g) {
            tbl.src_start[g] = src_row - src0;
            tbl.dst_start[g] = dst_row - dst0;
            if (g < kPadGroups) tbl.rows[g] = 0;
        }
        const int64_t rows = dst_row - dst0;
        if (rows == 0 || row_bytes == 0) continue;
        dim3 grid;
        if (!grid_rows((row_bytes + 64 * pieces * vec - 1) / (64 * pieces * vec), (rows + 3) / 4, grid)) return kErrTooManyBlocks;
        const uint8_t* xp = static_cast<const uint8_t*>(x) + src0 * row_bytes;
        uint8_t* yp = static_cast<uint8_t*>(y) + dst0 * row_bytes;
#define MDY_PAD(VEC, PIECES) launch_kernel((group_pad_kernel<VEC, PIECES>), grid, dim3(256), 0, stream, xp, yp, row_bytes, rows, tbl)
#define MDY_PAD_P(VEC) do { if (unpad) MDY_PAD(VEC, kUnpadPieces); else MDY_PAD(VEC, kPadPieces); } while (0)
        if (vec == 16) MDY_PAD_P(16);
        else if (vec == 2) MDY_PAD_P(2);
        else MDY_PAD_P(1);
#undef MDY_PAD_P
#undef MDY_PAD
        const int rc = (int)hipGetLastError();
        if (rc != 0) return rc;
    }
    return 0;
}

}  // namespace mdy
