// Device construction of the column-blocked SELL copy (tiled_layout.h), array
// for array what build_sell_blocks writes on the host: the segment bounds of
// every row in every column block, the row order of every sort window, and,
// once the host has placed the slices (place_sell_slices: their widths are a
// few kilobytes), the entries.  Also the check of a CSR's columns.
//
// The host build read the matrix three times on 8-16 threads and sent the
// copy over PCIe after the CSR itself: 9.4 of 14.3 ms of npbcg_create at
// n = 30011, and the host's check of the columns 1.5 ms.  Here the CSR is on
// the device anyway, so the copy costs its own traffic: npbcg_create takes
// 2.2 ms at n = 30011, 8.5 (48.5) at 75000 and 21 (144) at 150000, most of it
// the upload of the CSR and the digest of the caller's arrays.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cg_device.h"
#include "cg_kernels.h"

namespace npbcg_dev {

namespace {

constexpr int kSortBlock = 1024;

// flags[0]: a column outside [0, n); flags[1]: a row whose columns do not
// ascend.  16 lanes per row.
__global__ __launch_bounds__(kBlock) void csr_check_kernel(const int *__restrict__ rowstr,
                                                           const int *__restrict__ colidx, int n,
                                                           int *flags) {
    const int sl = threadIdx.x & 15;
    bool bad = false, unsorted = false;
    for (int j = (blockIdx.x * kBlock + threadIdx.x) / 16; j < n; j += gridDim.x * kBlock / 16) {
        const int s = rowstr[j], e = rowstr[j + 1];
        for (int k = s + sl; k < e; k += 16) {
            const int c = colidx[k];
            bad = bad || c < 0 || c >= n;
            unsorted = unsorted || (k > s && c <= colidx[k - 1]);
        }
    }
    if (bad) atomicOr(&flags[0], 1);
    if (unsorted) atomicOr(&flags[1], 1);
}

// First entry of row j at or past column b W; seg holds the bounds between
// blocks, seg[(b - 1) n + j] for b = 1 .. nblk - 1.
__device__ __forceinline__ int bound(const int *__restrict__ rowstr, const int *__restrict__ seg,
                                     int n, int nblk, int b, int j) {
    return b == 0 ? rowstr[j] : b == nblk ? rowstr[j + 1] : seg[(size_t)(b - 1) * n + j];
}

// seg: one thread per bound, a binary search of the row.
__global__ __launch_bounds__(kBlock) void sell_segments_kernel(const int *__restrict__ rowstr,
                                                               const int *__restrict__ colidx,
                                                               int n, int W, int nblk,
                                                               int *__restrict__ seg) {
    const long long count = (long long)n * (nblk - 1);
    for (long long i = blockIdx.x * (long long)kBlock + threadIdx.x; i < count;
         i += (long long)gridDim.x * kBlock) {
        const int b = (int)(i / n) + 1, j = (int)(i % n);
        int lo = rowstr[j], hi = rowstr[j + 1];
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (colidx[mid] < (long long)b * W)
                lo = mid + 1;
            else
                hi = mid;
        }
        seg[i] = lo;
    }
}

// One workgroup per sort window: its rows ordered by segment length (longest
// first, ties by row) into order[b n + first row ..], and the width of each
// 64-row slice.  A key holds the length and the row's place in the window, so
// no two are alike and the bitonic network gives the stable order.
__global__ __launch_bounds__(kSortBlock) void sell_sort_kernel(
    const int *__restrict__ rowstr, const int *__restrict__ seg, int n, int nblk, int R,
    int nrange, int window, int wins, int size,
    const int *__restrict__ wg_slice, int *__restrict__ order, int *__restrict__ width) {
    extern __shared__ unsigned key[];  // size entries, a power of two
    const int wg = blockIdx.x / wins, w0 = (blockIdx.x % wins) * window;
    const int b = wg / nrange, r0 = (wg % nrange) * R;
    const int r1 = min(n, r0 + R);
    const int rows = min(window, r1 - r0 - w0);
    if (rows <= 0) return;  // uniform: a short last range has fewer windows
    for (int i = threadIdx.x; i < size; i += kSortBlock) {
        key[i] = ~0u;
        if (i < rows) {
            const int j = r0 + w0 + i;
            const int len =
                bound(rowstr, seg, n, nblk, b + 1, j) - bound(rowstr, seg, n, nblk, b, j);
            key[i] = (unsigned)(65536 - len) << kSellSortBits | (unsigned)i;
        }
    }
    __syncthreads();
    for (int k = 2; k <= size; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = threadIdx.x; t < size / 2; t += kSortBlock) {
                const int i = 2 * t - (t & (j - 1)), p = i + j;
                const unsigned x = key[i], y = key[p];
                if ((x > y) == ((i & k) == 0)) {
                    key[i] = y;
                    key[p] = x;
                }
            }
            __syncthreads();
        }
    for (int i = threadIdx.x; i < rows; i += kSortBlock) {
        const unsigned k = key[i];
        order[(size_t)b * n + r0 + w0 + i] = r0 + w0 + (int)(k & ((1u << kSellSortBits) - 1));
        if (i % kWave == 0) width[wg_slice[wg] + (w0 + i) / kWave] = 65536 - (int)(k >> kSellSortBits);
    }
}

// One wavefront per slice: lane l takes the l-th row from order[src[s]] on.
__global__ __launch_bounds__(kBlock) void sell_fill_kernel(
    const int *__restrict__ rowstr, const int *__restrict__ colidx, const double *__restrict__ a,
    const int *__restrict__ seg,
    const int *__restrict__ order, const int *__restrict__ src,
    const int *__restrict__ slice_off, int slices, int n, int nblk, int W, int R,
    int *__restrict__ slice_row, int *__restrict__ row_slot, double *__restrict__ val,
    uint16_t *__restrict__ col) {
    const int s = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / kWave) +
                                                 (int)(threadIdx.x / kWave));
    if (s >= slices) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int from = src[s], b = from / n, at = from % n;
    const bool live = at + lane < min(n, (at / R + 1) * R);
    const int row = live ? order[from + lane] : -1;
    int lo = 0, len = 0;
    if (live) {
        lo = bound(rowstr, seg, n, nblk, b, row);
        len = bound(rowstr, seg, n, nblk, b + 1, row) - lo;
        row_slot[(size_t)b * n + row] = s * kWave + lane;
    }
    slice_row[(size_t)s * kWave + lane] = row;
    const int off = slice_off[s], width = (slice_off[s + 1] - off) / kWave;
#pragma unroll 4
    for (int j = 0; j < width; j++) {
        const size_t to = (size_t)off + (size_t)j * kWave + lane;
        val[to] = j < len ? a[lo + j] : 0.0;
        col[to] = j < len ? (uint16_t)(colidx[lo + j] - b * W) : (uint16_t)0;
    }
}

}  // namespace

hipError_t launch_csr_check(const int *rowstr, const int *colidx, int n, int *flags,
                            hipStream_t st) {
    csr_check_kernel<<<std::min(2048, (n + 15) / 16), kBlock, 0, st>>>(rowstr, colidx, n, flags);
    return hipGetLastError();
}

hipError_t launch_sell_order(const SellBuild &sb, hipStream_t st) {
    hipError_t e = hipSuccess;
    if (sb.nblk > 1) {
        const long long bounds = (long long)sb.n * (sb.nblk - 1);
        sell_segments_kernel<<<(int)std::min<long long>(8192, (bounds + kBlock - 1) / kBlock),
                               kBlock, 0, st>>>(sb.rowstr, sb.colidx, sb.n, sb.W, sb.nblk, sb.seg);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    const int rows = std::min(sb.R, sb.n);
    const int wins = (rows + sb.window - 1) / sb.window;
    int size = 2;
    while (size < std::min(sb.window, rows)) size <<= 1;
    sell_sort_kernel<<<sb.nblk * sb.nrange * wins, kSortBlock, sizeof(unsigned) * size, st>>>(
        sb.rowstr, sb.seg, sb.n, sb.nblk, sb.R, sb.nrange, sb.window, wins, size, sb.wg_slice,
        sb.order, sb.width);
    return hipGetLastError();
}

hipError_t launch_sell_fill(const SellBuild &sb, const int *src, const int *slice_off, int slices,
                            int *slice_row, int *row_slot, double *val, uint16_t *col,
                            hipStream_t st) {
    if (slices < 1) return hipSuccess;
    const int per = kBlock / kWave;
    sell_fill_kernel<<<(slices + per - 1) / per, kBlock, 0, st>>>(
        sb.rowstr, sb.colidx, sb.a, sb.seg, sb.order, src, slice_off, slices, sb.n, sb.nblk, sb.W,
        sb.R, slice_row, row_slot, val, col);
    return hipGetLastError();
}

}  // namespace npbcg_dev
