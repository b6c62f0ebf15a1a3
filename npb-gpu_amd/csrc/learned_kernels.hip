// Device kernels of the learned sparse preconditioner (gfx950).
//
// A message-passing network over the CSR row graph predicts, for every row j,
// two scale corrections g_j, h_j of a sparse approximate inverse:
//   M^-1 = S D^-1 S - Q (N + N^T) Q,  S = diag(e^g), Q = diag(e^(g+h)),
//   N_jk = a_jk / (a_jj a_kk) on the top-K off-diagonals of row j.
//
//   graph     top-K off-diagonals of each row by |a_jk| (ties: lower column);
//             message weights |a_jk| / sqrt|a_jj a_kk|, normalised to sum 1
//   features  8 dimensionless row statistics, standardised per model
//   network   H0 = ReLU(X0 W0 + b0)                     X0: features, 32 wide
//             H_l = ReLU([H_{l-1} | sum_k w_jk H_{l-1,k}] W_l + b_l), l = 1..3
//             g = G tanh(ug . H3 + cg),  h = G tanh(uh . H3 + ch)
//   loss      residual/correction pairs (r_p, e_p = A^-1 r_p) logged from plain
//             CG: L = sum_p |M^-1 r_p - e_p|^2 / (P |e_p|^2)
// GEMMs run on v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32 accumulation).
// Activations are stored BF16; gradients are FP32 until they feed an MFMA.
// Every reduction has a fixed order, so a run repeats bit for bit.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cg_device.h"
#include "learned_kernels.h"

namespace npbcg_dev {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

namespace {

// Workgroups of a grid-stride kernel (capped; the kernel loops).
int blocks_for(long long items, int per_block = kBlock, int cap = 65535) {
    long long b = (items + per_block - 1) / per_block;
    return (int)std::max<long long>(1, std::min<long long>(b, cap));
}

// Workgroups of a kernel that covers exactly one item per thread group (no
// loop, so no cap).
int exact_blocks(long long items, int per_block) {
    return (int)std::max<long long>(1, (items + per_block - 1) / per_block);
}

}  // namespace

int row_blocks(int n) { return exact_blocks((long long)n * 16, kBlock); }
int pair_blocks(int n) { return exact_blocks((long long)n * kPairs, kBlock); }

// ---------------------------------------------------------------------------
// Graph and features (once per matrix)
// ---------------------------------------------------------------------------

// a_jj of every row, 16 lanes per row (0 when the row stores no diagonal).
__global__ __launch_bounds__(kBlock) void diag_kernel(const int *__restrict__ rowstr,
                                                     const int *__restrict__ colidx,
                                                     const double *__restrict__ a,
                                                     double *__restrict__ adiag, int n) {
    const long long gid = blockIdx.x * (long long)kBlock + threadIdx.x;
    const int j = (int)(gid / 16), sub = (int)(gid % 16);
    double d = 0.0;
    if (j < n)
        for (int k = rowstr[j] + sub; k < rowstr[j + 1]; k += 16)
            if (colidx[k] == j) d = a[k];
    d = segment_sum<16>(d);  // one lane holds the diagonal, the others 0
    if (j < n && sub == 0) adiag[j] = d;
}

__device__ __forceinline__ double wave_max(double v) {
    for (int m = 32; m >= 1; m >>= 1) v = fmax(v, __shfl_xor(v, m, kWave));
    return v;
}

__device__ __forceinline__ double safe_abs(double d) { return d != 0.0 ? fabs(d) : 1.0; }

// One wavefront per row: the features and the top-K neighbours.  Selection
// round t takes the best candidate (|a| descending, column ascending) strictly
// after round t-1's; a row with fewer than K off-diagonals is padded with
// zero-weight self edges.  A row of at most kFeatCache * 64 entries is loaded
// into registers once (lane l holds entries l, l + 64, ...; absent entries
// carry column j, which every pass skips as it skips the diagonal) and the
// feature pass and the K selection rounds read it from there, in the same
// order as from memory; longer rows are read from memory in every pass.
__global__ __launch_bounds__(kBlock) void graph_features_kernel(
    const int *__restrict__ rowstr, const int *__restrict__ colidx,
    const double *__restrict__ a, const double *__restrict__ adiag, int n,
    float *__restrict__ feat, int *__restrict__ nbr, float *__restrict__ wgt,
    float *__restrict__ nval) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    constexpr int kFeatCache = 8;
    const int nw = gridDim.x * kWavesPerBlock;
    for (int j = blockIdx.x * kWavesPerBlock + wave; j < n; j += nw) {
        const int s = rowstr[j], e = rowstr[j + 1];
        const double dj = adiag[j];
        const double aj = safe_abs(dj);
        const bool cached = e - s <= kFeatCache * kWave;  // the same for the whole wavefront
        int cc[kFeatCache];
        double cv[kFeatCache], cd[kFeatCache];
        if (cached) {
#pragma unroll
            for (int u = 0; u < kFeatCache; u++) {
                const int k = s + lane + u * kWave;
                cc[u] = k < e ? colidx[k] : j;
                cv[u] = k < e ? a[k] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < kFeatCache; u++) cd[u] = cc[u] != j ? adiag[cc[u]] : 1.0;
        }
        double s_abs = 0, s_sq = 0, s_sgn = 0, s_nb = 0, s_w = 0, mx = 0;
        auto feature_terms = [&](int c, double v, double adc) {
            const double av = fabs(v);
            const double ak = safe_abs(adc);
            s_abs += av;
            s_sq += v * v;
            s_sgn += v;
            s_nb += v * v / (aj * ak);
            s_w += av / sqrt(aj * ak);
            mx = fmax(mx, av);
        };
        if (cached) {
#pragma unroll
            for (int u = 0; u < kFeatCache; u++)
                if (cc[u] != j) feature_terms(cc[u], cv[u], cd[u]);
        } else {
            for (int k = s + lane; k < e; k += kWave) {
                const int c = colidx[k];
                if (c == j) continue;
                feature_terms(c, a[k], adiag[c]);
            }
        }
        s_abs = segment_sum<64>(s_abs);
        s_sq = segment_sum<64>(s_sq);
        s_sgn = segment_sum<64>(s_sgn);
        s_nb = segment_sum<64>(s_nb);
        s_w = segment_sum<64>(s_w);
        mx = wave_max(mx);
        if (lane == 0) {
            float *f = feat + (size_t)j * kFeat;
            f[0] = (float)(s_abs / aj);
            f[1] = (float)(s_sq / (aj * aj));
            f[2] = (float)(mx / aj);
            f[3] = (float)(s_sgn / aj);
            f[4] = (float)s_nb;
            f[5] = (float)s_w;
            f[6] = (float)(log2((double)(e - s)) / 8.0);
            f[7] = (float)(log10(aj) / 3.0);
        }
        double pv = INFINITY;
        int pc = -1;
        double wk[kNbr], nk[kNbr];
        int ck[kNbr];
        double wsum = 0.0;
#pragma unroll
        for (int t = 0; t < kNbr; t++) {
            double bv = -1.0, bval = 0.0;
            int bc = 0x7fffffff;
            auto candidate = [&](int c, double v) {
                const double av = fabs(v);
                const bool after = av < pv || (av == pv && c > pc);
                const bool better = av > bv || (av == bv && c < bc);
                if (after && better) {
                    bv = av;
                    bc = c;
                    bval = v;
                }
            };
            if (cached) {
#pragma unroll
                for (int u = 0; u < kFeatCache; u++)
                    if (cc[u] != j) candidate(cc[u], cv[u]);
            } else {
                for (int k = s + lane; k < e; k += kWave) {
                    const int c = colidx[k];
                    if (c == j) continue;
                    candidate(c, a[k]);
                }
            }
            for (int m = 32; m >= 1; m >>= 1) {
                const double ov = __shfl_xor(bv, m, kWave);
                const int oc = __shfl_xor(bc, m, kWave);
                const double oval = __shfl_xor(bval, m, kWave);
                if (ov > bv || (ov == bv && oc < bc)) {
                    bv = ov;
                    bc = oc;
                    bval = oval;
                }
            }
            if (bv >= 0.0 && bc != 0x7fffffff) {
                const double ak = adiag[bc];
                ck[t] = bc;
                wk[t] = bv / sqrt(aj * safe_abs(ak));
                nk[t] = (dj != 0.0 && ak != 0.0) ? bval / (dj * ak) : 0.0;
            } else {
                ck[t] = j;
                wk[t] = 0.0;
                nk[t] = 0.0;
            }
            wsum += wk[t];
            pv = bv;
            pc = bc;
        }
        if (lane == 0) {
            const double inv = wsum > 0.0 ? 1.0 / wsum : 0.0;
#pragma unroll
            for (int t = 0; t < kNbr; t++) {
                const size_t at = (size_t)j * kNbr + t;
                nbr[at] = ck[t];
                wgt[at] = (float)(wk[t] * inv);
                nval[at] = (float)nk[t];
            }
        }
    }
}

// In-degree of every node over the edges with nonzero weight.
__global__ __launch_bounds__(kBlock) void indegree_kernel(const int *__restrict__ nbr,
                                                          const float *__restrict__ wgt, int n,
                                                          int *__restrict__ cnt) {
    const long long m = (long long)n * kNbr;
    for (long long e = blockIdx.x * (long long)kBlock + threadIdx.x; e < m;
         e += (long long)gridDim.x * kBlock)
        if (wgt[e] != 0.0f) atomicAdd(&cnt[nbr[e]], 1);
}

// ptr[j] = sum of cnt[0..j) for j <= n (exact, so any order gives the same
// values): one 1024-thread workgroup walks the counts in tiles of 8192, each
// thread taking 8 consecutive counts (coalesced across the wavefront), a
// wavefront scan of the thread sums, then the wavefront totals through LDS,
// with a running carry between tiles.
__global__ __launch_bounds__(1024) void scan_kernel(const int *__restrict__ cnt,
                                                    int *__restrict__ ptr, int n) {
    constexpr int kPer = 8, kTile = 1024 * kPer, kWaves = 1024 / kWave;
    __shared__ int wsum[kWaves];
    const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
    int carry = 0;
    for (int base = 0; base < n; base += kTile) {
        int v[kPer], s = 0;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = base + t * kPer + k;
            v[k] = i < n ? cnt[i] : 0;
            s += v[k];
        }
        int x = s;  // inclusive scan over the wavefront
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const int y = __shfl_up(x, off, kWave);
            if (lane >= off) x += y;
        }
        if (lane == kWave - 1) wsum[w] = x;
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int i = 0; i < kWaves; i++) {
            if (i < w) before += wsum[i];
            total += wsum[i];
        }
        int e = carry + before + x - s;  // exclusive prefix of this thread's first count
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = base + t * kPer + k;
            if (i < n) ptr[i] = e;
            e += v[k];
        }
        carry += total;
        __syncthreads();  // wsum is rewritten by the next tile
    }
    if (t == 0) ptr[n] = carry;
}

__global__ __launch_bounds__(kBlock) void transpose_fill_kernel(
    const int *__restrict__ nbr, const float *__restrict__ wgt, const float *__restrict__ nval,
    int n, const int *__restrict__ ptr, int *__restrict__ cursor, int *__restrict__ tsrc,
    float *__restrict__ tw, float *__restrict__ tval) {
    const long long m = (long long)n * kNbr;
    for (long long e = blockIdx.x * (long long)kBlock + threadIdx.x; e < m;
         e += (long long)gridDim.x * kBlock) {
        if (wgt[e] == 0.0f) continue;
        const int k = nbr[e];
        const int at = ptr[k] + atomicAdd(&cursor[k], 1);
        tsrc[at] = (int)(e / kNbr);
        tw[at] = wgt[e];
        tval[at] = nval[e];
    }
}

// Orders each in-list by source row (insertion sort; lists are short), so
// sums over in-edges do not depend on the atomic fill order.
__global__ __launch_bounds__(kBlock) void transpose_sort_kernel(const int *__restrict__ ptr,
                                                                int *__restrict__ tsrc,
                                                                float *__restrict__ tw,
                                                                float *__restrict__ tval,
                                                                int n) {
    for (int k = blockIdx.x * kBlock + threadIdx.x; k < n; k += gridDim.x * kBlock) {
        const int lo = ptr[k], hi = ptr[k + 1];
        for (int i = lo + 1; i < hi; i++) {
            const int sv = tsrc[i];
            const float wv = tw[i], nv = tval[i];
            int p = i - 1;
            while (p >= lo && tsrc[p] > sv) {
                tsrc[p + 1] = tsrc[p];
                tw[p + 1] = tw[p];
                tval[p + 1] = tval[p];
                p--;
            }
            tsrc[p + 1] = sv;
            tw[p + 1] = wv;
            tval[p + 1] = nv;
        }
    }
}

// Mean and standard deviation of each feature over the rows (one workgroup,
// fixed-order tree).  stats = [mean[kFeat], std[kFeat]].
__global__ __launch_bounds__(1024) void feature_stats_kernel(const float *__restrict__ feat,
                                                             int n, float *__restrict__ stats) {
    __shared__ double acc[2 * kFeat][1024 / kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wid = threadIdx.x / kWave;
    double s[2 * kFeat] = {};
    for (int j = threadIdx.x; j < n; j += 1024)
#pragma unroll
        for (int c = 0; c < kFeat; c++) {
            const double v = feat[(size_t)j * kFeat + c];
            s[c] += v;
            s[kFeat + c] += v * v;
        }
#pragma unroll
    for (int c = 0; c < 2 * kFeat; c++) {
        const double t = segment_sum<64>(s[c]);
        if (lane == 0) acc[c][wid] = t;
    }
    __syncthreads();
    if (threadIdx.x < kFeat) {
        const int c = threadIdx.x;
        double m = 0.0, q = 0.0;
        for (int w = 0; w < 1024 / kWave; w++) {
            m += acc[c][w];
            q += acc[kFeat + c][w];
        }
        m /= n;
        const double var = fmax(q / n - m * m, 0.0);
        stats[c] = (float)m;
        stats[kFeat + c] = (float)fmax(sqrt(var), 1e-3);
    }
}

// ---------------------------------------------------------------------------
// Training data: right-hand sides and residual/correction pairs
// ---------------------------------------------------------------------------

// Uniform(-1, 1) right-hand side from a 64-bit mix of (seed, j).
__global__ __launch_bounds__(kBlock) void random_rhs_kernel(double *__restrict__ b, int n,
                                                            unsigned long long seed) {
    for (int j = blockIdx.x * kBlock + threadIdx.x; j < n; j += gridDim.x * kBlock) {
        unsigned long long x = seed * 0x9E3779B97F4A7C15ull + (unsigned long long)j;
        x ^= x >> 30;
        x *= 0xBF58476D1CE4E5B9ull;
        x ^= x >> 27;
        x *= 0x94D049BB133111EBull;
        x ^= x >> 31;
        b[j] = 2.0 * ((double)(x >> 11) * (1.0 / 9007199254740992.0)) - 1.0;
    }
}

// r_p = r, e_p = xstar - z (FP32), partials of |e_p|^2.
__global__ __launch_bounds__(kBlock) void log_pair_kernel(
    const double *__restrict__ r, const double *__restrict__ z,
    const double *__restrict__ xstar, int n, float *__restrict__ r_out,
    float *__restrict__ e_out, double *__restrict__ part) {
    double acc = 0.0;
    for (int j = blockIdx.x * kBlock + threadIdx.x; j < n; j += gridDim.x * kBlock) {
        const float ej = (float)(xstar[j] - z[j]);
        r_out[j] = (float)r[j];
        e_out[j] = ej;
        acc += (double)ej * (double)ej;
    }
    store_block_partial<kBlock>(acc, part);
}

__global__ __launch_bounds__(kBlock) void pair_weights_kernel(const double *__restrict__ part,
                                                              int parts, int pairs,
                                                              float *__restrict__ omega) {
    for (int p = 0; p < pairs; p++) {
        const double s = reduce_partials<kBlock>(part + (size_t)p * parts, parts);
        if (threadIdx.x == 0) omega[p] = s > 0.0 ? (float)(1.0 / (pairs * s)) : 0.0f;
    }
}

__global__ __launch_bounds__(kBlock) void sum_kernel(const double *__restrict__ part, int count,
                                                     double *__restrict__ out) {
    const double s = reduce_partials<kBlock>(part, count);
    if (threadIdx.x == 0) out[0] = s;
}

// ---------------------------------------------------------------------------
// Network forward
// ---------------------------------------------------------------------------

// Y[n x 64] = ReLU(X[n x K] W + b): a wavefront computes the four 16x16
// output blocks of a 16-row tile, K in steps of 32.  Wt is W transposed (64 x K,
// BF16), which the workgroup's four wavefronts share in LDS.  Lane l supplies
// A[l%16][8(l/16)..+7] and B[8(l/16)..+7][l%16] and receives
// D[4(l/16)..+3][l%16] of each 16x16x32 product.  Bound by the chain neighbours ->
// their rows -> products -> stores with few wavefronts to cover it (2.4 a SIMD at
// n = 40009): W in registers, 64 of them a lane, and two tiles a wavefront to read it
// half as often took the network 33, 50 and 66 us at 10007, 40009 and 75000; LDS and
// one tile take 24, 36 and 48 (two tiles: 29, 42, 53).
//
// Layer kinds.  kEmbed (K = 32): X is formed here, the eight standardised features
// zero-padded to 32 columns (BF16), by the 16 lanes whose columns they are, and stored for
// the backward pass when `keep` (a kernel of its own: 4.5 us and a launch boundary).
// kMessage and kLast (K = 128, message passing): columns 64.. of X are formed here,
// X[j, 64:128] = sum_t w[j,t] X[nbr[j,t], 0:64] in FP32, rounded to BF16, each lane
// its 16 columns of its row (the four lanes of a row read whole lines of the
// neighbours), and stored for the backward pass when `keep`.  (As a kernel of its own
// before the product 5.8 us at n = 40009 and a launch boundary.)
// kLast also computes the readout g = G tanh(ug . H3 + cg), h = G tanh(uh . H3 + ch) from
// its rounded outputs, FP64 sums as in readout_sums: a lane's four columns, then the eight
// sums (four rows, g and h) over 16 lanes, every step handing half of them on, so that
// each pair of lanes ends with one sum and the tile needs one tanh; H3 itself is stored
// for the backward pass alone.  (A kernel of its own read H3 back: 5.7 us at n = 40009
// and a launch boundary; here 2.7.)
enum LayerKind { kEmbed, kMessage, kLast };
template <int K, LayerKind KIND>
__global__ __launch_bounds__(kBlock) void gemm_fwd_kernel(__bf16 *x, int ldx, int n,
                                                          const __bf16 *__restrict__ wt,
                                                          const float *__restrict__ bias,
                                                          __bf16 *__restrict__ y, int ldy,
                                                          const int *__restrict__ nbr,
                                                          const float *__restrict__ wgt,
                                                          const float *__restrict__ feat,
                                                          const float *__restrict__ norm,
                                                          const float *__restrict__ ro,
                                                          float gmax, float *__restrict__ gh,
                                                          int keep) {
    constexpr bool AGG = KIND != kEmbed;
    constexpr int KS = K / 32;
    constexpr int KL = AGG ? KS / 2 : KS;        // fragments that are loaded
    constexpr int WV = K * kHid / 8 / kBlock;    // vectors of W^T a thread loads
    __shared__ __bf16 ws[kHid][K + 8];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int row0 = (blockIdx.x * kWavesPerBlock + wave) * 16;
    const int ar = row0 + (lane & 15);
    const int at = min(ar, n - 1);  // every wavefront reaches the barrier
    const int kq = 8 * (lane >> 4);
    int k[kNbr];
    float wv[kNbr];
    if constexpr (AGG)
#pragma unroll
        for (int t = 0; t < kNbr; t++) {
            k[t] = nbr[(size_t)at * kNbr + t];
            wv[t] = wgt[(size_t)at * kNbr + t];
        }
    bf16x8 wl[WV];
#pragma unroll
    for (int u = 0; u < WV; u++)
        wl[u] = *reinterpret_cast<const bf16x8 *>(wt + (size_t)(threadIdx.x + u * kBlock) * 8);
    bf16x8 cur[KS], hv[AGG ? kNbr : 1][KL];
    if constexpr (AGG) {
#pragma unroll
        for (int q = 0; q < KL; q++) {
            cur[q] = *reinterpret_cast<const bf16x8 *>(x + (size_t)at * ldx + 32 * q + kq);
            if (ar >= n) cur[q] = bf16x8{};
        }
#pragma unroll
        for (int t = 0; t < kNbr; t++)
#pragma unroll
            for (int q = 0; q < KL; q++)
                hv[t][q] = *reinterpret_cast<const bf16x8 *>(x + (size_t)k[t] * ldx + 32 * q + kq);
    } else {
        float f[kFeat];
#pragma unroll
        for (int c = 0; c < kFeat; c++) f[c] = (feat[(size_t)at * kFeat + c] - norm[c]) / norm[kFeat + c];
        cur[0] = bf16x8{};
        if (kq == 0 && ar < n)
#pragma unroll
            for (int c = 0; c < kFeat; c++) cur[0][c] = (__bf16)f[c];
        if (keep && ar < n) *reinterpret_cast<bf16x8 *>(x + (size_t)ar * ldx + kq) = cur[0];
    }
    float bj[4], ug[4], uh[4];
#pragma unroll
    for (int jb = 0; jb < 4; jb++) {
        bj[jb] = bias[jb * 16 + (lane & 15)];
        if constexpr (KIND == kLast) {
            ug[jb] = ro[jb * 16 + (lane & 15)];
            uh[jb] = ro[kHid + 1 + jb * 16 + (lane & 15)];
        }
    }
#pragma unroll
    for (int u = 0; u < WV; u++) {
        const int i = (threadIdx.x + u * kBlock) * 8;
        *reinterpret_cast<bf16x8 *>(&ws[i / K][i % K]) = wl[u];
    }
    __syncthreads();
    if (row0 >= n) return;
    if constexpr (AGG) {
#pragma unroll
        for (int q = 0; q < KL; q++) {
            bf16x8 o;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                float acc = 0.f;
#pragma unroll
                for (int t = 0; t < kNbr; t++) acc = fmaf(wv[t], (float)hv[t][q][c], acc);
                o[c] = (__bf16)acc;
            }
            if (ar >= n) o = bf16x8{};
            cur[KL + q] = o;
            if (keep && ar < n)
                *reinterpret_cast<bf16x8 *>(x + (size_t)ar * ldx + kHid + 32 * q + kq) = o;
        }
    }
    f32x4 acc[4] = {};
#pragma unroll
    for (int q = 0; q < KS; q++)
#pragma unroll
        for (int jb = 0; jb < 4; jb++) {
            const bf16x8 bv = *reinterpret_cast<const bf16x8 *>(&ws[jb * 16 + (lane & 15)][32 * q + kq]);
            acc[jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur[q], bv, acc[jb], 0, 0, 0);
        }
    double sums[8] = {};  // g of the lane's four rows, then h
#pragma unroll
    for (int jb = 0; jb < 4; jb++) {
        const int j = jb * 16 + (lane & 15);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int row = row0 + 4 * (lane >> 4) + q;
            const __bf16 v = (__bf16)fmaxf(acc[jb][q] + bj[jb], 0.0f);
            if (row < n && (KIND != kLast || keep)) y[(size_t)row * ldy + j] = v;
            if constexpr (KIND == kLast) {
                sums[q] += (double)((float)v * ug[jb]);
                sums[4 + q] += (double)((float)v * uh[jb]);
            }
        }
    }
    if constexpr (KIND == kLast) {
        // sum i of the eight ends in the lanes with bits 3, 2, 1 of the lane = bits 2, 1, 0 of i
#pragma unroll
        for (int half = 4; half >= 1; half /= 2) {
            const bool up = (lane & (2 * half)) != 0;
#pragma unroll
            for (int i = 0; i < half; i++) {
                const double give = up ? sums[i] : sums[i + half];
                const double mine = up ? sums[i + half] : sums[i];
                sums[i] = mine + __shfl_xor(give, 2 * half, 16);
            }
        }
        sums[0] += __shfl_xor(sums[0], 1, 16);
        const int i = (lane & 15) >> 1;
        const int row = row0 + 4 * (lane >> 4) + (i & 3);
        const double sum = sums[0] + (double)(i < 4 ? ro[kHid] : ro[2 * kHid + 1]);
        const float v = (float)(gmax * tanh(sum));
        if ((lane & 1) == 0 && row < n) gh[(i < 4 ? 0 : n) + row] = v;
    }
}

// The readout's sums ug . H3 + cg and uh . H3 + ch of kReadRows rows from j0 for a
// group of 16 lanes, four columns a lane: lane t of the group keeps row j0 + t's
// sums (lanes past kReadRows: the last row's), so that one tanh serves kReadRows
// rows; hv holds the lane's columns of every row.  FP64 tanh is most of the
// readout's backward kernel (a row per group: 11.1 us at n = 40009, now 7.5).
constexpr int kReadRows = 4;
__device__ __forceinline__ void readout_sums(const __bf16 *__restrict__ h3,
                                             const float (&ug)[4], const float (&uh)[4],
                                             double cg, double ch, long long j0, int n,
                                             bf16x4 (&hv)[kReadRows], double &sg, double &sh) {
    const int sub = threadIdx.x & 15;
#pragma unroll
    for (int t = 0; t < kReadRows; t++) {
        hv[t] = bf16x4{};
        if (j0 + t < n)
            hv[t] = *reinterpret_cast<const bf16x4 *>(h3 + (size_t)(j0 + t) * kHid + sub * 4);
    }
    sg = sh = 0.0;
#pragma unroll
    for (int t = 0; t < kReadRows; t++) {
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            a += (double)((float)hv[t][q] * ug[q]);
            b += (double)((float)hv[t][q] * uh[q]);
        }
        a = segment_sum<16>(a) + cg;
        b = segment_sum<16>(b) + ch;
        if (sub >= t) {
            sg = a;
            sh = b;
        }
    }
}

// ---------------------------------------------------------------------------
// Pair loss under the preconditioner of (g, h)
// ---------------------------------------------------------------------------

// Eight lanes per row, one per pair: 40009 rows are 5000 wavefronts that gather
// at the same time, where a thread per row left 2.4 of them on a CU, each with 64
// gathers of its own in turn (forward and backward 56 and 55 us; now 10 and 10).
static_assert(kPairs == 8, "a row's lanes");

// Sum over the symmetric pattern of row j of C_jk q_k v_k for the lane's pair,
// C = N + N^T, q_k = exp(g_k + h_k): out-edges of j first, then in-edges, the
// lanes of the row taking the next eight edges together.  v_k of the lane's pair
// is v[k * stride].
__device__ __forceinline__ float gather_sym(const NetSystem &sys, const float *__restrict__ gh,
                                            int n, int j, const float *__restrict__ v,
                                            int stride) {
    const int sub = threadIdx.x & (kPairs - 1);
    const int t0 = sys.tptr[j] - kNbr, m = sys.tptr[j + 1] - t0;  // edge e >= kNbr at t0 + e
    float out = 0.0f;
    for (int e0 = 0; e0 < m; e0 += kPairs) {
        const int e = e0 + sub;
        float c = 0.0f;
        int k = -1;
        if (e < kNbr) {
            c = sys.nval[(size_t)j * kNbr + e];
            k = sys.nbr[(size_t)j * kNbr + e];
        } else if (e < m) {
            c = sys.tval[t0 + e];
            k = sys.tsrc[t0 + e];
        }
        if (c == 0.0f) k = -1;
        const float cq = k >= 0 ? c * expf(gh[k] + gh[n + k]) : 0.0f;
        float x[kPairs];
        int kk[kPairs];
#pragma unroll
        for (int t = 0; t < kPairs; t++) {
            kk[t] = __shfl(k, t, kPairs);
            x[t] = v[(size_t)max(kk[t], 0) * stride];
        }
#pragma unroll
        for (int t = 0; t < kPairs; t++) {
            const float ct = __shfl(cq, t, kPairs);
            if (kk[t] >= 0) out = fmaf(ct, x[t], out);
        }
    }
    return out;
}

// y_p = s2_j r_p - q_j w_p, w_p = (C Q r_p)_j; loss partials; pw = w, pd = dL/dy
// ([row][kPairs]).
__global__ __launch_bounds__(kBlock) void pair_loss_fwd_kernel(NetSystem sys,
                                                               const float *__restrict__ gh,
                                                               PairSet ps,
                                                               float *__restrict__ pw,
                                                               float *__restrict__ pd,
                                                               double *__restrict__ loss_part) {
    const int n = sys.n;
    const long long gid = blockIdx.x * (long long)kBlock + threadIdx.x;
    const int j = (int)(gid / kPairs), p = (int)(gid % kPairs);
    double acc = 0.0;
    if (j < n) {
        const size_t column = (size_t)min(p, ps.count - 1) * n;
        const float w = gather_sym(sys, gh, n, j, ps.rt + min(p, ps.count - 1), kPairs);
        if (p < ps.count) {
            const float g = gh[j], h = gh[n + j];
            const float s2 = (float)(exp(2.0 * g) / sys.adiag[j]);
            const float q = expf(g + h);
            const float y = s2 * ps.rt[gid] - q * w;
            const float diff = y - ps.e[column + j];
            acc = (double)ps.omega[p] * (double)diff * (double)diff;
            pw[gid] = w;
            pd[gid] = 2.0f * ps.omega[p] * diff;
        }
    }
    store_block_partial<kBlock>(acc, loss_part);
}

// dL/dq_j = sum_p (-d_pj w_pj - r_pj (C Q d_p)_j); dL/dg = 2 s2 sum_p d r + q dL/dq;
// dL/dh = q dL/dq (the pairs in order, in every lane of the row).
__global__ __launch_bounds__(kBlock) void pair_loss_bwd_kernel(NetSystem sys,
                                                               const float *__restrict__ gh,
                                                               PairSet ps,
                                                               const float *__restrict__ pw,
                                                               const float *__restrict__ pd,
                                                               float *__restrict__ dgh) {
    const int n = sys.n;
    const long long gid = blockIdx.x * (long long)kBlock + threadIdx.x;
    const int j = (int)(gid / kPairs), p = min((int)(gid % kPairs), ps.count - 1);
    if (j >= n) return;
    const float phi = gather_sym(sys, gh, n, j, pd + p, kPairs);
    const size_t at = (size_t)j * kPairs + p;
    const float d = pd[at], r = ps.rt[at];
    const float term = d * pw[at] + r * phi;
    float dq = 0.0f, ds = 0.0f;
    for (int t = 0; t < ps.count; t++) {
        dq -= __shfl(term, t, kPairs);
        ds = fmaf(__shfl(d, t, kPairs), __shfl(r, t, kPairs), ds);
    }
    if (gid % kPairs == 0) {
        const float g = gh[j], h = gh[n + j];
        const float s2 = (float)(exp(2.0 * g) / sys.adiag[j]);
        const float q = expf(g + h);
        dgh[j] = 2.0f * s2 * ds + q * dq;
        dgh[n + j] = q * dq;
    }
}

// ---------------------------------------------------------------------------
// Network backward
// ---------------------------------------------------------------------------

// From dL/dg, dL/dh: dZ3 = (dtg ug + dth uh) * (H3 > 0) in BF16, and this
// workgroup's partial readout gradient [ug(64), cg, uh(64), ch] over its rows
// (16 lanes a row, the sums of a lane's rows in registers; as many workgroups
// as there are parts, kReadoutParts at most: a part for every 16 rows took the
// reduction 44 us at n = 40009).
__global__ __launch_bounds__(kBlock) void readout_bwd_kernel(const __bf16 *__restrict__ h3,
                                                             const float *__restrict__ ro,
                                                             float gmax, int n,
                                                             const float *__restrict__ dgh,
                                                             __bf16 *__restrict__ dz,
                                                             float *__restrict__ rpart) {
    constexpr int kRows = kBlock / 16;
    __shared__ float lds[kRows][kReadout];
    const int sub = threadIdx.x & 15, f = sub * 4;
    const int grp = threadIdx.x / 16;
    float ug[4], uh[4], pg[4] = {}, ph[4] = {}, cg = 0.f, ch = 0.f;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        ug[q] = ro[f + q];
        uh[q] = ro[kHid + 1 + f + q];
    }
    const double cg0 = ro[kHid], ch0 = ro[2 * kHid + 1];
    for (long long b0 = (long long)blockIdx.x * kRows * kReadRows; b0 < n;
         b0 += (long long)gridDim.x * kRows * kReadRows) {
        const long long j0 = b0 + grp * kReadRows;
        bf16x4 hv[kReadRows];
        double sg, sh;
        readout_sums(h3, ug, uh, cg0, ch0, j0, n, hv, sg, sh);
        float mine_g = 0.f, mine_h = 0.f;
        if (sub < kReadRows && j0 + sub < n) {
            const double tg = tanh(sg), th = tanh(sh);
            mine_g = (float)(dgh[j0 + sub] * gmax * (1.0 - tg * tg));
            mine_h = (float)(dgh[n + j0 + sub] * gmax * (1.0 - th * th));
        }
#pragma unroll
        for (int t = 0; t < kReadRows; t++) {
            const float dtg = __shfl(mine_g, t, 16), dth = __shfl(mine_h, t, 16);
            bf16x4 o;
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float h = (float)hv[t][q];
                o[q] = (__bf16)(h > 0.f ? dtg * ug[q] + dth * uh[q] : 0.f);
                pg[q] += dtg * h;
                ph[q] += dth * h;
            }
            if (j0 + t < n) *reinterpret_cast<bf16x4 *>(dz + (size_t)(j0 + t) * kHid + f) = o;
            cg += dtg;
            ch += dth;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        lds[grp][f + q] = pg[q];
        lds[grp][kHid + 1 + f + q] = ph[q];
    }
    if ((threadIdx.x & 15) == 0) {
        lds[grp][kHid] = cg;
        lds[grp][2 * kHid + 1] = ch;
    }
    __syncthreads();
    if (threadIdx.x < kReadout) {
        float s = 0.f;
        for (int r = 0; r < kRows; r++) s += lds[r][threadIdx.x];
        rpart[(size_t)blockIdx.x * kReadout + threadIdx.x] = s;
    }
}

// The top 16 bits of eight floats as BF16 (truncated); v keeps what is left over.
// Three of them hold all 24 bits of a float, so a product over the three is one
// over the FP32 value.  A value without a remainder (infinity, NaN) leaves 0.
__device__ __forceinline__ bf16x8 take_bf16(float *v) {
    union {
        unsigned short h[8];
        bf16x8 b;
    } o;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const unsigned bits = __float_as_uint(v[c]);
        o.h[c] = (unsigned short)(bits >> 16);
        const float rest = v[c] - __uint_as_float(bits & 0xffff0000u);
        v[c] = fabsf(v[c]) < INFINITY ? rest : 0.f;
    }
    return o.b;
}

// Data gradient of a message-passing layer, W row-major [128 x 64] (BF16):
//   dH[k] = dZ[k] W[0:64]^T + (sum over in-edges (j -> k) of w dZ[j]) W[64:128]^T
//   dZprev = dH * (Hprev > 0) in BF16, Hprev = X[:, 0:64] of the layer's input.
// The sum over the in-edges is taken in FP32 before the product, where a row is 128
// bytes of BF16, not of the product's FP32 result; as three BF16 terms (take_bf16) it
// enters the matrix units whole.  A workgroup owns 64 rows: eight lanes a row gather, 8
// columns each, four edges a round with the next round's edges loaded ahead, and leave the
// terms in LDS beside W; then each of the eight wavefronts makes half of a 16-row
// tile's output.  Bound by the chain row pointer -> edges -> gathers and the longest
// in-edge list of a wavefront's rows.
// As a product to FP32 rows in memory and an aggregation kernel, 11.0 + 12.3 us and a
// launch boundary at n = 40009; with a tile and its gathers (four lanes a row) to a
// wavefront 15.3; now 13.9 (loss and gradient at 17003 170 us, now 163; at 40009 210 and
// 207).
constexpr int kWPad = kHid + 8;
constexpr int kBwdBlock = 512, kBwdRows = kBwdBlock / 8;
__global__ __launch_bounds__(kBwdBlock) void layer_bwd_kernel(
    const __bf16 *__restrict__ dz, const int *__restrict__ tptr, const int *__restrict__ tsrc,
    const float *__restrict__ tw, const __bf16 *__restrict__ w, const __bf16 *__restrict__ x,
    int n, __bf16 *__restrict__ dzprev) {
    __shared__ __bf16 ws[kXW][kWPad];
    __shared__ __bf16 terms[3][kBwdRows][kWPad];
    constexpr int WV = kXW * kHid / 8 / kBwdBlock;  // vectors of W a thread loads
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int block0 = blockIdx.x * kBwdRows;
    const int local = threadIdx.x / 8, col = 8 * (threadIdx.x & 7);
    int e0 = 0, e1 = 0;
    if (block0 + local < n) {
        e0 = tptr[block0 + local];
        e1 = tptr[block0 + local + 1];
    }
    bf16x8 wv[WV];
#pragma unroll
    for (int u = 0; u < WV; u++)
        wv[u] = *reinterpret_cast<const bf16x8 *>(w + (size_t)(threadIdx.x + u * kBwdBlock) * 8);
    // the wavefront's part of the output: tile wave / 2, columns 32 (wave % 2) ..
    const int tile = 16 * (wave / 2), row0 = block0 + tile, j0 = 32 * (wave & 1);
    const int kq = 8 * (lane >> 4);
    bf16x8 own[2];
    __bf16 h[2][4];
#pragma unroll
    for (int q = 0; q < 2; q++)
        own[q] = *reinterpret_cast<const bf16x8 *>(
            dz + (size_t)min(row0 + (lane & 15), n - 1) * kHid + 32 * q + kq);
#pragma unroll
    for (int jb = 0; jb < 2; jb++)
#pragma unroll
        for (int t = 0; t < 4; t++)
            h[jb][t] = x[(size_t)min(row0 + 4 * (lane >> 4) + t, n - 1) * kXW + j0 + jb * 16 + (lane & 15)];
    int src[4];
    float wt[4];
    auto edges = [&](int b) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = min(b + u, e1 - 1);
            src[u] = tsrc[e];
            wt[u] = tw[e];
        }
    };
    if (e0 < e1) edges(e0);
    float s[8] = {};
    for (int b = e0; b < e1; b += 4) {
        bf16x8 g[4];
        float cur[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            cur[u] = wt[u];
            g[u] = *reinterpret_cast<const bf16x8 *>(dz + (size_t)src[u] * kHid + col);
        }
        if (b + 4 < e1) edges(b + 4);
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (b + u < e1)
#pragma unroll
                for (int c = 0; c < 8; c++) s[c] = fmaf(cur[u], (float)g[u][c], s[c]);
    }
#pragma unroll
    for (int t = 0; t < 3; t++)
        *reinterpret_cast<bf16x8 *>(&terms[t][local][col]) = take_bf16(s);
#pragma unroll
    for (int u = 0; u < WV; u++) {
        const int i = (threadIdx.x + u * kBwdBlock) * 8;
        *reinterpret_cast<bf16x8 *>(&ws[i / kHid][i % kHid]) = wv[u];
    }
    __syncthreads();
#pragma unroll
    for (int jb = 0; jb < 2; jb++) {
        const int j = j0 + jb * 16 + (lane & 15);
        f32x4 acc = {};
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const bf16x8 b1 = *reinterpret_cast<const bf16x8 *>(&ws[j][32 * q + kq]);
            const bf16x8 b2 = *reinterpret_cast<const bf16x8 *>(&ws[kHid + j][32 * q + kq]);
#pragma unroll
            for (int t = 2; t >= 0; t--) {
                const bf16x8 at =
                    *reinterpret_cast<const bf16x8 *>(&terms[t][tile + (lane & 15)][32 * q + kq]);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at, b2, acc, 0, 0, 0);
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(own[q], b1, acc, 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int row = row0 + 4 * (lane >> 4) + t;
            if (row < n)
                dzprev[(size_t)row * kHid + j] = (__bf16)((float)h[jb][t] > 0.f ? acc[t] : 0.f);
        }
    }
}

// Per-workgroup partial dW[K x 64] = X^T dZ and db[64] = column sums of dZ
// over this workgroup's rows, in chunks of 64 rows; the MFMA reduction
// dimension is the row index.  The chunk is stored in LDS by column, so a lane's
// eight rows of a fragment are one 16-byte read, and the next chunk's loads are
// on their way while this one is multiplied.  Eight wavefronts, one 16-row block
// of dW each (K = 128).  part holds K*64 + 64 floats per workgroup; 256 of them
// a gradient instead of 512 halve what the reduction reads.  All four gradients are one
// launch (blockIdx.y), after the data gradients, which keep every layer's dZ: a launch
// per layer took 7.4 us at n = 40009 (K = 128; 10.3 with 32-row chunks read from LDS two
// bytes at a time), 4 x and their boundaries; now 13.6 for the four.
constexpr int kWgBlock = 512;
constexpr int kWgRows = 64;
struct WeightSet {
    const __bf16 *x, *dz;  // the layer's input [n][K] and dZ [n][kHid]
    float *part;
};
struct WeightSets {
    WeightSet set[kLayers + 1];  // layers 1 to 3 (K = kXW), then the embedding (K = kK0)
};

template <int K>
__device__ __forceinline__ void weight_gradient(const __bf16 *__restrict__ x, int n,
                                                const __bf16 *__restrict__ dz,
                                                float *__restrict__ part,
                                                __bf16 (*xs)[kWgRows + 8],
                                                __bf16 (*gs)[kWgRows + 8]) {
    constexpr int RB = K / 16;                               // 16-row blocks of dW
    constexpr int XV = kWgRows * K / 8 / kWgBlock;           // vectors of X a thread loads
    constexpr int XT = XV > 0 ? XV : 1;
    static_assert(RB <= kWgBlock / kWave && kWgRows * kHid / 8 == kWgBlock, "chunk shape");
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int rr = lane;  // a wavefront loads 8 columns of the chunk's 64 rows
    f32x4 acc[4] = {};
    float db = 0.f;
    bf16x8 xv[XT], gv;
    auto load = [&](int r0) {
        const int row = r0 + rr;
#pragma unroll
        for (int u = 0; u < XT; u++) {
            const int cc = (wave + u * (kWgBlock / kWave)) * 8;
            xv[u] = bf16x8{};
            if (row < n && cc < K)
                xv[u] = *reinterpret_cast<const bf16x8 *>(x + (size_t)row * K + cc);
        }
        gv = bf16x8{};
        if (row < n) gv = *reinterpret_cast<const bf16x8 *>(dz + (size_t)row * kHid + wave * 8);
    };
    int r0 = blockIdx.x * kWgRows;
    if (r0 < n) load(r0);
    for (; r0 < n; r0 += gridDim.x * kWgRows) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < XT; u++) {
            const int cc = (wave + u * (kWgBlock / kWave)) * 8;
            if (cc < K)
#pragma unroll
                for (int t = 0; t < 8; t++) xs[cc + t][rr] = xv[u][t];
        }
#pragma unroll
        for (int t = 0; t < 8; t++) gs[wave * 8 + t][rr] = gv[t];
        __syncthreads();
        if (r0 + (int)gridDim.x * kWgRows < n) load(r0 + gridDim.x * kWgRows);
        const int kq = 8 * (lane >> 4);
        if (wave < RB) {
#pragma unroll
            for (int ks = 0; ks < kWgRows / 32; ks++) {
                const bf16x8 av =
                    *reinterpret_cast<const bf16x8 *>(&xs[wave * 16 + (lane & 15)][ks * 32 + kq]);
#pragma unroll
                for (int jb = 0; jb < 4; jb++) {
                    const bf16x8 bv =
                        *reinterpret_cast<const bf16x8 *>(&gs[jb * 16 + (lane & 15)][ks * 32 + kq]);
                    acc[jb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc[jb], 0, 0, 0);
                }
            }
        }
        if (threadIdx.x < kHid)
#pragma unroll
            for (int q = 0; q < kWgRows; q += 8) {
                const bf16x8 v = *reinterpret_cast<const bf16x8 *>(&gs[threadIdx.x][q]);
#pragma unroll
                for (int t = 0; t < 8; t++) db += (float)v[t];
            }
    }
    float *out = part + (size_t)blockIdx.x * (K * kHid + kHid);
    if (wave < RB) {
#pragma unroll
        for (int jb = 0; jb < 4; jb++)
#pragma unroll
            for (int t = 0; t < 4; t++)
                out[(size_t)(wave * 16 + 4 * (lane >> 4) + t) * kHid + jb * 16 + (lane & 15)] =
                    acc[jb][t];
    }
    if (threadIdx.x < kHid) out[K * kHid + threadIdx.x] = db;
}

__global__ __launch_bounds__(kWgBlock) void gemm_bwd_weight_kernel(WeightSets sets, int n) {
    __shared__ __bf16 xs[kXW][kWgRows + 8];
    __shared__ __bf16 gs[kHid][kWgRows + 8];
    const WeightSet ws = sets.set[blockIdx.y];
    if (blockIdx.y < kLayers)
        weight_gradient<kXW>(ws.x, n, ws.dz, ws.part, xs, gs);
    else
        weight_gradient<kK0>(ws.x, n, ws.dz, ws.part, xs, gs);
}

// out[i] = sum over p of part[p * stride + i], i < count, p in increasing
// order within each of kRedWaves interleaved groups, the groups then added in
// order (a fixed order: the same bits every run), for every gradient of a
// backward pass in one launch.  A 1024-thread workgroup takes 64 consecutive
// columns of one of them; wavefront w sums the parts p = w, w + 16, ... of its
// lane's column, eight loads in flight, so the loads are coalesced and 16
// wavefronts share a column's parts.  (A launch per gradient, one load in flight:
// 83 us at n = 40009; now 6.8.)
constexpr int kRedWaves = 16;
constexpr int kRedSets = kLayers + 2;
struct RedSet {
    const float *part;
    float *out;
    int parts, stride, first_block;  // columns: stride
};
struct RedSets {
    RedSet set[kRedSets];
};
__global__ __launch_bounds__(kRedWaves * kWave) void reduce_parts_kernel(RedSets sets) {
    __shared__ float ws[kRedWaves][kWave];
    int which = 0;
#pragma unroll
    for (int i = 1; i < kRedSets; i++)
        if ((int)blockIdx.x >= sets.set[i].first_block) which = i;
    const RedSet rs = sets.set[which];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int i = (blockIdx.x - rs.first_block) * kWave + lane;
    float s = 0.f;
    if (i < rs.stride) {
        const float *from = rs.part + i;
        int p = wave;
        for (; p + 7 * kRedWaves < rs.parts; p += 8 * kRedWaves) {
            float t[8];
#pragma unroll
            for (int u = 0; u < 8; u++) t[u] = from[(size_t)(p + u * kRedWaves) * rs.stride];
#pragma unroll
            for (int u = 0; u < 8; u++) s += t[u];
        }
        for (; p < rs.parts; p += kRedWaves) s += from[(size_t)p * rs.stride];
    }
    ws[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && i < rs.stride) {
        float t = ws[0][lane];
        for (int w = 1; w < kRedWaves; w++) t += ws[w][lane];
        rs.out[i] = t;
    }
}

// Adam step on the FP32 master parameters (bias-corrected moments).
__global__ __launch_bounds__(kBlock) void adam_kernel(float *__restrict__ p,
                                                      const float *__restrict__ g,
                                                      float *__restrict__ m1,
                                                      float *__restrict__ m2, int count, float lr,
                                                      float b1, float b2, float eps, float c1,
                                                      float c2) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < count; i += gridDim.x * kBlock) {
        const float gi = g[i];
        const float a = b1 * m1[i] + (1.f - b1) * gi;
        const float v = b2 * m2[i] + (1.f - b2) * gi * gi;
        m1[i] = a;
        m2[i] = v;
        p[i] -= lr * (a / c1) / (sqrtf(v / c2) + eps);
    }
}

// g *= 1 / den[0] (per-system weighting of a gradient; den > 0).
__global__ __launch_bounds__(kBlock) void scale_inverse_kernel(float *__restrict__ g, int count,
                                                               const double *__restrict__ den) {
    const double d = den[0];
    const float s = d > 0.0 ? (float)(1.0 / d) : 1.0f;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < count; i += gridDim.x * kBlock) g[i] *= s;
}

// BF16 copies of the layer weights: W (K x 64, row-major) and W^T (64 x K).
__global__ __launch_bounds__(kBlock) void pack_weights_kernel(const float *__restrict__ params,
                                                              __bf16 *__restrict__ wb) {
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < kWtElems; i += gridDim.x * kBlock) {
        int K, base, src;
        if (i < kK0 * kHid) {
            K = kK0;
            base = 0;
            src = kOffW0;
        } else {
            const int l = (i - kK0 * kHid) / (kXW * kHid);
            K = kXW;
            base = kK0 * kHid + l * kXW * kHid;
            src = kOffW1 + l * kLayerStride;
        }
        const int local = i - base;
        const int kin = local / kHid, jo = local % kHid;
        const __bf16 v = (__bf16)params[src + local];
        wb[kWtRowMajor + base + local] = v;           // W[kin][jo]
        wb[kWtTransposed + base + jo * K + kin] = v;  // W^T[jo][kin]
    }
}

// ---------------------------------------------------------------------------
// Preconditioner operator
// ---------------------------------------------------------------------------

// Eight lanes per row (9 entries on average): entry 0 is the diagonal
// exp(2 g_j) / a_jj, the others -exp(g_j + h_j + g_k + h_k) N (0 for padding).
// (A thread per row, its entries in turn: 24 us at n = 60013; now 11.8 us.)
__global__ __launch_bounds__(kBlock) void precond_values_kernel(
    int n, const int *__restrict__ off, const int *__restrict__ col,
    const float *__restrict__ src_val, const double *__restrict__ adiag,
    const float *__restrict__ gh, double *__restrict__ val, float *__restrict__ val32) {
    const long long gid = blockIdx.x * (long long)kBlock + threadIdx.x;
    const int j = (int)(gid / 8);
    if (j >= n) return;
    const int e0 = off[j], e1 = off[j + 1];
    const double gj = (double)gh[j] + gh[n + j];
    for (int e = e0 + (int)(gid % 8); e < e1; e += 8) {
        double v;
        if (e == e0) {
            const double d = adiag[j];
            v = d != 0.0 ? exp(2.0 * (double)gh[j]) / d : 0.0;
        } else {
            const float sv = src_val[e];
            const int k = col[e];
            v = sv != 0.0f ? -exp(gj + gh[k] + gh[n + k]) * sv : 0.0;
        }
        val[e] = v;
        val32[e] = (float)v;
    }
}

// z = M^-1 r, 4 lanes per row; p = z when p is given; r.z partials.  A row
// holds the diagonal, 4 out-neighbours and its in-neighbours (9 entries on
// average), so a lane's entries e, e + 4, e + 8 are loaded together and one
// round of dependent loads (row bounds, then columns and values, then the
// gathered r) serves the whole row.  The gathers are latency-bound, so the
// workgroups are 1024 wide and the vector kernels' grid (the partial count
// the next kernel expects) holds every row of n = 150000 in one pass.
constexpr int kApplyBlock = 1024;
template <typename T>
__global__ __launch_bounds__(kApplyBlock) void precond_apply_kernel(
    int n, const int *__restrict__ off, const int *__restrict__ col, const T *__restrict__ val,
    const T *__restrict__ r, T *__restrict__ z, T *__restrict__ p, double *__restrict__ rz_part,
    const Scalars *__restrict__ sc) {
    constexpr int kLanes = 4;
    constexpr int kUnroll = 3;
    constexpr int kRows = kApplyBlock / kLanes;
    if (sc && sc->done) return;
    const int sub = threadIdx.x % kLanes;
    double acc = 0.0;
    const long long stride = (long long)gridDim.x * kRows;
    for (long long j = blockIdx.x * (long long)kRows + threadIdx.x / kLanes; j < n;
         j += stride) {
        T zj = 0;
        const int e1 = off[j + 1];
        for (int e = off[j] + sub; e < e1; e += kLanes * kUnroll) {
            T v[kUnroll];
            int c[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; u++) {
                const bool in = e + u * kLanes < e1;
                v[u] = in ? val[e + u * kLanes] : T(0);
                c[u] = in ? col[e + u * kLanes] : (int)j;
            }
#pragma unroll
            for (int u = 0; u < kUnroll; u++) zj += v[u] * r[c[u]];
        }
#pragma unroll
        for (int m = kLanes / 2; m >= 1; m >>= 1) zj += __shfl_xor(zj, m, kWave);
        if (sub == 0) {
            z[j] = zj;
            if (p) p[j] = zj;
            acc += (double)r[j] * (double)zj;
        }
    }
    store_block_partial<kApplyBlock>(acc, rz_part);
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------

hipError_t launch_graph_features(const int *rowstr, const int *colidx, const double *a, int n,
                                 double *adiag, float *feat, int *nbr, float *wgt, float *nval,
                                 hipStream_t st) {
    diag_kernel<<<row_blocks(n), kBlock, 0, st>>>(rowstr, colidx, a, adiag, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    graph_features_kernel<<<blocks_for(n, kWavesPerBlock), kBlock, 0, st>>>(
        rowstr, colidx, a, adiag, n, feat, nbr, wgt, nval);
    return hipGetLastError();
}

hipError_t launch_transpose(const int *nbr, const float *wgt, const float *nval, int n, int *cnt,
                            int *tptr, int *tsrc, float *tw, float *tval, hipStream_t st) {
    hipError_t e = hipMemsetAsync(cnt, 0, sizeof(int) * (size_t)n, st);
    if (e != hipSuccess) return e;
    indegree_kernel<<<blocks_for((long long)n * kNbr), kBlock, 0, st>>>(nbr, wgt, n, cnt);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    scan_kernel<<<1, 1024, 0, st>>>(cnt, tptr, n);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = hipMemsetAsync(cnt, 0, sizeof(int) * (size_t)n, st)) != hipSuccess) return e;
    transpose_fill_kernel<<<blocks_for((long long)n * kNbr), kBlock, 0, st>>>(
        nbr, wgt, nval, n, tptr, cnt, tsrc, tw, tval);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    transpose_sort_kernel<<<blocks_for(n), kBlock, 0, st>>>(tptr, tsrc, tw, tval, n);
    return hipGetLastError();
}

// Structure of the operator M^-1 = D (I + G N + N^T H) D as a CSR: row j is
// [j | its K out-neighbours | its in-neighbours (transpose order)], so its
// first entry sits at j (1 + K) + tptr[j] and no scan is needed.  src holds
// the neighbour values (0 for the diagonal slot).  One thread per row, grid
// stride (row n only writes off[n]).
__global__ __launch_bounds__(kBlock) void build_op_kernel(const int *__restrict__ nbr,
                                                          const float *__restrict__ nval,
                                                          const int *__restrict__ tptr,
                                                          const int *__restrict__ tsrc,
                                                          const float *__restrict__ tval, int n,
                                                          int *__restrict__ off,
                                                          int *__restrict__ col,
                                                          float *__restrict__ src) {
    for (int j = blockIdx.x * kBlock + threadIdx.x; j <= n; j += gridDim.x * kBlock) {
        const int t0 = tptr[j];
        const int base = j * (1 + kNbr) + t0;
        off[j] = base;
        if (j == n) break;
        col[base] = j;
        src[base] = 0.0f;
#pragma unroll
        for (int t = 0; t < kNbr; t++) {
            col[base + 1 + t] = nbr[(size_t)j * kNbr + t];
            src[base + 1 + t] = nval[(size_t)j * kNbr + t];
        }
        const int t1 = tptr[j + 1];
        for (int e = t0; e < t1; e++) {
            col[base + 1 + kNbr + e - t0] = tsrc[e];
            src[base + 1 + kNbr + e - t0] = tval[e];
        }
    }
}

hipError_t launch_build_op(const int *nbr, const float *nval, const int *tptr, const int *tsrc,
                           const float *tval, int n, int *off, int *col, float *src,
                           hipStream_t st) {
    build_op_kernel<<<blocks_for((long long)n + 1), kBlock, 0, st>>>(nbr, nval, tptr, tsrc, tval,
                                                                    n, off, col, src);
    return hipGetLastError();
}

hipError_t launch_feature_stats(const float *feat, int n, float *stats, hipStream_t st) {
    feature_stats_kernel<<<1, 1024, 0, st>>>(feat, n, stats);
    return hipGetLastError();
}

hipError_t launch_log_pair(const double *r, const double *z, const double *xstar, int n,
                           float *r_out, float *e_out, double *part, int blocks,
                           hipStream_t st) {
    log_pair_kernel<<<blocks, kBlock, 0, st>>>(r, z, xstar, n, r_out, e_out, part);
    return hipGetLastError();
}

// rt[j][p] = r[p][j], so that a row's lanes read the pairs of a neighbour as one run.
__global__ __launch_bounds__(kBlock) void interleave_pairs_kernel(const float *__restrict__ r,
                                                                  int pairs, int n,
                                                                  float *__restrict__ rt) {
    const long long gid = blockIdx.x * (long long)kBlock + threadIdx.x;
    const int j = (int)(gid / kPairs), p = (int)(gid % kPairs);
    if (j < n) rt[gid] = p < pairs ? r[(size_t)p * n + j] : 0.0f;
}

hipError_t launch_interleave_pairs(const float *r, int pairs, int n, float *rt, hipStream_t st) {
    interleave_pairs_kernel<<<pair_blocks(n), kBlock, 0, st>>>(r, pairs, n, rt);
    return hipGetLastError();
}

hipError_t launch_pair_weights(const double *part, int parts, int pairs, float *omega,
                               hipStream_t st) {
    pair_weights_kernel<<<1, kBlock, 0, st>>>(part, parts, pairs, omega);
    return hipGetLastError();
}

hipError_t launch_random_rhs(double *b, int n, unsigned long long seed, hipStream_t st) {
    random_rhs_kernel<<<blocks_for(n), kBlock, 0, st>>>(b, n, seed);
    return hipGetLastError();
}

hipError_t launch_sum(const double *part, int count, double *out, hipStream_t st) {
    sum_kernel<<<1, kBlock, 0, st>>>(part, count, out);
    return hipGetLastError();
}

hipError_t launch_net_forward(const NetBuffers &nb, const NetSystem &sys, const float *params,
                              const __bf16 *wb, float gmax, int keep, hipStream_t st) {
    const int n = sys.n;
    hipError_t e;
    const int blocks = exact_blocks(n, 16 * kWavesPerBlock);  // one 16-row tile per wavefront
    gemm_fwd_kernel<kK0, kEmbed><<<blocks, kBlock, 0, st>>>(
        nb.x0, kK0, n, wb + kWtTransposed, params + kOffB0, nb.x[0], kXW, nullptr, nullptr, sys.feat,
        nb.norm, nullptr, 0.f, nullptr, keep);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    for (int l = 0; l < kLayers; l++) {
        const bool last = l + 1 == kLayers;
        const auto kernel = last ? gemm_fwd_kernel<kXW, kLast> : gemm_fwd_kernel<kXW, kMessage>;
        kernel<<<blocks, kBlock, 0, st>>>(
            nb.x[l], kXW, n, wb + kWtTransposed + kK0 * kHid + l * kXW * kHid,
            params + kOffB1 + l * kLayerStride, last ? nb.h3 : nb.x[l + 1], last ? kHid : kXW,
            sys.nbr, sys.wgt, nullptr, nullptr, params + kOffR, gmax, nb.gh, keep);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_pair_loss(const NetBuffers &nb, const NetSystem &sys, const PairSet &ps,
                            int want_grad, hipStream_t st) {
    const int blocks = pair_blocks(sys.n);
    pair_loss_fwd_kernel<<<blocks, kBlock, 0, st>>>(sys, nb.gh, ps, nb.pw, nb.pd, nb.loss_part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !want_grad) return e;
    pair_loss_bwd_kernel<<<blocks, kBlock, 0, st>>>(sys, nb.gh, ps, nb.pw, nb.pd, nb.dgh);
    return hipGetLastError();
}

hipError_t launch_net_backward(const NetBuffers &nb, const NetSystem &sys, const float *params,
                               const __bf16 *wb, float gmax, float *grad, hipStream_t st) {
    const int n = sys.n;
    hipError_t e;
    const int rb = std::min(kReadoutParts, exact_blocks((long long)n * 16, kBlock * kReadRows));
    readout_bwd_kernel<<<rb, kBlock, 0, st>>>(nb.h3, params + kOffR, gmax, n, nb.dgh,
                                              nb.dz[kLayers], nb.rpart);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    RedSets sets;
    int blocks = 0, used = 0;
    auto reduce = [&](const float *part, int parts, int columns, float *out) {
        sets.set[used++] = {part, out, parts, columns, blocks};
        blocks += (columns + kWave - 1) / kWave;
    };
    reduce(nb.rpart, rb, kReadout, grad + kOffR);
    const int wgb = std::min(kWeightParts, exact_blocks(n, kWgRows));
    WeightSets ws;
    for (int l = kLayers - 1; l >= 0; l--) {
        layer_bwd_kernel<<<exact_blocks(n, kBwdRows), kBwdBlock, 0, st>>>(
            nb.dz[l + 1], sys.tptr, sys.tsrc, sys.tw,
            wb + kWtRowMajor + kK0 * kHid + l * kXW * kHid, nb.x[l], n, nb.dz[l]);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        float *part = nb.wpart + (size_t)l * kWeightParts * kLayerStride;
        ws.set[l] = {nb.x[l], nb.dz[l + 1], part};
        reduce(part, wgb, kLayerStride, grad + kOffW1 + l * kLayerStride);
    }
    float *part = nb.wpart + (size_t)kLayers * kWeightParts * kLayerStride;
    ws.set[kLayers] = {nb.x0, nb.dz[0], part};
    reduce(part, wgb, kK0 * kHid + kHid, grad + kOffW0);
    gemm_bwd_weight_kernel<<<dim3(wgb, kLayers + 1), kWgBlock, 0, st>>>(ws, n);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    reduce_parts_kernel<<<blocks, kRedWaves * kWave, 0, st>>>(sets);
    return hipGetLastError();
}

hipError_t launch_adam(float *p, const float *g, float *m1, float *m2, int count, float lr,
                       float b1, float b2, float eps, int step, hipStream_t st) {
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    adam_kernel<<<blocks_for(count), kBlock, 0, st>>>(p, g, m1, m2, count, lr, b1, b2, eps, c1,
                                                      c2);
    return hipGetLastError();
}

hipError_t launch_scale_inverse(float *g, int count, const double *den, hipStream_t st) {
    scale_inverse_kernel<<<blocks_for(count), kBlock, 0, st>>>(g, count, den);
    return hipGetLastError();
}

hipError_t launch_pack_weights(const float *params, __bf16 *wb, hipStream_t st) {
    pack_weights_kernel<<<blocks_for(kWtElems), kBlock, 0, st>>>(params, wb);
    return hipGetLastError();
}

hipError_t launch_precond_values(const PrecondOp &op, const double *adiag, const float *gh,
                                 hipStream_t st) {
    precond_values_kernel<<<exact_blocks((long long)op.n * 8, kBlock), kBlock, 0, st>>>(
        op.n, op.off, op.col, op.src_val, adiag, gh, op.val, op.val32);
    return hipGetLastError();
}

hipError_t launch_precond_apply(const PrecondOp &op, const double *r, double *z, double *p,
                                double *rz_part, int blocks, const Scalars *sc,
                                hipStream_t st) {
    precond_apply_kernel<double><<<blocks, kApplyBlock, 0, st>>>(op.n, op.off, op.col, op.val, r,
                                                                 z, p, rz_part, sc);
    return hipGetLastError();
}

hipError_t launch_precond_apply32(const PrecondOp &op, const float *r, float *z, float *p,
                                  double *rz_part, int blocks, const Scalars *sc,
                                  hipStream_t st) {
    precond_apply_kernel<float><<<blocks, kApplyBlock, 0, st>>>(op.n, op.off, op.col, op.val32,
                                                                r, z, p, rz_part, sc);
    return hipGetLastError();
}

}  // namespace npbcg_dev
