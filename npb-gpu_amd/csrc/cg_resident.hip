// Resident FP64 CG for small orders (gfx950): one launch runs whole conj_grads
// (cg.cu:803-846) or one solve, with a single exchange between workgroups per
// CG step and the matrix held in registers.
//
// Every workgroup keeps the whole residual r in its LDS and the whole q in
// its registers; the rows are dealt out, and the product, p and z of a row
// belong to its workgroup.  A step is the one-reduction form of
// update_cg_kernel:
//   s = A r of the own rows, from r in LDS, and their part of r.s
//   exchange: every workgroup reads every s and every part; while the words
//   travel it forms rho = r.r, beta = rho / rho_prev and beta rho / alpha_prev
//   q = s + beta q (= A p), alpha = rho / (r.s - beta rho / alpha_prev)
//   p = r + beta p, z += alpha p of the own rows; r -= alpha q over all rows
// so the vector work that needs all rows is repeated by every workgroup.  They
// add the same numbers in the same order, hold the same bits of r, q, alpha
// and beta, and take the same branches.  The reference's order with the same
// exchange (p in LDS; rho, beta and p = r + beta p before the next product)
// took 2.8, 5.0 and 8.3 us a step at n = 1400, 7000 and 14000 against 2.2,
// 3.8 and 7.0 (both with kernels for five word counts; with those below 1.9,
// 3.5 and 6.4).
//
// Exchange: a value is its own flag.  Each exchange of a launch has its own
// buffer, filled with the all-ones NaN before the launch (resident_arm_kernel,
// ordered by the launch boundary); a word is stored once and every workgroup
// reads it until it is something else.  Both are relaxed device-scope atomics
// on one 8-byte word, so nothing else has to be ordered: no fence, no L2
// write-back or invalidate, no counter.  A result that is itself the all-ones
// NaN is stored as the default NaN.  Measured (256 workgroups, exchange
// alone): 1.4 us at n = 1400, 2.3 at 7000, 3.5 at 14000; a flag per workgroup
// followed by plain loads takes 3.1, 5.7 and 6.9 us.
// The grid fits the GPU at one workgroup per CU, and the host lets one such
// launch run at a time on a device (in_resident_order), so the workgroups wait
// for each other only.  It is not a cooperative launch: the runtime gives its
// cooperative queue to one process at a time, and a second process on the GPU
// would be refused.  Where another process's kernels keep workgroups from
// starting, every wait is bounded: one longer than spin_limit wall-clock ticks
// sets the abort word, after which no read waits, so the grid always drains.
// The word is cleared once a call: the later launches of a power loop whose
// results start from that one's do nothing, and the host sees the word and
// runs the multi-kernel engine from the untouched x.
//
// Words: the exchange buffers and the LDS vector are cut into chunks of C
// words, C - 1 rows and the chunk's partial.  One wavefront owns a chunk and
// stores it whole, in 128-byte lines that nobody else writes (the rows of a
// chunk stored by several wavefronts: 3.8 against 2.3 us a step at n = 1400,
// 7.4 against 3.8 at 7000).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cg_device.h"
#include "cg_kernels.h"

namespace npbcg_dev {

namespace {

constexpr int kResBlock = 512;  // 256 vector registers a thread
constexpr int kResWaves = kResBlock / kWave;
typedef unsigned long long u64;
constexpr u64 kEmpty = ~0ull;             // an entry not stored yet
constexpr u64 kNan = 0x7FF8000000000000ull;

struct ResArgs {
    const double *val;     // entry u of lane l of wave w at (wave_off[w] + u) * 64 + l
    const uint16_t *col;   // word of the column
    const int *wave_off;   // [G * 8 + 1]
    const int *word_row;   // [words] row of a word; -1: a partial, or past the rows
    int n, words, stride;  // words in use; words of one exchange buffer
    u64 *xchg;
    unsigned *abort_word;  // set by a wait that ran out; [1] by one of an earlier launch
    long long spin_limit;
    double *x, *z, *p, *q, *r;
    double *part;          // [niter][2][chunks]: ||x - A z||^2 and x.z
    double *zz;            // [niter]
    Scalars *sc;
    int steps;             // CG steps (at most, in a solve)
    int niter, scale_first;
    int solve;             // x is b; stop once r.r <= rtol2 * r0.r0
    double rtol2;
};

__device__ __forceinline__ void put(u64 *p, double v) {
    u64 b = (u64)__double_as_longlong(v);
    if (b == kEmpty) b = kNan;
    __hip_atomic_store(p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ u64 get(const u64 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Reads words tid + 512 k, k < COUNT, once all are stored (the arm kernel
// stores zeros in the words nobody stores).  All loads of
// the first round are in flight together; later rounds read what was still
// empty only, so workgroups that wait leave the memory to those that store.
// A uniform base and an opaque 32-bit offset keep the addresses out of the
// vector registers.
template <int COUNT>
__device__ __forceinline__ void wait_for(const u64 *p, unsigned *abort_word, long long limit,
                                         u64 (&t)[COUNT]) {
    const char *base = reinterpret_cast<const char *>(p);
    auto load = [&](int k) {
        unsigned at = 8u * (threadIdx.x + k * kResBlock);
        asm volatile("" : "+v"(at));
        return get(reinterpret_cast<const u64 *>(base + at));
    };
#pragma unroll
    for (int k = 0; k < COUNT; k++) t[k] = load(k);
    long long t0 = 0;
    for (int spin = 1;; spin++) {
        bool all = true;
#pragma unroll
        for (int k = 0; k < COUNT; k++) all = all && t[k] != kEmpty;
        if (__builtin_amdgcn_ballot_w64(!all) == 0) return;  // the whole wavefront goes on
        if ((spin & 15) == 0) {
            if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(
                    abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
                return;
            const long long now = wall_clock64();
            if (t0 == 0) {
                t0 = now;
            } else if (now - t0 > limit) {
                __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                return;
            }
        }
        __builtin_amdgcn_s_sleep(1);
#pragma unroll
        for (int k = 0; k < COUNT; k++)
            if (t[k] == kEmpty) t[k] = load(k);
    }
}

// A value that all lanes hold, in scalar registers.
__device__ __forceinline__ double uniform(double v) { return read_lane(v, 0); }

// Sum of the 8 wave sums, the same bits in every lane.
__device__ __forceinline__ double sum_waves(const double *w) {
    static_assert(kResWaves == 8, "one wave sum per lane of an 8-lane group");
    return uniform(segment_sum<8>(w[threadIdx.x & (kResWaves - 1)]));
}

// LPR lanes per row, PER words per thread (at most 512 PER words), C words a
// chunk, CH chunks a workgroup; the first HELD matrix entries of each lane stay
// in registers (longer rows read the rest from memory in every step).  Bound
// by the exchange: every CU reads all words in every step, about 13 TB/s over
// the chip, and a step has one such round trip.
template <int LPR, int PER, int C, int CH, int HELD>
__global__ __launch_bounds__(kResBlock) void cg_resident_kernel(ResArgs a) {
    extern __shared__ double vec[];  // r (or z) by word; 0 in words without a row
    __shared__ double w_pq[kResWaves], w_rr[kResWaves], row_sum[CH * C];
    static_assert(CH * C * LPR <= kResBlock, "a lane group per row");
    static_assert(kResBlock % C == 0 && (CH == 1 || C == kWave), "a wavefront per chunk");
    static_assert(HELD % 2 == 0, "columns are held in pairs");
    constexpr int kAhead = 8;
    const unsigned gave_up = a.abort_word[1];  // written between launches only: the same for
                                               // every thread
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    // threads 0 .. CH * C - 1 own the workgroup's words; the last word of a
    // chunk is its partial (and so for every word tid + 512 k of this thread)
    const bool partial = (tid & (C - 1)) == C - 1;
    const int word = blockIdx.x * (CH * C) + tid;
    const int row = tid < CH * C ? a.word_row[word] : -1;
    const bool own = row >= 0;
    const int off = __builtin_amdgcn_readfirstlane(a.wave_off[blockIdx.x * kResWaves + wave]);
    const int cnt =
        __builtin_amdgcn_readfirstlane(a.wave_off[blockIdx.x * kResWaves + wave + 1]) - off;
    const double *vp = a.val + (size_t)off * kWave + lane;
    const uint16_t *cp = a.col + (size_t)off * kWave + lane;
    double av[HELD];
    unsigned ac[HELD / 2];
#pragma unroll
    for (int u = 0; u < HELD; u++) av[u] = u < cnt ? vp[u * kWave] : 0.0;
#pragma unroll
    for (int u = 0; u < HELD; u += 2) {
        const unsigned lo = u < cnt ? cp[u * kWave] : 0u;
        const unsigned hi = u + 1 < cnt ? cp[(u + 1) * kWave] : 0u;
        ac[u / 2] = lo | (hi << 16);
    }
    // row_sum[g] = (A vec) of the row of word g of the workgroup
    auto product = [&]() {
        double s = 0.0, s1 = 0.0;
        // groups of 8 entries, 8 LDS reads in flight each
#pragma unroll
        for (int u = 0; u < HELD; u += 8) {
            if (u < cnt) {  // the same for the whole wavefront
                double x[8];
#pragma unroll
                for (int e = 0; e < 8 && u + e < HELD; e += 2) {
                    unsigned c = ac[(u + e) / 2];
                    asm volatile("" : "+v"(c));  // unpacked here, not held unpacked
                    x[e] = vec[c & 0xFFFFu];
                    x[e + 1] = vec[c >> 16];
                }
#pragma unroll
                for (int e = 0; e < 8 && u + e < HELD; e += 2) {
                    s = fma(av[u + e], x[e], s);
                    s1 = fma(av[u + e + 1], x[e + 1], s1);
                }
            }
        }
        for (int u = HELD; u < cnt; u += kAhead) {
            double v[kAhead];
            int c[kAhead];
#pragma unroll
            for (int e = 0; e < kAhead; e++) {
                const int k = min(u + e, cnt - 1) * kWave;
                v[e] = vp[k];
                c[e] = cp[k];
            }
#pragma unroll
            for (int e = 0; e < kAhead; e++) s = fma(u + e < cnt ? v[e] : 0.0, vec[c[e]], s);
        }
        s += s1;
        s = segment_sum<LPR>(s);
        if (tid % LPR == 0 && tid / LPR < CH * C) row_sum[tid / LPR] = s;
        __syncthreads();
    };
    // The sum of v over the rows of a chunk, in its partial's thread.
    auto chunk_sum = [&](double v) { return segment_sum<C>(own ? v : 0.0); };

    u64 *buf = a.xchg;
    double q[PER], xo = 0.0, zo = 0.0, po = 0.0, qo = 0.0, ro = 0.0;
    double xscale = a.scale_first ? uniform(a.sc->xscale) : 1.0;
    const double *src = a.scale_first ? a.z : a.x;
    // r = x = xscale * z of the previous call, or x itself
    double rr = 0.0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int w = tid + k * kResBlock;
        const int j = w < a.words ? a.word_row[w] : -1;
        const double v = j >= 0 ? xscale * src[j] : 0.0;
        vec[w] = v;
        rr += v * v;
    }
    if (own) xo = xscale * src[row];
    asm volatile("" ::: "memory");  // the loads are on their way
    if (gave_up) return;
    int k = 0;
    double rho = 0.0, rho0 = 0.0;
    for (int it = 0; it < a.niter; it++) {
        po = qo = zo = 0.0;
#pragma unroll
        for (int e = 0; e < PER; e++) q[e] = 0.0;
        double alpha = 1.0, rho_prev = 1.0;
        __syncthreads();  // vec is written
        for (k = 0; k < a.steps; k++) {
            product();
            double so = 0.0;
            if (tid < CH * C) {
                if (own) {
                    ro = vec[word];
                    so = row_sum[tid];
                }
                const double rs = chunk_sum(ro * so);
                if (own || partial) put(buf + word, own ? so : rs);
            }
            // while the words travel: rho = r.r, beta, and p.q less r.s
            rr = segment_sum<64>(rr);
            if (lane == 0) w_rr[wave] = rr;
            __syncthreads();
            rho = sum_waves(w_rr);
            double beta = 0.0, less = 0.0;
            if (k == 0) {
                rho0 = rho;
            } else {
                beta = uniform(rho / rho_prev);
                less = uniform(beta * (rho / alpha));
                if (a.solve && fabs(rho) <= a.rtol2 * fabs(rho0)) {
                    buf += a.stride;
                    break;  // the same decision in every workgroup
                }
            }
            u64 t[PER];
            wait_for<PER>(buf, a.abort_word, a.spin_limit, t);
            double rs = 0.0;
            if (partial) {
                double s1 = 0.0;
#pragma unroll
                for (int e = 0; e < PER; e++) {
                    if (e & 1)
                        s1 += __longlong_as_double((long long)t[e]);
                    else
                        rs += __longlong_as_double((long long)t[e]);
                }
                rs += s1;
            }
            rs = segment_sum<64>(rs);
            if (lane == 0) w_pq[wave] = rs;
#pragma unroll
            for (int e = 0; e < PER; e++)
                q[e] = __longlong_as_double((long long)t[e]) + beta * q[e];
            __syncthreads();
            alpha = uniform(rho / (sum_waves(w_pq) - less));
            po = ro + beta * po;
            qo = so + beta * qo;
            zo += alpha * po;
            const double step = partial ? 0.0 : alpha;
            rr = 0.0;
            double rr1 = 0.0;
#pragma unroll
            for (int e = 0; e < PER; e++) {
                const double v = vec[tid + e * kResBlock] - step * q[e];
                vec[tid + e * kResBlock] = v;
                if (e & 1)
                    rr1 += v * v;
                else
                    rr += v * v;
            }
            rr += rr1;
            rho_prev = rho;
            buf += a.stride;
            __syncthreads();
        }
        if (!a.solve && k > 0) {  // p = r + beta p closing the last step
            rr = segment_sum<64>(rr);
            if (lane == 0) w_rr[wave] = rr;
            __syncthreads();
            rho = sum_waves(w_rr);
            if (own) po = vec[word] + rho / rho_prev * po;
        }
        // every workgroup gets z and z.z; r = A z on the own rows
        if (tid < CH * C) {
            const double zz = chunk_sum(zo * zo);
            if (own || partial) put(buf + word, own ? zo : zz);
        }
        u64 t[PER];
        wait_for<PER>(buf, a.abort_word, a.spin_limit, t);
        buf += a.stride;
        __syncthreads();  // vec has been read
        double zz = 0.0;
#pragma unroll
        for (int e = 0; e < PER; e++) {
            const double v = __longlong_as_double((long long)t[e]);
            vec[tid + e * kResBlock] = partial ? 0.0 : v;
            zz += partial ? v : 0.0;
        }
        zz = segment_sum<64>(zz);
        if (lane == 0) w_pq[wave] = zz;
        __syncthreads();
        zz = sum_waves(w_pq);
        product();
        if (tid < CH * C) {
            if (own) ro = row_sum[tid];
            const double d = xo - ro;
            const double e0 = chunk_sum(d * d), e1 = chunk_sum(xo * zo);
            if (partial) {
                const int chunks = gridDim.x * CH;
                double *pt = a.part + (size_t)it * 2 * chunks;
                pt[word / C] = e0;
                pt[chunks + word / C] = e1;
            }
        }
        if (blockIdx.x == 0 && tid == 0) a.zz[it] = zz;
        if (it + 1 < a.niter) {  // the next outer iteration starts from z / ||z||
            xscale = uniform(1.0 / sqrt(zz));
            xo = xscale * zo;
            rr = 0.0;
#pragma unroll
            for (int e = 0; e < PER; e++) {
                const double v = xscale * vec[tid + e * kResBlock];
                vec[tid + e * kResBlock] = v;
                rr += v * v;
            }
        }
    }
    if (own) {
        a.z[row] = zo;
        a.p[row] = po;
        a.q[row] = qo;
        a.r[row] = ro;
    }
    if (a.solve && blockIdx.x == 0 && tid == 0) {
        a.sc->steps = k;
        a.sc->rho = rho;
        a.sc->bb = rho0;
        a.sc->tol2 = a.rtol2 * fabs(rho0);
        a.sc->rtol2 = a.rtol2;
        a.sc->stop_enabled = 1;
    }
}

// Before a launch: every word that will be stored empty, the others zero; the
// abort words clear before the first launch of a call, else what the launches
// before left.  hole: a word of the first buffer left empty though nobody stores
// it, so that the launch gives up (-1: none).
__global__ __launch_bounds__(kBlock) void resident_arm_kernel(
    u64 *xchg, const int *__restrict__ word_row, int words, int chunk, int stride, int buffers,
    int hole, int clear, unsigned *abort_word) {
    const int per = stride / 2;  // 16-byte pairs of a buffer
    ulonglong2 *x2 = reinterpret_cast<ulonglong2 *>(xchg);
    auto first = [&](int w) {  // a row, or the partial of a chunk
        return w < words && (word_row[w] >= 0 || (w & (chunk - 1)) == chunk - 1) ? kEmpty : 0ull;
    };
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < per; i += gridDim.x * kBlock) {
        const ulonglong2 v = make_ulonglong2(first(2 * i), first(2 * i + 1));
        for (int b = blockIdx.y; b < buffers; b += gridDim.y)
            x2[(size_t)b * per + i] = b == 0 && i == hole >> 1 ? make_ulonglong2(kEmpty, kEmpty) : v;
    }
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
        if (clear) abort_word[0] = 0u;
        abort_word[1] = abort_word[0];
    }
}

// After a launch, one workgroup per outer iteration: rnorm = ||x - A z||,
// zeta = shift + 1 / (x.z) and the scale 1 / sqrt(z.z) (cg.cu:505-514), as
// resid_finish_kernel records them; index n as cg.cu:671-676 leaves it.
__global__ __launch_bounds__(kBlock) void resident_finish_kernel(
    const double *__restrict__ part, int count, const double *__restrict__ zz, int niter,
    Scalars *sc, double *__restrict__ zeta_hist, double *__restrict__ rnorm_hist, int hist_cap,
    int first, int record, const unsigned *__restrict__ abort_word, const double *__restrict__ x,
    double *__restrict__ z, double *__restrict__ p, double *__restrict__ q,
    double *__restrict__ r, int n) {
    const int it = blockIdx.x;
    if (abort_word[0]) {  // of this launch or an earlier one: nothing here is valid
        if (it == 0 && threadIdx.x == 0) sc->aborted = 1;
        return;
    }
    const double *pt = part + (size_t)it * 2 * count;
    double s0, s1;
    reduce_partials2<kBlock>(pt, count, pt + count, count, s0, s1);
    if (threadIdx.x != 0) return;
    const double rnorm = sqrt(s0);
    const double zeta = sc->shift + 1.0 / s1;
    if (record && first + it < hist_cap) {
        zeta_hist[first + it] = zeta;
        rnorm_hist[first + it] = rnorm;
    }
    if (it + 1 < niter) return;
    sc->rnorm = rnorm;
    sc->xz = s1;
    sc->zz = zz[it];
    sc->xscale = 1.0 / sqrt(zz[it]);
    sc->zeta = zeta;
    if (record) sc->iter = first + niter;
    sc->aborted = 0;
    const double xn = x[n];
    q[n] = 0.0;
    z[n] = 0.0;
    r[n] = xn;
    p[n] = xn;
}

// Entry u of lane sl of the group of word g: the row's entry sl + u LPR (its
// column as a word), or (0, 0) past its end.
__global__ __launch_bounds__(kResBlock) void resident_fill_kernel(
    const int *__restrict__ rowstr, const int *__restrict__ colidx, const double *__restrict__ a,
    const int *__restrict__ wave_off, const int *__restrict__ word_row,
    const int *__restrict__ row_word, int words_wg, int lpr, double *__restrict__ val,
    uint16_t *__restrict__ col) {
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int g = tid / lpr;
    const int row = g < words_wg ? word_row[blockIdx.x * words_wg + g] : -1;
    const int s = row >= 0 ? rowstr[row] : 0, e = row >= 0 ? rowstr[row + 1] : 0;
    const int off = wave_off[blockIdx.x * kResWaves + wave];
    const int cnt = wave_off[blockIdx.x * kResWaves + wave + 1] - off;
    for (int u = 0; u < cnt; u++) {
        const int k = s + tid % lpr + u * lpr;
        const size_t at = (size_t)(off + u) * kWave + lane;
        val[at] = k < e ? a[k] : 0.0;
        col[at] = k < e ? (uint16_t)row_word[colidx[k]] : (uint16_t)0;
    }
}

// Kernels by words per thread, smallest first.  Few words a thread go with
// many lanes per row: the fewer rows a workgroup has, the more lanes each
// gets, and all of them still find a place in one pass.  A step grows with the
// words a thread reads in the exchange, whether they are rows or not, by
// 0.06 to 0.15 us a word, so there is a kernel for every second word
// count and every one up to 8; as many entries are held as leave no spills.  With
// 4, 8, 16, 32 and 38 words only, and now, us a step: n = 1400 2.02 and 1.94, 2000
// 2.50 and 2.16, 4500 3.45 and 2.81, 8100 6.48 and 4.52, 10000 6.91 and 5.26, 14000
// 6.72 and 6.35, 17000 9.44 and 8.55.
struct ResKernel {
    int lpr, per, chunk, chunks;  // as the kernel's template
    const void *fn;
};
template <int LPR, int PER, int C, int CH, int HELD>
ResKernel res_kernel() {
    return {LPR, PER, C, CH,
            reinterpret_cast<const void *>(&cg_resident_kernel<LPR, PER, C, CH, HELD>)};
}
const ResKernel kResKernels[] = {
    res_kernel<32, 2, 16, 1, 8>(),   res_kernel<32, 3, 16, 1, 8>(),
    res_kernel<32, 4, 16, 1, 8>(),   res_kernel<32, 5, 16, 1, 12>(),
    res_kernel<32, 6, 16, 1, 12>(),  res_kernel<32, 7, 16, 1, 12>(),
    res_kernel<32, 8, 16, 1, 12>(),  res_kernel<16, 10, 32, 1, 24>(),
    res_kernel<16, 12, 32, 1, 24>(), res_kernel<16, 14, 32, 1, 24>(),
    res_kernel<16, 16, 32, 1, 24>(), res_kernel<8, 18, 64, 1, 24>(),
    res_kernel<8, 20, 64, 1, 24>(),  res_kernel<8, 22, 64, 1, 24>(),
    res_kernel<8, 24, 64, 1, 24>(),  res_kernel<8, 26, 64, 1, 20>(),
    res_kernel<8, 28, 64, 1, 20>(),  res_kernel<8, 30, 64, 1, 16>(),
    res_kernel<8, 32, 64, 1, 16>(),  res_kernel<4, 34, 64, 2, 8>(),
    res_kernel<4, 36, 64, 2, 8>(),   res_kernel<4, 38, 64, 2, 8>(),
};

}  // namespace

bool resident_shape(int n, const int *rowstr, int cus, int lds_cap, ResidentShape *out) {
    if (n < 1) return false;
    for (int i = 0; i < (int)(sizeof(kResKernels) / sizeof(kResKernels[0])); i++) {
        const ResKernel &rk = kResKernels[i];
        const int rows_chunk = rk.chunk - 1, chunks = (n + rows_chunk - 1) / rows_chunk;
        const int grid = (chunks + rk.chunks - 1) / rk.chunks;
        const int words_wg = rk.chunk * rk.chunks, words = grid * words_wg;
        const int lds = rk.per * kResBlock * 8;
        if (words > rk.per * kResBlock || grid > cus || lds + 2048 > lds_cap) continue;
        ResidentShape &s = *out;
        s.kernel = i;
        s.grid = grid;
        s.lpr = rk.lpr;
        s.chunk = rk.chunk;
        s.words_wg = words_wg;
        s.words = words;
        s.lds_bytes = lds;
        s.stride = rk.per * kResBlock;
        // Rows by length, longest first, dealt out to the workgroups in turn:
        // every workgroup gets the same mix, and the rows of one wavefront,
        // padded to its longest, are of like length.
        int longest = 0;
        for (int j = 0; j < n; j++) longest = std::max(longest, rowstr[j + 1] - rowstr[j]);
        std::vector<int> at((size_t)longest + 2, 0), order((size_t)n);
        for (int j = 0; j < n; j++) at[longest - (rowstr[j + 1] - rowstr[j]) + 1]++;
        for (int l = 0; l <= longest; l++) at[l + 1] += at[l];
        for (int j = 0; j < n; j++) order[at[longest - (rowstr[j + 1] - rowstr[j])]++] = j;
        s.word_row.assign((size_t)words, -1);
        s.row_word.assign((size_t)n, 0);
        int next = 0;
        for (int g = 0; g < words_wg; g++) {
            if (g % rk.chunk == rk.chunk - 1) continue;  // the partial
            for (int wg = 0; wg < grid && next < n; wg++, next++) {
                s.word_row[(size_t)wg * words_wg + g] = order[next];
                s.row_word[order[next]] = wg * words_wg + g;
            }
        }
        // entries of each wavefront: its longest row, shared by lpr lanes
        const int per_wave = kWave / rk.lpr;
        s.wave_off.assign((size_t)grid * kResWaves + 1, 0);
        long long total = 0;
        for (int w = 0; w < grid * kResWaves; w++) {
            int most = 0;
            for (int e = 0; e < per_wave; e++) {
                const int g = w % kResWaves * per_wave + e;
                const int j = g < words_wg ? s.word_row[(size_t)(w / kResWaves) * words_wg + g] : -1;
                if (j >= 0) most = std::max(most, rowstr[j + 1] - rowstr[j]);
            }
            const int cnt = (most + rk.lpr - 1) / rk.lpr;
            if (cnt > kResidentMaxEntries) return false;
            total += cnt;
            s.wave_off[(size_t)w + 1] = (int)total;
        }
        return true;
    }
    return false;
}

hipError_t resident_capacity(const ResidentShape &s, int *per_cu) {
    const void *fn = kResKernels[s.kernel].fn;
    hipError_t e =
        hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, s.lds_bytes);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, fn, kResBlock,
                                                        (size_t)s.lds_bytes);
}

size_t resident_partials(const ResidentShape &s, int niter) {
    return (size_t)niter * (2 * (size_t)(s.words / s.chunk) + 1);
}

hipError_t launch_resident_fill(const Fp64Problem &pb, const ResidentShape &s,
                                const ResidentState &rs, hipStream_t st) {
    resident_fill_kernel<<<s.grid, kResBlock, 0, st>>>(pb.rowstr, pb.colidx, pb.a, rs.wave_off,
                                                       rs.word_row, rs.row_word, s.words_wg,
                                                       s.lpr, rs.val, rs.col);
    return hipGetLastError();
}

hipError_t launch_resident(const Fp64Problem &pb, const ResidentShape &s, const ResidentState &rs,
                           int steps, int niter, int scale_first, int first, int record,
                           int solve, double rtol, hipStream_t st) {
    ResArgs a{};
    a.val = rs.val;
    a.col = rs.col;
    a.wave_off = rs.wave_off;
    a.n = pb.n;
    a.words = s.words;
    a.word_row = rs.word_row;
    a.stride = s.stride;
    a.xchg = reinterpret_cast<u64 *>(rs.xchg);
    a.abort_word = rs.abort_word;
    a.spin_limit = rs.spin_limit;
    a.x = pb.x;
    a.z = pb.z;
    a.p = pb.p;
    a.q = pb.q;
    a.r = pb.r;
    const int count = s.words / s.chunk;
    a.part = rs.part;
    a.zz = rs.part + (size_t)niter * 2 * count;
    a.sc = pb.sc;
    a.steps = steps;
    a.niter = niter;
    a.scale_first = scale_first;
    a.solve = solve;
    a.rtol2 = rtol * rtol;
    const int buffers = niter * (steps + 1);
    int hole = -1;
    if (rs.give_up_at >= first && rs.give_up_at < first + niter) {  // (tests)
        hole = s.words;
        a.spin_limit = rs.spin_limit / 100;
    }
    resident_arm_kernel<<<dim3(std::min(8, s.stride / (2 * kBlock)), std::min(buffers, 256)),
                          kBlock, 0, st>>>(a.xchg, rs.word_row, s.words, s.chunk, s.stride,
                                           buffers, hole, first == 0 ? 1 : 0, rs.abort_word);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (pb.marks) pb.marks->note("resident_arm_kernel", kBlock, st);
    void *args[] = {&a};
    e = hipLaunchKernel(kResKernels[s.kernel].fn, dim3(s.grid), dim3(kResBlock), args,
                        (size_t)s.lds_bytes, st);
    if (e != hipSuccess) return e;
    if (pb.marks) pb.marks->note("cg_resident_kernel", kResBlock, st);
    resident_finish_kernel<<<niter, kBlock, 0, st>>>(
        rs.part, count, a.zz, niter, pb.sc, pb.zeta_hist, pb.rnorm_hist, pb.hist_cap, first,
        record, rs.abort_word, pb.x, pb.z, pb.p, pb.q, pb.r, pb.n);
    e = hipGetLastError();
    if (e == hipSuccess && pb.marks) pb.marks->note("resident_finish_kernel", kBlock, st);
    return e;
}

}  // namespace npbcg_dev
