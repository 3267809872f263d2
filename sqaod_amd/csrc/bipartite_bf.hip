/*
 * Bipartite brute-force search: E(x0, x1) = b0.x0 + b1.x1 + x1^T W x0 over a
 * rectangle of (x0, x1) pairs (calculate_E_2d, SharedFormulas.cpp:123-144),
 * keeping the minimum and the pairs that reach it.  The list semantics are
 * one sqaod.cpu worker's (CPUBipartiteGraphBatchSearch.cpp:29-62 driven by
 * searchRangeSingleThread, CPUBipartiteGraphBFSearcher.cpp:166-198): pairs
 * are met in the order (x0 / T0, x1, x0 % T0) with T0 the x0 tile size, a
 * strictly lower E restarts the list and an equal E appends while the list
 * holds fewer than N0 + N1 pairs -- so the list is the N0 + N1 smallest
 * visiting keys among the minimisers.
 *
 * For a fixed x1, E is linear in x0:  E = B(x1) + sum_{pos in x0} d_pos(x1)
 * with d_pos = b0[pos] + sum_{i in x1} W[i][pos] and B = b1.x1.  Split x0 =
 * (xH, xL) with xL its low L = min(N0, 10) bits (bit N0-1-pos of a packed x
 * is x[pos], Common.cpp:79-86): E = (B + SH(xH)) + TL(xL), both subset sums
 * of d, taken from the lowest bit up, formed in double and rounded to the
 * solver's real once.
 *
 * The least E over x0 is that of the x0 holding exactly the positions with
 * d < 0 (in a rectangle of high patterns: among the bits that vary there), not
 * only in exact sums but in the rounded ones: going up the bits, that x0's
 * partial sum stays the least, because rounded addition is monotone and leaves
 * s + d <= s for d < 0.  So a rectangle's scan costs N0 N1 additions per x1
 * instead of 2^N0, and is bound by its launch and the read-back of its minimum
 * (16 x 16, per 4096 x1: 7.2 us against 93.3 us for all 2^16 x0 of each).
 *
 *   bgScan   : a block per 64 x1, four waves sharing the positions: each x1's
 *              least E over the rectangle's x0.
 *   bgSelect : for each x1 whose least E is the range minimum, blocks of 16
 *              high patterns append their first K minimisers in ascending x0
 *              (for a fixed x1 that is the visiting order); high patterns whose
 *              own least E is another are passed over.
 * The host merges the lists by visiting key.
 */
#include <cfloat>

#include "common.h"
#include "kernels.h"

namespace sqaod_rocm {

namespace {

constexpr int kThreads = 256;
constexpr int kScanThreads = 4 * kBGBFScanBlock; /* a rectangle is at most 4096 x1: 64 blocks */
constexpr int kLowMax = 10;
constexpr int kMaxN = 63;

struct BGBlockTables {
    double d[64];
    double SH[kBGBFHighPerBlock];
    double B, TLmin;
};

template <class real>
__device__ void buildBlock(const BGBFArgs &a, const real *b0, const real *b1, const real *W, BGBlockTables &t,
                           unsigned long long x1, unsigned long long xH0) {
    const int N0 = a.N0, N1 = a.N1;
    if ((int)threadIdx.x < N0) {
        const int pos = threadIdx.x;
        double s = a.sgn * (double)b0[pos];
        for (int i = 0; i < N1; ++i)
            if ((x1 >> (N1 - 1 - i)) & 1ull)
                s += a.sgn * (double)W[(size_t)i * N0 + pos];
        t.d[pos] = s;
    }
    if (threadIdx.x == 0) {
        double s = 0.;
        for (int i = 0; i < N1; ++i)
            if ((x1 >> (N1 - 1 - i)) & 1ull)
                s += a.sgn * (double)b1[i];
        t.B = s;
    }
    __syncthreads();
    if (threadIdx.x == 64) {
        double s = 0.;
        for (int b = 0; b < a.L; ++b)
            if (t.d[N0 - 1 - b] < 0.)
                s += t.d[N0 - 1 - b];
        t.TLmin = s;
    }
    if ((int)threadIdx.x < kBGBFHighPerBlock) {
        const unsigned long long xH = xH0 + threadIdx.x;
        double s = 0.;
        for (int b = 0; b < a.nH; ++b)
            if ((xH >> b) & 1ull)
                s += t.d[N0 - 1 - (a.L + b)];
        t.SH[threadIdx.x] = s;
    }
    __syncthreads();
}

/* TL of the low pattern xL */
__device__ __forceinline__ double lowSum(const BGBFArgs &a, const BGBlockTables &t, int xL) {
    double s = 0.;
    for (int b = 0; b < a.L; ++b)
        if ((xL >> b) & 1)
            s += t.d[a.N0 - 1 - b];
    return s;
}

template <class real>
__device__ __forceinline__ real pairEnergy(const BGBlockTables &t, int r, double tl) {
    return (real)((t.B + t.SH[r]) + tl);
}

template <class real>
__global__ __launch_bounds__(kScanThreads) void bgScanKernel(BGBFArgs a, const real *b0, const real *b1, const real *W,
                                                             real *x1Min, real *blockMin,
                                                             unsigned long long *nPairs) {
    __shared__ double sW[kMaxN * kMaxN];
    __shared__ double sd[kMaxN][kBGBFScanBlock]; /* d by bit of x0 */
    __shared__ double sb0[kMaxN], sb1[kMaxN];
    const int lane = threadIdx.x % kBGBFScanBlock, w = threadIdx.x / kBGBFScanBlock;
    const int N0 = a.N0, N1 = a.N1;
    for (int i = threadIdx.x; i < N0 * N1; i += kScanThreads)
        sW[i] = a.sgn * (double)W[i];
    if ((int)threadIdx.x < N0)
        sb0[threadIdx.x] = a.sgn * (double)b0[threadIdx.x];
    if ((int)threadIdx.x < N1)
        sb1[threadIdx.x] = a.sgn * (double)b1[threadIdx.x];
    if (blockIdx.x == 0 && threadIdx.x == 0)
        *nPairs = 0;
    __syncthreads();
    const unsigned long long i1 = (unsigned long long)blockIdx.x * kBGBFScanBlock + lane;
    const unsigned long long x1 = a.x1b + (i1 < a.nX1 ? i1 : a.nX1 - 1);
    const unsigned long long varying = a.he - a.hb - 1; /* the high bits that vary (hb is a multiple of he - hb) */
    for (int bit0 = 4 * w; bit0 < N0; bit0 += 16) { /* four positions at a time: independent chains */
        double d[4];
        int pos[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            pos[k] = bit0 + k < N0 ? N0 - 1 - bit0 - k : 0;
            d[k] = sb0[pos[k]];
        }
        for (int i = 0; i < N1; ++i) {
            const bool on = (x1 >> (N1 - 1 - i)) & 1ull;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double v = d[k] + sW[i * N0 + pos[k]];
                d[k] = on ? v : d[k];
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (bit0 + k < N0)
                sd[bit0 + k][lane] = d[k];
    }
    __syncthreads();
    if (w != 0)
        return;
    double B = 0.;
    for (int i = 0; i < N1; ++i) {
        const double v = B + sb1[i];
        B = ((x1 >> (N1 - 1 - i)) & 1ull) ? v : B;
    }
    double SH = 0., TL = 0.;
    for (int bit = 0; bit < a.L; ++bit) {
        const double d = sd[bit][lane];
        TL = d < 0. ? TL + d : TL;
    }
    for (int bit = a.L; bit < N0; ++bit) {
        const double d = sd[bit][lane];
        const bool take = ((varying >> (bit - a.L)) & 1ull) ? d < 0. : ((a.hb >> (bit - a.L)) & 1ull);
        SH = take ? SH + d : SH;
    }
    const real e = (real)((B + SH) + TL);
    real mn = e < (real)FLT_MAX ? e : (real)FLT_MAX;
    if (i1 < a.nX1)
        x1Min[i1] = mn;
    for (int off = 32; off > 0; off >>= 1) {
        const real o = __shfl_xor(mn, off);
        mn = o < mn ? o : mn;
    }
    if (threadIdx.x == 0) /* host memory */
        __hip_atomic_store(&blockMin[blockIdx.x], mn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
static_assert(kBGBFScanBlock == 64, "a lane per x1");

template <class real>
__global__ __launch_bounds__(kThreads) void bgSelectKernel(BGBFArgs a, const real *b0, const real *b1, const real *W,
                                                           const real *x1Min, real Emin, unsigned long long nItems,
                                                           unsigned long long *pairs, unsigned long long *nPairs) {
    __shared__ BGBlockTables t;
    __shared__ int wsum[kThreads / 64];
    __shared__ int base, nHit;
    __shared__ unsigned short hit[kThreads];
    __shared__ unsigned long long found[2 * kMaxN], at;
    /* items (x1, 16 high patterns), 256 a block */
    const unsigned long long item0 = (unsigned long long)blockIdx.x * kThreads;
    if (threadIdx.x == 0)
        nHit = 0;
    __syncthreads();
    if (item0 + threadIdx.x < nItems && x1Min[(item0 + threadIdx.x) % a.nX1] == Emin)
        hit[atomicAdd(&nHit, 1)] = (unsigned short)threadIdx.x;
    __syncthreads();
    const int n = nHit, nL = 1 << a.L;
    const int lane = threadIdx.x & 63, w = threadIdx.x / 64;
    for (int h = 0; h < n; ++h) {
        const unsigned long long item = item0 + hit[h];
        const unsigned long long x1 = a.x1b + item % a.nX1, xH0 = a.hb + item / a.nX1 * kBGBFHighPerBlock;
        buildBlock<real>(a, b0, b1, W, t, x1, xH0);
        if (threadIdx.x == 0)
            base = 0;
        __syncthreads();
        const int nR = (int)((a.he - xH0) < (unsigned long long)kBGBFHighPerBlock ? (a.he - xH0) : kBGBFHighPerBlock);
        /* ascending x0 = (r, xL): r outer, then xL = k * 256 + t (k outer, t inner) */
        for (int r = 0; r < nR && base < a.K; ++r) {
            if (pairEnergy<real>(t, r, t.TLmin) != Emin) /* the least of these 2^L */
                continue;
            for (int k0 = 0; k0 < nL; k0 += kThreads) {
                const int xL = k0 + (int)threadIdx.x;
                bool tie = false;
                if (xL < nL)
                    tie = pairEnergy<real>(t, r, lowSum(a, t, xL)) == Emin;
                const unsigned long long bal = __ballot(tie);
                if (lane == 0)
                    wsum[w] = __popcll(bal);
                __syncthreads();
                int before = base;
                for (int v = 0; v < w; ++v)
                    before += wsum[v];
                const int pos = before + __popcll(bal & ((1ull << lane) - 1ull));
                if (tie && pos < a.K)
                    found[pos] = ((xH0 + (unsigned long long)r) << a.L) | (unsigned long long)xL;
                __syncthreads();
                if (threadIdx.x == 0) {
                    int tot = 0;
                    for (int v = 0; v < kThreads / 64; ++v)
                        tot += wsum[v];
                    base += tot;
                }
                __syncthreads();
                if (base >= a.K)
                    break;
            }
        }
        const int nFound = base < a.K ? base : a.K;
        if (threadIdx.x == 0)
            at = atomicAdd(nPairs, (unsigned long long)nFound);
        __syncthreads();
        if ((int)threadIdx.x < nFound) {
            pairs[2 * (at + threadIdx.x)] = found[threadIdx.x];
            pairs[2 * (at + threadIdx.x) + 1] = x1;
        }
        __syncthreads();
    }
}

}  // namespace

BGBFArgs bgBFPlan(int N0, int N1) {
    BGBFArgs a{};
    a.N0 = N0;
    a.N1 = N1;
    a.L = N0 < kLowMax ? N0 : kLowMax;
    a.nH = N0 - a.L;
    a.K = N0 + N1;
    return a;
}

template <class real>
void bgBFScan(const BGBFArgs &a, const real *d_b0, const real *d_b1, const real *d_W, real *d_x1Min,
              real *d_blockMin, unsigned long long *d_nPairs, hipStream_t stream) {
    SQ_THROW_IF(a.N0 < 1 || a.N0 > kMaxN || a.N1 < 1 || a.N1 > kMaxN || a.L != (a.N0 < kLowMax ? a.N0 : kLowMax),
                "bipartite BF: bad plan");
    SQ_THROW_IF(a.he <= a.hb || a.nX1 == 0 || a.x1b + a.nX1 > (1ull << a.N1) || a.he > (1ull << a.nH),
                "bipartite BF: bad range");
    const unsigned long long nHigh = a.he - a.hb;
    SQ_THROW_IF((nHigh & (nHigh - 1)) != 0 || a.hb % nHigh != 0, "bipartite BF: high patterns are not an aligned run");
    bgScanKernel<real><<<(unsigned)bgBFScanBlocks(a), kScanThreads, 0, stream>>>(a, d_b0, d_b1, d_W, d_x1Min,
                                                                                d_blockMin, d_nPairs);
    HIP_CHECK(hipGetLastError());
}

template <class real>
void bgBFSelect(const BGBFArgs &a, const real *d_b0, const real *d_b1, const real *d_W, const real *d_x1Min,
                real Emin, unsigned long long *d_pairs, unsigned long long *d_nPairs, hipStream_t stream) {
    const unsigned long long n = bgBFItems(a);
    bgSelectKernel<real><<<(unsigned)((n + kThreads - 1) / kThreads), kThreads, 0, stream>>>(
        a, d_b0, d_b1, d_W, d_x1Min, Emin, n, d_pairs, d_nPairs);
    HIP_CHECK(hipGetLastError());
}

unsigned long long bgBFItems(const BGBFArgs &a) {
    return a.nX1 * ((a.he - a.hb + kBGBFHighPerBlock - 1) / kBGBFHighPerBlock);
}
unsigned long long bgBFScanBlocks(const BGBFArgs &a) { return (a.nX1 + kBGBFScanBlock - 1) / kBGBFScanBlock; }

template void bgBFScan<float>(const BGBFArgs &, const float *, const float *, const float *, float *, float *,
                              unsigned long long *, hipStream_t);
template void bgBFScan<double>(const BGBFArgs &, const double *, const double *, const double *, double *, double *,
                               unsigned long long *, hipStream_t);
template void bgBFSelect<float>(const BGBFArgs &, const float *, const float *, const float *, const float *, float,
                                unsigned long long *, unsigned long long *, hipStream_t);
template void bgBFSelect<double>(const BGBFArgs &, const double *, const double *, const double *, const double *,
                                 double, unsigned long long *, unsigned long long *, hipStream_t);

}  // namespace sqaod_rocm
