/*
 * Dense brute-force search: E(x) = x^T W x over every x in [xb, xe), keeping
 * the minimum and the ascending list of the x that reach it.  The semantics
 * are those of one sqaod.cpu batch searcher (CPUDenseGraphBatchSearch.cpp:
 * 26-50) and of the CUDA device's tile merge (CUDADenseGraphBFSearcher.cpp:
 * 155-185): a strictly lower minimum replaces the list, an equal one appends,
 * and the list keeps the first `cap` (= tile size) x in ascending order.
 *
 * Bit t of the packed x is x[N-1-t] (Common.cpp:79-93); V[t][u] =
 * W[N-1-t][N-1-u].  The bits are split, from the lowest, into b (5 bits), a
 * (7), c (up to 5) and the high rest H:
 *   E(x) = ((EL(a,b) + g_H(b)) + f_H(a)) + G(c,b)          = X(a,b) + G(c,b)
 *        + (Y(c,a) + S_H(c))
 * with EL the energy of the bits below 12, G and Y the cross sums
 * 2 sum V over set bits of c and b / a, g_H and f_H the same of H with b / a
 * (f_H with H's own energy), and S_H(c) the energy of c and its cross sum with
 * H.  EL, G, Y and the energies of c do not depend on H: bfTablesKernel forms
 * them once a search.  A unit is one H, i.e. a run of 2^(12 + |c|) consecutive
 * x, and a block scans it: lane L holds the 2 x 32 values X(L, .) and
 * X(64 + L, .) in registers, and for each c, shared out over the four waves,
 * takes the least X(a,b) + G(c,b) over b -- G(c, .) is the same in all lanes,
 * read from LDS once for both rows -- plus Y + S.  A candidate thus costs one
 * double add and one minimum, a row of 32 three operations more.  Adding Y + S
 * to the least of a row gives the least of the sums (rounded addition is
 * monotone), so the scan and the select, which evaluates each candidate of a
 * row in this order, agree bit for bit.  Sums are formed in double and rounded
 * to the solver's real once.
 *
 * What bounds it: FP64 adds and minima at 16 lanes a cycle and SIMD (2^30
 * candidates: 58 us), and per span of 2^26 candidates the launches and the
 * chain of memory round trips of a block's set-up.  Measured: 17.3 us a span
 * (against 101 us for three LDS reads and three adds a candidate with tables of
 * 2^12 low energies built by every block), 9.5 us for a whole search at N=20
 * (49 us); the select 6.7 us a span on average, most with nothing to list
 * (24 us).  Read as scalar loads instead of from LDS, G made it 20.8 us: each
 * value of c then waits for its own round trip.
 *
 *   bfScan   : per unit its min E; the block that ends last finds the range
 *              minimum, applies the list rule and lists the units holding it.
 *   bfSelect : each listed unit counts its minimisers, takes its place in the
 *              list from the unit before it and writes them in ascending order.
 * Nothing is read back to the host between ranges.
 */
#include <cfloat>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace sqaod_rocm {

namespace {

constexpr int kThreads = 256;
constexpr int kWave = 64;
constexpr int kWaves = kThreads / kWave;
constexpr int kSelBlocks = 128;
constexpr int kB = 5, kA = 7, kCMax = 5; /* bits of b, a and (at most) c */
constexpr int kRows = (1 << kA) / kWave;   /* rows of a lane: a = 64 row + lane */
constexpr int kNB = 1 << kB, kNA = 1 << kA, kNC = 1 << kCMax;
constexpr int kLowBits = kB + kA + kCMax;

/* the tables in global memory, in doubles */
constexpr int kTabEL = 0;                     /* [b][a] */
constexpr int kTabG = kTabEL + kNB * kNA;     /* [c][b] */
constexpr int kTabY = kTabG + kNC * kNB;      /* [c][a] */
constexpr int kTabEC = kTabY + kNC * kNA;     /* [c] */
static_assert(kTabEC + kNC == kBFTableDoubles, "table layout");

/* the energy of the set bits of x among bits [t0, t0 + n), and twice the sum
 * of V over pairs of a bit of x (bits t0..) and a bit of z (bits u0..) */
__device__ double energyOf(const double (*V)[kLowBits], int x, int t0, int n) {
    double e = 0.;
    for (int i = 0; i < n; ++i) {
        if (!((x >> i) & 1))
            continue;
        double s = 0.;
        for (int k = 0; k < n; ++k)
            if ((x >> k) & 1)
                s += V[t0 + i][t0 + k];
        e += s;
    }
    return e;
}
__device__ double crossOf(const double (*V)[kLowBits], int x, int t0, int n, int z, int u0, int nz) {
    double e = 0.;
    for (int i = 0; i < n; ++i) {
        if (!((x >> i) & 1))
            continue;
        double s = 0.;
        for (int k = 0; k < nz; ++k)
            if ((z >> k) & 1)
                s += V[t0 + i][u0 + k];
        e += s;
    }
    return 2. * e;
}

/* One thread per table entry.  Bits past N - 1 do not exist: patterns of b
 * and a that would set them get an infinite EL. */
__global__ __launch_bounds__(kThreads) void bfTablesKernel(const double *W, BFPlan p, double *tab) {
    __shared__ double V[kLowBits][kLowBits];
    for (int i = threadIdx.x; i < kLowBits * kLowBits; i += kThreads) {
        const int t = i / kLowBits, u = i % kLowBits;
        V[t][u] = (t < p.N && u < p.N) ? W[(size_t)(p.N - 1 - t) * p.N + (p.N - 1 - u)] : 0.;
    }
    __syncthreads();
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i < kTabG) {
        const int b = i / kNA, a = i % kNA, x = (a << kB) | b;
        tab[i] = (p.N < kB + kA && (x >> p.N)) ? HUGE_VAL : energyOf(V, x, 0, kB + kA);
    } else if (i < kTabY) {
        const int c = (i - kTabG) / kNB, b = (i - kTabG) % kNB;
        tab[i] = crossOf(V, c, kB + kA, kCMax, b, 0, kB);
    } else if (i < kTabEC) {
        const int c = (i - kTabY) / kNA, a = (i - kTabY) % kNA;
        tab[i] = crossOf(V, c, kB + kA, kCMax, a, kB, kA);
    } else if (i < kBFTableDoubles) {
        tab[i] = energyOf(V, i - kTabEC, kB + kA, kCMax);
    }
}

/* What a block keeps: its unit's sums, and G. */
struct UnitTables {
    double r[kLowBits];  /* 2 sum of V over set high bits, per low bit */
    double eh[kWave];    /* per high bit: its row sum if it is set */
    double f[kNA], g[kNB], S[kNC];
    __align__(16) double G[kNC][kNB];
};

/* Fills t for high pattern xH: the rows' sums over the high bits by 8 lanes a
 * row in a fixed order, then the subset sums.  Every load is unconditional, so
 * that they go out together. */
__device__ void buildUnit(UnitTables &t, const double *W, const double *tab, const BFPlan &p, unsigned long long xH) {
    const int N = p.N, U = p.U < N ? p.U : N, nH = p.nH;
    for (int i = threadIdx.x; i < (kNB << p.nC); i += kThreads)
        t.G[i / kNB][i % kNB] = tab[kTabG + i];
    if (threadIdx.x < kWave)
        t.eh[threadIdx.x] = 0.;
    if ((int)threadIdx.x < kLowBits)
        t.r[threadIdx.x] = 0.; /* stays so for bits past N - 1, or high */
    __syncthreads();
    const int part = threadIdx.x & 7;
    for (int row = threadIdx.x >> 3; row < U + nH; row += kThreads / 8) {
        const double *Wr = W + (size_t)(N - 1 - row) * N;
        double s = 0.;
#pragma unroll 2
        for (int k = part; k < nH; k += 8) {
            const double v = Wr[N - 1 - U - k];
            s += ((xH >> k) & 1ull) ? v : 0.;
        }
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        s += __shfl_xor(s, 4);
        if (part == 0) {
            if (row < U)
                t.r[row] = 2. * s;
            else
                t.eh[row - U] = ((xH >> (row - U)) & 1ull) ? s : 0.;
        }
    }
    __syncthreads();
    const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
    /* the sum of r over the set bits of v, bits [t0, t0 + n) */
    auto subset = [&](double s, int v, int t0, auto nTag) {
#pragma unroll
        for (int i = 0; i < decltype(nTag)::value; ++i) {
            const double x = t.r[t0 + i];
            s += ((v >> i) & 1) ? x : 0.;
        }
        return s;
    };
    if (w < kRows) {
        double e = t.eh[l]; /* at most 63 high bits */
        for (int o = 1; o < kWave; o <<= 1)
            e += __shfl_xor(e, o);
        t.f[w * kWave + l] = subset(e, w * kWave + l, kB, std::integral_constant<int, kA>());
    } else if (w == kRows) {
        if (l < kNB)
            t.g[l] = subset(0., l, 0, std::integral_constant<int, kB>());
    } else if (l < kNC) {
        t.S[l] = subset(tab[kTabEC + l], l, kB + kA, std::integral_constant<int, kCMax>());
    }
    __syncthreads();
}
static_assert(kRows + 2 <= kWaves, "a wave for each of the subset sums");

/* EL of the lane's rows: loaded before the unit's tables are formed, the round
 * trips to memory in flight together */
__device__ __forceinline__ void loadRows(const double *__restrict__ tab, double (*X)[kNB]) {
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
        for (int b = 0; b < kNB; ++b)
            X[r][b] = tab[kTabEL + b * kNA + r * kWave + threadIdx.x % kWave];
}
__device__ __forceinline__ void addUnit(const UnitTables &t, double (*X)[kNB]) {
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const double f = t.f[r * kWave + threadIdx.x % kWave];
#pragma unroll
        for (int b = 0; b < kNB; ++b)
            X[r][b] = (X[r][b] + t.g[b]) + f;
    }
}
/* Y(c,a) of the lane's rows */
__device__ __forceinline__ void loadY(const double *__restrict__ tab, int c, double *y) {
#pragma unroll
    for (int r = 0; r < kRows; ++r)
        y[r] = tab[kTabY + c * kNA + r * kWave + threadIdx.x % kWave];
}
/* the least X + G of each of the lane's rows */
__device__ __forceinline__ void rowMins(double (*X)[kNB], const double *G, double *least) {
    double m[kRows][2];
#pragma unroll
    for (int b = 0; b < kNB; ++b) {
        const double g = G[b];
#pragma unroll
        for (int r = 0; r < kRows; ++r)
            m[r][b & 1] = b < 2 ? X[r][b] + g : __builtin_fmin(m[r][b & 1], X[r][b] + g);
    }
#pragma unroll
    for (int r = 0; r < kRows; ++r)
        least[r] = __builtin_fmin(m[r][0], m[r][1]);
}
/* the first x of the lane's row r */
__device__ __forceinline__ unsigned long long rowX(const BFPlan &p, unsigned long long unit, int c, int r) {
    return (unit << p.U) |
           ((unsigned long long)((c << kA) | (r * kWave) | (int)(threadIdx.x % kWave)) << kB);
}

/* the wave's share of the unit's c values, uniform per wave */
__device__ __forceinline__ void waveRange(const BFPlan &p, int &c0, int &c1) {
    const int nC = 1 << p.nC, per = (nC + kWaves - 1) / kWaves;
    c0 = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)) * per;
    c1 = c0 + per < nC ? c0 + per : nC;
}

/* Whether this block is the last of the grid to arrive here (one thread; the
 * block's agent-scope stores before it are seen by the last block's agent-scope
 * loads after it).  Such a store is written through to where all XCDs see it,
 * so waiting for its completion orders it before the count; a fence would also
 * write back and invalidate the XCD's L2, which every block would then wait
 * for and refill (a scan of 512 blocks took 23.5 us
 * that way, 17.3 us without).  Blocks count themselves in
 * by 16 counters of a cache line each and the last of each group in a 17th,
 * since additions to one word from all XCDs queue up.  The counters are left at
 * zero. */
__device__ __forceinline__ bool lastBlock(unsigned *arrived) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned g = blockIdx.x % kBFArriveGroups;
    const unsigned inGroup = (gridDim.x - g + kBFArriveGroups - 1) / kBFArriveGroups;
    const unsigned groups = gridDim.x < (unsigned)kBFArriveGroups ? gridDim.x : kBFArriveGroups;
    if (atomicAdd(&arrived[(1 + g) * kBFArriveStride], 1u) != inGroup - 1)
        return false;
    if (atomicAdd(&arrived[0], 1u) != groups - 1)
        return false;
    for (unsigned i = 0; i <= groups; ++i)
        arrived[i * kBFArriveStride] = 0;
    return true;
}

template <class real>
__device__ __forceinline__ real waveMin(real v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const real w = __shfl_xor(v, o, kWave);
        v = w < v ? w : v;
    }
    return v;
}

__device__ __forceinline__ unsigned waveInclSum(unsigned v) {
    const int lane = threadIdx.x % kWave;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned u = __shfl_up(v, o, kWave);
        if (lane >= o)
            v += u;
    }
    return v;
}

/* Applies the list rule of CPUDenseGraphBatchSearch.cpp:33-48 to the range as
 * a whole and lists the units holding its minimum (one block, all threads). */
template <class real>
__device__ void mergeRange(real *unitMin, int nUnits, BFState<real> *st, unsigned long long cap,
                           unsigned *hits, unsigned long long *slots) {
    __shared__ real wMin[kWaves];
    __shared__ unsigned wSum[kWaves];
    __shared__ int sActive;
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    /* the minima of the first 512 units are kept from the first look */
    real first[2] = {(real)HUGE_VAL, (real)HUGE_VAL};
    auto load = [&](int u) {
        return __hip_atomic_load(&unitMin[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto minOf = [&](int u) { return u < kThreads ? first[0] : u < 2 * kThreads ? first[1] : load(u); };
    if ((int)threadIdx.x < nUnits)
        first[0] = load(threadIdx.x);
    if ((int)threadIdx.x + kThreads < nUnits)
        first[1] = load(threadIdx.x + kThreads);
    real m = first[1] < first[0] ? first[1] : first[0];
    for (int u = threadIdx.x + 2 * kThreads; u < nUnits; u += kThreads) {
        const real v = load(u);
        m = v < m ? v : m;
    }
    m = waveMin(m);
    if (lane == 0)
        wMin[w] = m;
    __syncthreads();
    m = wMin[0];
    for (int i = 1; i < kWaves; ++i)
        m = wMin[i] < m ? wMin[i] : m;
    if (threadIdx.x == 0) {
        int active = 0;
        unsigned long long base = 0;
        if (m < st->Emin) { /* a lower minimum: the list restarts */
            st->Emin = m;
            active = 1;
        } else if (m == st->Emin) { /* ties append while the list is short of cap */
            base = st->count;
            active = base < cap;
        }
        st->base = base;
        st->ticket = 0;
        sActive = active;
    }
    __syncthreads();
    unsigned running = 0;
    for (int u0 = 0; sActive && u0 < nUnits; u0 += kThreads) {
        const int u = u0 + (int)threadIdx.x;
        const bool hit = u < nUnits && minOf(u) == m;
        const unsigned long long bal = __ballot(hit);
        if (lane == 0)
            wSum[w] = (unsigned)__popcll(bal);
        __syncthreads();
        unsigned pos = running + (unsigned)__popcll(bal & ((1ull << lane) - 1ull));
        for (int i = 0; i < w; ++i)
            pos += wSum[i];
        if (hit) {
            hits[pos] = (unsigned)u;
            slots[pos] = 0ull;
        }
        for (int i = 0; i < kWaves; ++i)
            running += wSum[i];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        st->nHit = running;
}

template <class real>
__global__ __launch_bounds__(kThreads) void bfScanKernel(const double *W, const double *__restrict__ tab, BFPlan p,
                                                         unsigned long long xb, unsigned long long xe,
                                                         unsigned long long unit0, real *unitMin, BFState<real> *st,
                                                         unsigned long long cap, unsigned *hits,
                                                         unsigned long long *slots) {
    __shared__ UnitTables t;
    __shared__ double wMin[kWaves];
    __shared__ int sLast;
    const unsigned long long unit = unit0 + blockIdx.x;
    double X[kRows][kNB], y[2][kRows];
    int c0, c1;
    waveRange(p, c0, c1);
    loadRows(tab, X);
    loadY(tab, c0, y[0]); /* c0 < 2^5 */
    buildUnit(t, W, tab, p, unit);
    addUnit(t, X);
    /* a range cut inside the unit (at a multiple of 256, or 2^N): whole rows */
    const unsigned long long u0 = unit << p.U, u1 = (unit + 1) << p.U;
    const bool cut = u0 < xb || u1 > xe;
    double best = HUGE_VAL;
    for (int c = c0; c < c1; ++c) {
        loadY(tab, c + 1 < kNC ? c + 1 : c, y[1]); /* the next c's */
        double least[kRows];
        rowMins(X, t.G[c], least);
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            const double e = least[r] + (y[0][r] + t.S[c]);
            const unsigned long long x = rowX(p, unit, c, r);
            if (!cut || (x >= xb && x < xe))
                best = __builtin_fmin(best, e);
            y[0][r] = y[1][r];
        }
    }
    best = waveMin(best);
    if (threadIdx.x % kWave == 0)
        wMin[threadIdx.x / kWave] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = wMin[0];
        for (int i = 1; i < kWaves; ++i)
            m = wMin[i] < m ? wMin[i] : m;
        __hip_atomic_store(&unitMin[blockIdx.x], (real)m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sLast = lastBlock(st->arrived);
    }
    __syncthreads();
    if (!sLast)
        return;
    mergeRange<real>(unitMin, (int)gridDim.x, st, cap, hits, slots);
}

/* Blocks take the listed units in order (tickets); a unit's place in the list
 * is published by the unit before it, whose block took an earlier ticket and
 * therefore runs: every wait ends. */
template <class real>
__global__ __launch_bounds__(kThreads) void bfSelectKernel(const double *W, const double *__restrict__ tab, BFPlan p,
                                                           unsigned long long xb, unsigned long long xe,
                                                           unsigned long long unit0, BFState<real> *st,
                                                           unsigned long long cap, const unsigned *hits,
                                                           unsigned long long *slots, unsigned long long *xList) {
    __shared__ UnitTables t;
    __shared__ uint32_t ties[kNC][kNA]; /* per row: the candidates that are minimisers */
    __shared__ unsigned wSum[kWaves];
    __shared__ unsigned sTicket;
    __shared__ unsigned long long sBefore;
    const unsigned nHit = st->nHit;
    if (blockIdx.x >= nHit)
        return; /* no more blocks than units are needed */
    const real Emin = st->Emin;
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    int c0, c1;
    waveRange(p, c0, c1);
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0)
            sTicket = atomicAdd(&st->ticket, 1u);
        double X[kRows][kNB];
        loadRows(tab, X);
        __syncthreads();
        const unsigned k = sTicket;
        if (k >= nHit)
            return;
        const unsigned long long unit = unit0 + hits[k];
        buildUnit(t, W, tab, p, unit);
        addUnit(t, X);
        unsigned cnt = 0;
        for (int c = c0; c < c1; ++c) {
            double least[kRows], y[kRows];
            loadY(tab, c, y);
            rowMins(X, t.G[c], least);
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const double rest = y[r] + t.S[c];
                const unsigned long long x = rowX(p, unit, c, r);
                const bool in = x >= xb && x < xe && (real)(least[r] + rest) == Emin;
                uint32_t bits = 0;
                if (__ballot(in)) {
#pragma unroll
                    for (int b = 0; b < kNB; ++b)
                        if (in && (real)((X[r][b] + t.G[c][b]) + rest) == Emin)
                            bits |= 1u << b;
                }
                ties[c][r * kWave + lane] = bits; /* read by this lane only */
                cnt += (unsigned)__popc(bits);
            }
        }
        const unsigned incl = waveInclSum(cnt);
        if (lane == kWave - 1)
            wSum[w] = incl;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned total = 0;
            for (int i = 0; i < kWaves; ++i)
                total += wSum[i];
            unsigned long long before = st->base;
            if (k > 0) {
                unsigned long long v; /* 1 + the list length up to the unit before */
                while ((v = __hip_atomic_load(&slots[k - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0ull)
                    __builtin_amdgcn_s_sleep(1);
                before = v - 1;
            }
            __hip_atomic_store(&slots[k], before + total + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (k == nHit - 1)
                st->count = before + total < cap ? before + total : cap;
            sBefore = before;
        }
        __syncthreads();
        unsigned long long pos = sBefore;
        for (int i = 0; i < w; ++i)
            pos += wSum[i];
        for (int c = c0; c < c1; ++c) {
#pragma unroll
            for (int r = 0; r < kRows; ++r) {
                const uint32_t bits = ties[c][r * kWave + lane];
                if (pos >= cap || !__ballot(bits != 0)) /* wave-uniform */
                    continue;
                const unsigned n = (unsigned)__popc(bits), upTo = waveInclSum(n);
                const unsigned long long x = rowX(p, unit, c, r);
                unsigned long long at = pos + upTo - n;
                for (uint32_t left = bits; left; left &= left - 1, ++at)
                    if (at < cap)
                        xList[at] = x | (unsigned long long)__builtin_ctz(left);
                pos += (unsigned)__shfl((int)upTo, kWave - 1);
            }
        }
    }
}

}  // namespace

BFPlan bfPlan(int N) {
    BFPlan p;
    p.N = N;
    /* units as large as leave 256 of them, with four values of c at least (one
     * a wave) and 2^17 candidates at most: a span of 2^26 then is 512 blocks,
     * two to a CU */
    const int rest = N - (kB + kA);
    const int want = rest - 8;
    p.nC = want < 2 ? 2 : want < kCMax ? want : kCMax;
    if (p.nC > rest)
        p.nC = rest < 0 ? 0 : rest;
    p.U = kB + kA + p.nC;
    p.nH = N > p.U ? N - p.U : 0;
    return p;
}

void bfTables(const double *d_W, const BFPlan &p, double *d_tab, hipStream_t stream) {
    bfTablesKernel<<<divru(kBFTableDoubles, kThreads), kThreads, 0, stream>>>(d_W, p, d_tab);
    HIP_CHECK(hipGetLastError());
}

template <class real>
void bfSearchRange(const double *d_W, const double *d_tab, const BFPlan &p, unsigned long long xb,
                   unsigned long long xe, BFState<real> *d_state, unsigned long long cap, real *d_unitMin,
                   unsigned *d_hits, unsigned long long *d_slots, int maxUnits, unsigned long long *d_xList,
                   hipStream_t stream) {
    if (xb >= xe)
        return;
    const unsigned long long unit0 = xb >> p.U;
    const unsigned long long unit1 = (xe + (1ull << p.U) - 1) >> p.U;
    const unsigned long long n = unit1 - unit0;
    SQ_THROW_IF(n > (unsigned long long)maxUnits, "bf search range of %llu units exceeds %d", n, maxUnits);
    SQ_THROW_IF(xb % kNB != 0 || (xe % kNB != 0 && xe != 1ull << p.N), "bf search range is not cut at whole rows");
    bfScanKernel<real><<<(unsigned)n, kThreads, 0, stream>>>(d_W, d_tab, p, xb, xe, unit0, d_unitMin, d_state, cap,
                                                            d_hits, d_slots);
    HIP_CHECK(hipGetLastError());
    bfSelectKernel<real><<<(unsigned)(n < kSelBlocks ? n : kSelBlocks), kThreads, 0, stream>>>(
        d_W, d_tab, p, xb, xe, unit0, d_state, cap, d_hits, d_slots, d_xList);
    HIP_CHECK(hipGetLastError());
}

template void bfSearchRange<float>(const double *, const double *, const BFPlan &, unsigned long long,
                                   unsigned long long, BFState<float> *, unsigned long long, float *, unsigned *,
                                   unsigned long long *, int, unsigned long long *, hipStream_t);
template void bfSearchRange<double>(const double *, const double *, const BFPlan &, unsigned long long,
                                    unsigned long long, BFState<double> *, unsigned long long, double *, unsigned *,
                                    unsigned long long *, int, unsigned long long *, hipStream_t);

}  // namespace sqaod_rocm
