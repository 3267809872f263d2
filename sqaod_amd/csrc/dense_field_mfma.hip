/*
 * Spin-matrix GEMM on the MFMA units (gfx950):
 *   F[y][c] = sum_k q[y][k] B[c][k]
 * with q the +-1 spins of m slices (packed bits, K per row) and B given by
 * rows.  The dense annealer's local-field refresh is B = J (symmetric, so
 * F = Q . J); the bipartite annealer's half-steps are B = J and B = J^T
 * (dEmat = qFixed . J^T, CPUBipartiteGraphAnnealer.cpp:351-352).
 *
 *  - bf16x2: J = hi + lo (two bf16 planes), spins +-1 exact in bf16,
 *    v_mfma_f32_16x16x32_bf16 twice per k-block, fp32 accumulation.
 *  - fp32:   J = hi + mid + lo exactly (three bf16 planes, bf16Split3), the
 *    same kernel with three MFMAs per k-block: every product is exact and
 *    accumulates in fp32, at a third of the v_mfma_f32_16x16x4_f32 cost.
 *  - fp8:    J as e4m3 bytes with a power-of-two scale per column, spins
 *    +-1 exact in e4m3, v_mfma_scale_f32_16x16x128_f8f6f4 with unit block
 *    scales; the column scale multiplies the reduced sum (exactly).
 *  - fp64:   J as it is stored, v_mfma_f64_16x16x4_f64 (a kernel of its own,
 *    fieldRefreshF64Kernel).
 *
 * J is read from a copy laid out in MFMA fragment order, built once per
 * problem: for column block cb (16 columns) and k-block kb, the 64 lanes'
 * B fragments are one contiguous run (1 KiB per plane), so every operand
 * load of a wave is a single fully coalesced 1 KiB request and a block
 * streams its columns' k-range front to back.
 *
 * Work split: one block of 4 waves owns 16 output columns and T tiles of 16
 * slice rows.  The k-range is split over the 4 waves in super-blocks of kDepth
 * k-blocks (interleaved), each wave double-buffers its operand loads, and the
 * four partial sums are added in a fixed order through LDS, so results are
 * deterministic and do not depend on T.  Each column block starts its k-range at
 * a different super-block, so concurrently running blocks read different address
 * ranges; the row groups of a column block run on one XCD, next to each other,
 * and find its fragments in that XCD's L2.
 *
 * What bounds it is the chain of a wave's round trips (operands, the spin table
 * in LDS), so T is the largest that leaves two blocks to each CU (rowTilesFor).
 * With T = 16 throughout, i.e. each column block in one block, whose spin words
 * went through a lane shuffle, the refresh of N=4096, m=256 (bf16x2) took
 * 35.2 us, that of N=1200, m=300 (fp32) 24.3 us and a half-step of the bipartite
 * 1024 + 1024, m=64 8.3 us; now 29.7, 8.5 and 4.1 us.  A large bf16 product
 * would take 14 us for the first, and so would reading its fragments once.
 *
 * Spins: lane L loads the packed spin words of row L % 16 of each tile for a
 * whole super-block (16 bytes); a byte of them picks 8 spins as bf16 +-1 from a
 * table in LDS.
 *
 * The k-blocks past the valid length read zero padding (rows of B are padded
 * to K with zeros, the fragment copy is zero for columns past B's rows, and
 * spin bits past the valid length are zero), so ragged shapes need no special
 * case.
 */
#include "common.h"
#include "kernels.h"
#include "bf16.h"

namespace sqaod_rocm {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWave = 64;
constexpr int kGroupedTiles = 4;  /* row tiles per block of a grouped launch */
constexpr int kSplitK = 4;        /* waves per block, each a share of the k-range */
constexpr int kDepth = 4;         /* k-blocks per super-block (the double-buffered unit) */
constexpr int kBlockThreads = kSplitK * kWave;

/* 8 spins (bits b0..b7 of `bits`) as bf16 +-1: each dword packs two
 * elements, 0xBF80 (-1) with the sign bit cleared where the spin bit is 1. */
__device__ __forceinline__ bf16x8 spinsBF16(uint32_t bits) {
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        v[j] = 0xBF80BF80u ^ (((bits >> (2 * j)) & 1u) << 15) ^ ((bits >> (2 * j + 1)) << 31);
    return __builtin_bit_cast(bf16x8, v);
}

/* The partial tiles: [w][4 t + r][lane] holds wave w's acc[t][r], i.e. row
 * 16 t + 4 (lane / 16) + r, column lane % 16. */
template <int T>
using RedTile = float[T * 4][kWave];

/* Fixed-order sum of the kSplitK partial tiles in LDS and the store of the
 * block's rows; colScale (if given) multiplies each column's sum. */
template <int T>
__device__ __forceinline__ void reduceStore(const f32x4 (&acc)[T], RedTile<T> *red, int y0, int m, int cb, int ldF,
                                            float *F, const float *colScale = nullptr) {
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            red[w][4 * t + r][lane] = acc[t][r];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t) {
        /* wave w adds register w of each tile */
        const int y = y0 + 16 * t + 4 * (lane >> 4) + w, col = cb * 16 + (lane & 15);
        if (y < m) {
            float s = red[0][4 * t + w][lane];
#pragma unroll
            for (int p = 1; p < kSplitK; ++p)
                s += red[p][4 * t + w][lane];
            if (colScale)
                s *= colScale[col];
            F[(long long)y * ldF + col] = s;
        }
    }
}

/* frag: [column blocks][K/32 k-blocks][PLANES][64 lanes] x 16 B (PLANES bf16
 * planes whose sum is B: hi + lo for the bf16x2 form, hi + mid + lo -- exactly
 * B -- for the fp32 form); the block writes columns [16 cb, 16 cb + 16) of rows
 * [y0, y0 + 16 T) of F (row stride ldF).  lut: byte -> 8 spins as bf16 +-1. */
template <int PLANES, int T>
__device__ __forceinline__ void refreshBF16Block(const uint4 *frag, const uint32_t *Qbits, int K, int m, int Nw,
                                                 int ldF, float *F, int cb, int y0, RedTile<T> *red,
                                                 const uint4 *lut) {
    const int lane = threadIdx.x % kWave;
    const int w = threadIdx.x / kWave;
    const int c = lane & 15, g = lane >> 4;
    const int nK = K / 32;      /* k-blocks of 32; K is a multiple of 256 */
    const int nS = nK / kDepth; /* super-blocks: wave w takes w, w + 4, ... */
    const int sOff = (int)(((long long)cb * 3) % nS);
    const uint4 *fb = frag + (size_t)cb * nK * PLANES * kWave + lane;
    f32x4 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 bp[PLANES][2][kDepth], qw[2][T];
    /* loads super-block l (logical index) into buffer buf; l < nS.  Rows past
     * m read row m - 1; their sums are not stored. */
    auto fetch = [&](int buf, int l) {
        int s = l + sOff;
        if (s >= nS)
            s -= nS;
        const int kb0 = s * kDepth;
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            const uint4 *p = fb + (size_t)(kb0 + d) * PLANES * kWave;
#pragma unroll
            for (int pl = 0; pl < PLANES; ++pl)
                bp[pl][buf][d] = p[pl * kWave];
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int y = y0 + 16 * t + c;
            qw[buf][t] = *reinterpret_cast<const uint4 *>(Qbits + (size_t)(y < m ? y : m - 1) * Nw + kb0);
        }
    };
    /* the A operands of a k-block are read from the table one k-block ahead of
     * the MFMAs that use them */
    auto gather = [&](int buf, int d, uint4 *av) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const uint4 q4 = qw[buf][t];
            const uint32_t word = d == 0 ? q4.x : d == 1 ? q4.y : d == 2 ? q4.z : q4.w;
            av[t] = lut[(word >> (8 * g)) & 0xffu];
        }
    };
    auto compute = [&](int buf) {
        uint4 av[2][T];
        gather(buf, 0, av[0]);
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            if (d + 1 < kDepth)
                gather(buf, d + 1, av[(d + 1) & 1]);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if (y0 + 16 * t >= m) /* wave-uniform */
                    continue;
#pragma unroll
                for (int pl = 0; pl < PLANES; ++pl)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8, av[d & 1][t]), __builtin_bit_cast(bf16x8, bp[pl][buf][d]), acc[t], 0,
                        0, 0);
            }
        }
    };
    /* buffers alternate with constant indices (no dynamic register indexing) */
    for (int l = w; l < nS; l += 2 * kSplitK) {
        if (l == w)
            fetch(0, l);
        if (l + kSplitK < nS)
            fetch(1, l + kSplitK);
        compute(0);
        if (l + kSplitK >= nS)
            break;
        if (l + 2 * kSplitK < nS)
            fetch(0, l + 2 * kSplitK);
        compute(1);
    }
    reduceStore<T>(acc, red, y0, m, cb, ldF, F);
}

__device__ __forceinline__ void fillLutBF16(uint4 *lut) {
    for (int i = threadIdx.x; i < 256; i += kBlockThreads)
        lut[i] = __builtin_bit_cast(uint4, spinsBF16((uint32_t)i));
    __syncthreads();
}

/* Column block and first row of a block: the row groups of one column block are
 * 8 apart, i.e. on one XCD one after the other (nColBlocks is a multiple of 8,
 * or the tail of it keeps the plain order). */
__device__ __forceinline__ void blockTile(int block, int nColBlocks, int nGroups, int rows, int &cb, int &y0) {
    const int whole = nColBlocks / 8 * 8 * nGroups;
    int group;
    if (block < whole) {
        const int i = block / 8;
        cb = i / nGroups * 8 + block % 8;
        group = i % nGroups;
    } else {
        cb = nColBlocks / 8 * 8 + (block - whole) / nGroups;
        group = (block - whole) % nGroups;
    }
    y0 = group * rows;
}

template <int PLANES, int T>
__global__ __launch_bounds__(kBlockThreads) void fieldRefreshBF16Kernel(const uint4 *frag, const uint32_t *Qbits,
                                                                        int nColBlocks, int nGroups, int K, int m,
                                                                        int Nw, int ldF, float *F) {
    __shared__ RedTile<T> red[kSplitK];
    __shared__ uint4 lut[256]; /* 4 KiB */
    int cb, y0;
    blockTile(blockIdx.x, nColBlocks, nGroups, 16 * T, cb, y0);
    fillLutBF16(lut);
    refreshBF16Block<PLANES, T>(frag, Qbits, K, m, Nw, ldF, F, cb, y0, red, lut);
}

/* Row tiles per block: the largest of 1, 2, 4 that leaves 512 blocks, two to each
 * of the 256 CUs.  (Eight take 292 registers, one wave to a SIMD: N=4096, m=256
 * bf16x2 33.1 us against 29.7 us with four.) */
int rowTilesFor(int nColBlocks, int m) {
    const int tiles = divru(m, 16);
    for (int t = 4; t > 1; t /= 2)
        if (nColBlocks * divru(tiles, t) >= 512)
            return t;
    return 1;
}

/* Double solvers: F[y][c] = sum_{k < K} q[y][k] B[k][c] with B row-major, as it
 * is stored (the dense annealer's J, the bipartite one's J or J^T).
 *
 * A block of 4 waves owns 16 columns and RT 16-row tiles; wave w takes the
 * k-blocks of 32 (one spin word a row) w, w + 4, ..., eight
 * v_mfma_f64_16x16x4_f64 per tile each, and the four partial tiles are added
 * in LDS in the order ((P0 + P1) + P2) + P3.  Lane L supplies B[k][c] and the
 * spin of row L % 16 for k = 32 kb + 4 t + L / 16: a load instruction reads
 * four 128-byte row pieces, and the next k-block's loads are in flight while
 * this one's products run.
 *
 * A matrix instruction takes 64 cycles, so the product itself is short (under
 * 2 us at N=500, m=125); at these sizes the kernel is bound by filling the
 * chip and by one memory round trip per k-block.  Hence a column block of 16,
 * the k-range over the four SIMDs of a CU, and RT = 1 until every CU has two
 * blocks: the vector kernel this replaced keeps 256 columns and 32 rows a
 * block, 8 blocks at that size.  Measured: 6.0 us against the vector kernel's
 * 245.6 us at N=500, m=125; 4.6 against 124.4 us for the bipartite half-steps
 * at 200 + 301 spins, m=125.
 */
typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kF64KBlock = 32;
constexpr int kF64Steps = kF64KBlock / 4;

template <int RT>
__global__ __launch_bounds__(kBlockThreads) void fieldRefreshF64Kernel(const double *B, int K, int ldB,
                                                                       const uint32_t *Qbits, int m, int Nw, int ldF,
                                                                       double *F) {
    __shared__ double red[kSplitK][RT * 4][kWave];
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int c = lane & 15, g = lane >> 4;
    const int y0 = blockIdx.y * 16 * RT;
    const double *Bc = B + blockIdx.x * 16 + c;
    const int nK = (K + kF64KBlock - 1) / kF64KBlock; /* nK <= Nw: K <= 32 Nw */
    f64x4 acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
        acc[t] = f64x4{0., 0., 0., 0.};
    double b[2][kF64Steps];
    uint32_t qw[2][RT];
    /* rows of B past K and slices past m are read at the last valid one; the
     * former enter as zeros, the latter's sums are not stored */
    auto fetch = [&](int buf, int kb) {
#pragma unroll
        for (int t = 0; t < kF64Steps; ++t) {
            const int k = kb * kF64KBlock + 4 * t + g;
            const double v = Bc[(size_t)(k < K ? k : K - 1) * ldB];
            b[buf][t] = k < K ? v : 0.;
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const int y = y0 + 16 * r + c;
            qw[buf][r] = Qbits[(size_t)(y < m ? y : m - 1) * Nw + kb];
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int t = 0; t < kF64Steps; ++t)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const double q = ((qw[buf][r] >> (4 * t + g)) & 1u) ? 1. : -1.;
                acc[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(q, b[buf][t], acc[r], 0, 0, 0);
            }
    };
    if (w < nK)
        fetch(0, w);
    for (int kb = w; kb < nK; kb += 2 * kSplitK) {
        if (kb + kSplitK < nK)
            fetch(1, kb + kSplitK);
        compute(0);
        if (kb + kSplitK >= nK)
            break;
        if (kb + 2 * kSplitK < nK)
            fetch(0, kb + 2 * kSplitK);
        compute(1);
    }
    /* register r of lane L: row 4 r + L / 16, column L % 16 of the tile */
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            red[w][4 * t + r][lane] = acc[t][r];
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        /* thread (w, lane) adds row piece r = w of each tile */
        const int y = y0 + 16 * t + 4 * w + g;
        double s = red[0][4 * t + w][lane];
#pragma unroll
        for (int p = 1; p < kSplitK; ++p)
            s += red[p][4 * t + w][lane];
        if (y < m)
            F[(size_t)y * ldF + blockIdx.x * 16 + c] = s;
    }
}

typedef int i32x8 __attribute__((ext_vector_type(8)));
constexpr int kDepth8 = 2; /* fp8: k-blocks of 128 per super-block (256 k = 8 spin words) */
constexpr int kE4M3Unit = 127; /* E8M0 block scale 2^0 */

/* 8 spins (bits of `bits`) as e4m3 +-1: 0x38 = +1, 0xB8 = -1 */
__device__ __forceinline__ uint2 spinsFP8(uint32_t bits) {
    uint32_t v[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t nib = (bits >> (4 * j)) & 15u;
        v[j] = 0xB8B8B8B8u ^ (((nib * 0x204081u) & 0x01010101u) << 7);
    }
    return uint2{v[0], v[1]};
}

/* frag: [column blocks][K/128 k-blocks][2 halves][64 lanes] x 16 B.  In
 * super-block s (k-blocks 2s, 2s + 1), lane group g of k-block 2s + d holds
 * k = 256 s + 64 g + 32 d + e, e < 32: spin word 8 s + 2 g + d of the row,
 * bit e -- so each lane's A operand for a whole super-block is the 8-byte
 * pair of words (8 s + 2 g, 8 s + 2 g + 1) of its row, loaded directly. */
template <int T>
__device__ __forceinline__ void refreshFP8Block(const uint4 *frag, const float *colScale, const uint32_t *Qbits,
                                                int K, int m, int Nw, int ldF, float *F, int cb, int y0,
                                                RedTile<T> *red, const uint2 *lut) {
    const int lane = threadIdx.x % kWave;
    const int w = threadIdx.x / kWave;
    const int c = lane & 15, g = lane >> 4;
    const int nK = K / 128;
    const int nS = nK / kDepth8;
    const int sOff = (int)(((long long)cb * 3) % nS);
    const uint4 *fb = frag + (size_t)cb * nK * 2 * kWave + lane;
    f32x4 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
        acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 b0[2][kDepth8], b1[2][kDepth8];
    uint2 qv[2][T];
    auto fetch = [&](int buf, int l) {
        int s = l + sOff;
        if (s >= nS)
            s -= nS;
#pragma unroll
        for (int d = 0; d < kDepth8; ++d) {
            const uint4 *p = fb + (size_t)(s * kDepth8 + d) * 2 * kWave;
            b0[buf][d] = p[0];
            b1[buf][d] = p[kWave];
        }
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const int y = y0 + 16 * t + c;
            qv[buf][t] = *reinterpret_cast<const uint2 *>(Qbits + (size_t)(y < m ? y : m - 1) * Nw + 8 * s + 2 * g);
        }
    };
    auto compute = [&](int buf) {
#pragma unroll
        for (int d = 0; d < kDepth8; ++d) {
            const uint4 x0 = b0[buf][d], x1 = b1[buf][d];
            const i32x8 bop = {(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w,
                               (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
            /* A operands (four table reads per tile) */
            i32x8 aop[T];
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const uint32_t word = d == 0 ? qv[buf][t].x : qv[buf][t].y;
                const uint2 l0 = lut[word & 0xffu], l1 = lut[(word >> 8) & 0xffu];
                const uint2 l2 = lut[(word >> 16) & 0xffu], l3 = lut[word >> 24];
                aop[t] = i32x8{(int)l0.x, (int)l0.y, (int)l1.x, (int)l1.y,
                               (int)l2.x, (int)l2.y, (int)l3.x, (int)l3.y};
            }
#pragma unroll
            for (int t = 0; t < T; ++t)
                if (y0 + 16 * t < m) /* wave-uniform */
                    acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(aop[t], bop, acc[t], 0, 0, 0, kE4M3Unit,
                                                                              0, kE4M3Unit);
        }
    };
    for (int l = w; l < nS; l += 2 * kSplitK) {
        if (l == w)
            fetch(0, l);
        if (l + kSplitK < nS)
            fetch(1, l + kSplitK);
        compute(0);
        if (l + kSplitK >= nS)
            break;
        if (l + 2 * kSplitK < nS)
            fetch(0, l + 2 * kSplitK);
        compute(1);
    }
    reduceStore<T>(acc, red, y0, m, cb, ldF, F, colScale);
}

__device__ __forceinline__ void fillLutFP8(uint2 *lut) {
    for (int i = threadIdx.x; i < 256; i += kBlockThreads)
        lut[i] = spinsFP8((uint32_t)i);
    __syncthreads();
}

template <int T>
__global__ __launch_bounds__(kBlockThreads) void fieldRefreshFP8Kernel(const uint4 *frag, const float *colScale,
                                                                       const uint32_t *Qbits, int nColBlocks,
                                                                       int nGroups, int K, int m, int Nw, int ldF,
                                                                       float *F) {
    __shared__ RedTile<T> red[kSplitK];
    __shared__ uint2 lut[256]; /* 2 KiB */
    int cb, y0;
    blockTile(blockIdx.x, nColBlocks, nGroups, 16 * T, cb, y0);
    fillLutFP8(lut);
    refreshFP8Block<T>(frag, colScale, Qbits, K, m, Nw, ldF, F, cb, y0, red, lut);
}

/* Many GEMMs of one form in one launch: block b runs block b - blockStart[j] of
 * job j, blockStart[j] <= b < blockStart[j + 1]. */
__device__ __forceinline__ int jobOfBlock(const int *blockStart, int nJobs) {
    int lo = 0, hi = nJobs - 1;
    const int b = blockIdx.x;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (blockStart[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

template <int FORM>
__global__ __launch_bounds__(kBlockThreads) void fieldRefreshGroupedKernel(const FieldGemmJob *jobs,
                                                                           const int *blockStart, int nJobs) {
    __shared__ RedTile<kGroupedTiles> red[kSplitK];
    __shared__ uint4 lut[256];
    const int j = jobOfBlock(blockStart, nJobs);
    const FieldGemmJob jb = jobs[j];
    const uint4 *frag = reinterpret_cast<const uint4 *>(jb.frag);
    int cb, y0;
    blockTile((int)blockIdx.x - blockStart[j], jb.nCols / 16, divru(jb.m, 16 * kGroupedTiles), 16 * kGroupedTiles, cb,
              y0);
    if constexpr (FORM == fieldFP8) {
        fillLutFP8(reinterpret_cast<uint2 *>(lut));
        refreshFP8Block<kGroupedTiles>(frag, jb.colScale, jb.Qbits, jb.K, jb.m, jb.Nw, jb.ldF, jb.F, cb, y0, red,
                                       reinterpret_cast<const uint2 *>(lut));
    } else {
        fillLutBF16(lut);
        refreshBF16Block<FORM == fieldBF16x2 ? 2 : 3, kGroupedTiles>(frag, jb.Qbits, jb.K, jb.m, jb.Nw, jb.ldF, jb.F,
                                                                     cb, y0, red, lut);
    }
}

/* One thread per (column block, k-block, lane): the 32 bytes of the lane's
 * column (a row of B8, stride ld8, zero past `rows`) in the order above. */
__global__ void buildFragFP8Kernel(const uint8_t *B8, int rows, int ld8, int nColBlocks, int K, uint4 *frag) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nK = K / 128;
    if (idx >= (size_t)nColBlocks * nK * kWave)
        return;
    const int lane = (int)(idx % kWave);
    const size_t rest = idx / kWave;
    const int kb = (int)(rest % nK), cb = (int)(rest / nK);
    const int col = cb * 16 + (lane & 15);
    const int k0 = 256 * (kb / kDepth8) + 64 * (lane >> 4) + 32 * (kb % kDepth8);
    uint4 v0 = {0u, 0u, 0u, 0u}, v1 = {0u, 0u, 0u, 0u};
    if (col < rows) {
        const uint4 *src = reinterpret_cast<const uint4 *>(B8 + (size_t)col * ld8 + k0);
        v0 = src[0];
        v1 = src[1];
    }
    uint4 *dst = frag + ((size_t)cb * nK + kb) * 2 * kWave + lane;
    dst[0] = v0;
    dst[kWave] = v1;
}

/* One thread per (column block, k-block, lane): the lane's 8 k values of its
 * column (a row of B, row stride ld, zero past `rows`), split into bf16 hi and lo. */
template <int PLANES>
__global__ void buildFragBF16Kernel(const float *B, int rows, int ld, int nColBlocks, int K, uint4 *frag) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int nK = K / 32;
    if (idx >= (size_t)nColBlocks * nK * kWave)
        return;
    const int lane = (int)(idx % kWave);
    const size_t rest = idx / kWave;
    const int kb = (int)(rest % nK), cb = (int)(rest / nK);
    const int col = cb * 16 + (lane & 15), k0 = kb * 32 + 8 * (lane >> 4);
    uint32_t pw[PLANES][4] = {};
    if (col < rows) {
        const float4 *src = reinterpret_cast<const float4 *>(B + (size_t)col * ld + k0);
        const float4 v0 = src[0], v1 = src[1];
        const float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            uint16_t h[3];
            if constexpr (PLANES == 2)
                bf16Split(v[e], h[0], h[1]);
            else
                bf16Split3(v[e], h[0], h[1], h[2]);
#pragma unroll
            for (int pl = 0; pl < PLANES; ++pl)
                pw[pl][e >> 1] |= (uint32_t)h[pl] << (16 * (e & 1));
        }
    }
    uint4 *dst = frag + ((size_t)cb * nK + kb) * PLANES * kWave + lane;
#pragma unroll
    for (int pl = 0; pl < PLANES; ++pl)
        dst[pl * kWave] = uint4{pw[pl][0], pw[pl][1], pw[pl][2], pw[pl][3]};
}

void checkGemm(int nCols, int K, int ld, int Nw) {
    SQ_THROW_IF(nCols <= 0 || nCols % 16 != 0, "field GEMM: %d output columns is not a positive multiple of 16",
                nCols);
    SQ_THROW_IF(K <= 0 || K % 256 != 0 || Nw * 32 != K, "field GEMM: K=%d must be a positive multiple of 256", K);
    SQ_THROW_IF(ld < K, "field GEMM: row stride %d is shorter than K=%d", ld, K);
}

}  // namespace

size_t fieldFragElemsBF16x2(int nCols, int K) { return 2 * (size_t)nCols * K; } /* hi and lo planes, uint16 each */
size_t fieldFragElemsF32(int nCols, int K) { return 3 * (size_t)nCols * K; } /* hi, mid and lo planes */
size_t fieldFragElemsFP8(int nCols, int K) { return (size_t)nCols * K; } /* bytes */

void buildFragFP8(const uint8_t *d_B8, int rows, int ld8, int nCols, int K, uint8_t *d_frag, size_t fragElems,
                  hipStream_t stream) {
    checkGemm(nCols, K, ld8, K / 32);
    SQ_THROW_IF(ld8 % 16 != 0, "fp8 fragments: row stride %d is not a multiple of 16 bytes", ld8);
    SQ_THROW_IF(rows > nCols, "field GEMM: %d rows exceed %d columns", rows, nCols);
    SQ_THROW_IF(fragElems < fieldFragElemsFP8(nCols, K), "fp8 fragment buffer holds %zu of %zu bytes", fragElems,
                fieldFragElemsFP8(nCols, K));
    const size_t threads = (size_t)(nCols / 16) * (K / 128) * kWave;
    buildFragFP8Kernel<<<(unsigned)((threads + 255) / 256), 256, 0, stream>>>(d_B8, rows, ld8, nCols / 16, K,
                                                                              reinterpret_cast<uint4 *>(d_frag));
    HIP_CHECK(hipGetLastError());
}

void fieldRefreshGrouped(int fieldFormat, const FieldGemmJob *d_jobs, const int *d_blockStart, int nJobs,
                         int totalBlocks, hipStream_t stream) {
    SQ_THROW_IF(nJobs <= 0 || totalBlocks <= 0, "grouped field GEMM: no work");
    if (fieldFormat == fieldBF16x2)
        fieldRefreshGroupedKernel<fieldBF16x2><<<totalBlocks, kBlockThreads, 0, stream>>>(d_jobs, d_blockStart, nJobs);
    else if (fieldFormat == fieldFP8)
        fieldRefreshGroupedKernel<fieldFP8><<<totalBlocks, kBlockThreads, 0, stream>>>(d_jobs, d_blockStart, nJobs);
    else
        fieldRefreshGroupedKernel<fieldF32><<<totalBlocks, kBlockThreads, 0, stream>>>(d_jobs, d_blockStart, nJobs);
    HIP_CHECK(hipGetLastError());
}

int fieldGemmJobBlocks(const FieldGemmJob &j) { return j.nCols / 16 * divru(j.m, 16 * kGroupedTiles); }

void checkFieldGemmJob(const FieldGemmJob &j, int fieldFormat) {
    checkGemm(j.nCols, j.K, j.K, j.Nw);
    SQ_THROW_IF(j.ldF < j.nCols || !j.frag || !j.Qbits || !j.F || (fieldFormat == fieldFP8 && !j.colScale),
                "grouped field GEMM: bad job");
}

void fieldRefreshFP8(const uint8_t *d_frag, size_t fragElems, const float *d_colScale, const uint32_t *d_Qbits,
                     int nCols, int K, int m, int Nw, int ldF, float *d_F, hipStream_t stream) {
    checkGemm(nCols, K, K, Nw);
    SQ_THROW_IF(ldF < nCols, "field GEMM: output stride %d < %d columns", ldF, nCols);
    SQ_THROW_IF(fragElems < fieldFragElemsFP8(nCols, K), "fp8 fragment buffer too small");
    SQ_THROW_IF(!d_colScale, "fp8 field GEMM: no column scales");
    const int nColBlocks = nCols / 16, t = rowTilesFor(nColBlocks, m);
    const int nGroups = divru(divru(m, 16), t);
    auto *kernel = t == 4 ? fieldRefreshFP8Kernel<4> : t == 2 ? fieldRefreshFP8Kernel<2> : fieldRefreshFP8Kernel<1>;
    kernel<<<nColBlocks * nGroups, kBlockThreads, 0, stream>>>(reinterpret_cast<const uint4 *>(d_frag), d_colScale, d_Qbits,
                                                               nColBlocks, nGroups, K, m, Nw, ldF, d_F);
    HIP_CHECK(hipGetLastError());
}

void buildFragBF16x2(const float *d_B, int rows, int ld, int nCols, int K, uint16_t *d_frag, size_t fragElems,
                     hipStream_t stream) {
    checkGemm(nCols, K, ld, K / 32);
    SQ_THROW_IF(rows > nCols, "field GEMM: %d rows exceed %d columns", rows, nCols);
    SQ_THROW_IF(fragElems < fieldFragElemsBF16x2(nCols, K), "bf16x2 fragment buffer holds %zu of %zu elements",
                fragElems, fieldFragElemsBF16x2(nCols, K));
    const size_t threads = (size_t)(nCols / 16) * (K / 32) * kWave;
    buildFragBF16Kernel<2><<<(unsigned)((threads + 255) / 256), 256, 0, stream>>>(d_B, rows, ld, nCols / 16, K,
                                                                               reinterpret_cast<uint4 *>(d_frag));
    HIP_CHECK(hipGetLastError());
}

void buildFragF32(const float *d_B, int rows, int ld, int nCols, int K, uint16_t *d_frag, size_t fragElems,
                  hipStream_t stream) {
    checkGemm(nCols, K, ld, K / 32);
    SQ_THROW_IF(rows > nCols, "field GEMM: %d rows exceed %d columns", rows, nCols);
    SQ_THROW_IF(fragElems < fieldFragElemsF32(nCols, K), "fp32 fragment buffer holds %zu of %zu elements", fragElems,
                fieldFragElemsF32(nCols, K));
    const size_t threads = (size_t)(nCols / 16) * (K / 32) * kWave;
    buildFragBF16Kernel<3><<<(unsigned)((threads + 255) / 256), 256, 0, stream>>>(d_B, rows, ld, nCols / 16, K,
                                                                               reinterpret_cast<uint4 *>(d_frag));
    HIP_CHECK(hipGetLastError());
}

void fieldRefreshBF16x2(const uint16_t *d_frag, size_t fragElems, const uint32_t *d_Qbits, int nCols, int K, int m,
                        int Nw, int ldF, float *d_F, hipStream_t stream) {
    checkGemm(nCols, K, K, Nw);
    SQ_THROW_IF(ldF < nCols, "field GEMM: output stride %d < %d columns", ldF, nCols);
    SQ_THROW_IF(fragElems < fieldFragElemsBF16x2(nCols, K), "bf16x2 fragment buffer too small");
    const int nColBlocks = nCols / 16, t = rowTilesFor(nColBlocks, m);
    const int nGroups = divru(divru(m, 16), t);
    auto *kernel = t == 4 ? fieldRefreshBF16Kernel<2, 4> : t == 2 ? fieldRefreshBF16Kernel<2, 2> : fieldRefreshBF16Kernel<2, 1>;
    kernel<<<nColBlocks * nGroups, kBlockThreads, 0, stream>>>(reinterpret_cast<const uint4 *>(d_frag), d_Qbits,
                                                               nColBlocks, nGroups, K, m, Nw, ldF, d_F);
    HIP_CHECK(hipGetLastError());
}

void fieldRefreshF32MFMA(const uint16_t *d_frag, size_t fragElems, const uint32_t *d_Qbits, int nCols, int K,
                         int m, int Nw, int ldF, float *d_F, hipStream_t stream) {
    checkGemm(nCols, K, K, Nw);
    SQ_THROW_IF(ldF < nCols, "field GEMM: output stride %d < %d columns", ldF, nCols);
    SQ_THROW_IF(fragElems < fieldFragElemsF32(nCols, K), "fp32 fragment buffer too small");
    const int nColBlocks = nCols / 16, t = rowTilesFor(nColBlocks, m);
    const int nGroups = divru(divru(m, 16), t);
    auto *kernel = t == 4 ? fieldRefreshBF16Kernel<3, 4> : t == 2 ? fieldRefreshBF16Kernel<3, 2> : fieldRefreshBF16Kernel<3, 1>;
    kernel<<<nColBlocks * nGroups, kBlockThreads, 0, stream>>>(reinterpret_cast<const uint4 *>(d_frag), d_Qbits,
                                                               nColBlocks, nGroups, K, m, Nw, ldF, d_F);
    HIP_CHECK(hipGetLastError());
}

void fieldRefreshF64MFMA(const double *d_B, int K, int nCols, int ldB, const uint32_t *d_Qbits, int m, int Nw,
                         int ldF, double *d_F, hipStream_t stream) {
    SQ_THROW_IF(nCols <= 0 || nCols % 16 != 0, "field GEMM: %d output columns is not a positive multiple of 16",
                nCols);
    SQ_THROW_IF(K <= 0 || K > Nw * 32 || ldB < nCols || ldF < nCols || m <= 0, "field GEMM: inconsistent shape");
    /* row tiles per block: as many as leave two blocks to each of 256 CUs (a
     * tile more reads B's columns once for twice the slices) */
    const int colBlocks = nCols / 16, rowTiles = divru(m, 16);
    const int rt = colBlocks * divru(rowTiles, 4) >= 512 ? 4 : colBlocks * divru(rowTiles, 2) >= 512 ? 2 : 1;
    const dim3 grid((unsigned)colBlocks, (unsigned)divru(rowTiles, rt));
    auto *kernel = rt == 4 ? fieldRefreshF64Kernel<4> : rt == 2 ? fieldRefreshF64Kernel<2> : fieldRefreshF64Kernel<1>;
    kernel<<<grid, kBlockThreads, 0, stream>>>(d_B, K, ldB, d_Qbits, m, Nw, ldF, d_F);
    HIP_CHECK(hipGetLastError());
}

}  // namespace sqaod_rocm
