/*
 * Flip phase of the bipartite annealer's half-steps
 * (CPUBipartiteGraphAnnealer.cpp:331-362 coloring, :485-530 SA coloring).
 *
 * Within a half-step the annealed part's spins do not interact with each
 * other: spin (im, iq) sees only the fixed part through dEmat[im][iq], its
 * field h[iq] and the same site of the two neighbouring Trotter slices.  The
 * CPU visits even slices, then odd slices, each site in order; since every
 * decision depends only on slices of the other colour, all sites of one
 * colour are decided at once.  A phase is one launch over (slice, 64-site
 * group): one wave per group, decisions collected with a ballot, each wave
 * rewriting the two spin words it owns.  With m odd, slices 0 and m-1 are
 * both even and adjacent, and the CPU reaches m-1 after 0, so m-1 is a phase
 * of its own between the even and the odd phase.
 *
 * The uniform of spin (im, iq) is the one the serial CPU order assigns it:
 * position rank(im) * N + iq of the half-step's stream (rank = position of
 * im in the visiting order), so an MT19937 replay matches sqaod.cpu bit for
 * bit; the Philox stream keys the same position.
 */
#include "common.h"
#include "kernels.h"
#include "rng_device.h"
#include "sq_expf.h"

#include <algorithm>

namespace sqaod_rocm {

namespace {

constexpr int kWave = 64;
constexpr int kMaxThreads = 1024;
constexpr int kSites = 8; /* of a block of all phases */
/* One launch for all phases up to here: it decides each spin for the three
 * sums its neighbours can have, which costs more than a launch once the chip
 * is full.  Kernel time of a half-step (two phases): 3.7 against 2 x 2.9 us
 * at 1024 x 64 spins, 6.6 against 2 x 4.8 at 8192 x 64, 9.8 against 2 x 4.9
 * at 4096 x 256, 16.2 against 2 x 7.2 at 8192 x 256. */
constexpr long long kMaxFusedSpins = 1 << 20;
/* A block walks all slices of its 8 sites, 128 at a time, however few blocks
 * there are, so it loses to launches over slices and sites once the slices are
 * many: two for an even number, three for an odd one.  A step (us, one launch a
 * side / by phase, N0 = N1; float): N = 64: 14.9 / 19.1 with m = 192, 20.0 /
 * 19.0 with 256, 73 / 19 with 2048, 19.7 / 27.3 with 321, 25.4 / 28.2 with 511;
 * N = 1024: 21.3 / 22.7, 27.5 / 23.8, (1024 slices) 65 / 47, 28.7 / 31.4,
 * 36.6 / 34.8; double N = 64: 15.1 / 16.6, 19.5 / 18.8, 74 / 18, 20.0 / 21.6,
 * 25.1 / 21.7. */
constexpr int kMaxFusedSlicesEven = 192, kMaxFusedSlicesOdd = 320;

template <class real>
__device__ __forceinline__ real expNeg(real x);
template <>
__device__ __forceinline__ float expNeg<float>(float x) {
    return sq_expf(x);
}
template <>
__device__ __forceinline__ double expNeg<double>(double x) {
    return exp(x);
}

/* The uniform of spin (im, iq). */
template <class real>
__device__ __forceinline__ real uniformOf(const BGFlipArgs<real> &a, int im, int iq) {
    /* position of this spin in the serial visiting order */
    const int rank = a.sa ? im : ((im & 1) ? a.nEven + (im >> 1) : (im >> 1));
    const long long pos = (long long)rank * a.N + iq;
    if (a.words) {
        if (sizeof(real) == 4)
            return (real)wordToUniform(a.words[pos]);
        return (real)wordsToUniform(a.words[2 * pos], a.words[2 * pos + 1]);
    }
    const U4 r = philox4x32_10(U4{(uint32_t)pos, (uint32_t)(pos >> 32), a.ctr0, a.ctr1}, a.key0, a.key1);
    return (sizeof(real) == 4) ? (real)wordToUniform(r.x) : (real)wordsToUniform(r.x, r.y);
}

template <class real>
__global__ __launch_bounds__(kWave) void bgFlipKernel(BGFlipArgs<real> a) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x;
    const int iq = blockIdx.x * kWave + lane;
    const int im = a.slice0 + (int)blockIdx.y * a.sliceStep;
    const bool valid = iq < a.N;
    const long long wordIdx = (long long)im * a.Nw + (iq >> 5);
    const uint32_t myWord = a.Q[(long long)im * a.Nw + ((blockIdx.x * kWave + (lane & 32)) >> 5)];
    bool flip = false;
    if (valid) {
        const real q = ((myWord >> (iq & 31)) & 1u) ? real(1.) : real(-1.);
        const real dEv = a.dEmat[(long long)im * a.ldE + iq];
        real dE;
        if (a.sa) {
            /* tryFlipSA, :485-496 */
            dE = real(2.) * q * (a.h[iq] + dEv);
        } else {
            /* tryFlip, :331-344 (no factor 2 on dEmat) */
            const int n0 = (im + a.m - 1) % a.m, n1 = (im + 1) % a.m;
            const real q0 = ((a.Q[(long long)n0 * a.Nw + (iq >> 5)] >> (iq & 31)) & 1u) ? real(1.) : real(-1.);
            const real q1 = ((a.Q[(long long)n1 * a.Nw + (iq >> 5)] >> (iq & 31)) & 1u) ? real(1.) : real(-1.);
            dE = a.twoDivM * q * (a.h[iq] + dEv);
            dE -= q * (q0 + q1) * a.coef;
        }
        const real thresh = dE < real(0.) ? real(1.) : expNeg<real>(-dE * a.beta);
        const real u = uniformOf(a, im, iq);
        flip = thresh > u;
    }
    /* lanes 0..31 own word 2*bx, lanes 32..63 word 2*bx+1 of the row */
    const unsigned long long mask = __ballot(flip);
    if ((lane & 31) == 0 && (blockIdx.x * kWave + lane) < a.Nw * 32) {
        const uint32_t bits = (uint32_t)(mask >> (lane & 32));
        a.Q[wordIdx] = myWord ^ bits;
    }
}

/* All phases of a coloring half-step.  The phases of different sites do not
 * interact, so a block owns one byte (8 sites) of every slice.  What a spin
 * does is worked out for both neighbours down, one up and both up, all slices
 * at once; the phases are then bit operations on bytes in LDS, a barrier
 * between them.  Bound by latency (launch, loads, exp): 8 sites a block
 * rather than 32 put four times the blocks on the chip, 3.7 against 5.9 us at
 * N = 1024, m = 64, and no slower up to 16384 x 64 (10.0, 9.7).  Half-step of
 * 1024 x 64 in two launches: 5.8 us; of 200 x 125 float64 in three: 13.7, now
 * 4.5. */
template <class real>
__global__ __launch_bounds__(kMaxThreads) void bgFlipsKernel(BGFlipArgs<real> a) {
#pragma clang fp contract(off)
    extern __shared__ uint8_t spins[];
    uint8_t *const ifDown = spins + a.m, *const ifMixed = ifDown + a.m, *const ifUp = ifMixed + a.m;
    uint8_t *const Q = reinterpret_cast<uint8_t *>(a.Q) + blockIdx.x;
    const long long ldQ = (long long)a.Nw * 4;
    const int site = threadIdx.x % kSites, iq = blockIdx.x * kSites + site;
    const int shift = (threadIdx.x & (kWave - 1)) - site; /* of this slice's bits in a ballot */

    for (int im = threadIdx.x / kSites; im < a.m; im += blockDim.x / kSites) {
        const uint8_t w = Q[im * ldQ];
        bool down = false, mixed = false, up = false;
        if (iq < a.N) {
            /* tryFlip, :331-344 (no factor 2 on dEmat) */
            const real q = ((w >> site) & 1u) ? real(1.) : real(-1.);
            const real field = a.twoDivM * q * (a.h[iq] + a.dEmat[(long long)im * a.ldE + iq]);
            const real u = uniformOf(a, im, iq);
            const auto flips = [&](real neighbours) {
                const real dE = field - q * neighbours * a.coef;
                const real thresh = dE < real(0.) ? real(1.) : expNeg<real>(-dE * a.beta);
                return thresh > u;
            };
            down = flips(real(-2.));
            mixed = flips(real(0.));
            up = flips(real(2.));
        }
        const unsigned long long bDown = __ballot(down), bMixed = __ballot(mixed), bUp = __ballot(up);
        if (site == 0) {
            spins[im] = w;
            ifDown[im] = (uint8_t)(bDown >> shift);
            ifMixed[im] = (uint8_t)(bMixed >> shift);
            ifUp[im] = (uint8_t)(bUp >> shift);
        }
    }
    __syncthreads();

    const auto decide = [&](int im) {
        const uint8_t w = spins[im], n0 = spins[im == 0 ? a.m - 1 : im - 1], n1 = spins[im == a.m - 1 ? 0 : im + 1];
        const uint8_t now = w ^ ((n0 & n1 & ifUp[im]) | ((n0 ^ n1) & ifMixed[im]) | (~(n0 | n1) & ifDown[im]));
        spins[im] = now;
        Q[im * ldQ] = now;
    };
    /* even slices (all of them when m is even; without m-1 when m is odd) */
    for (int im = 2 * threadIdx.x; im < a.m / 2 * 2; im += 2 * blockDim.x)
        decide(im);
    __syncthreads();
    if (a.m % 2 == 1) {
        /* slice m-1: even, adjacent to slice 0, visited after it */
        if (threadIdx.x == 0)
            decide(a.m - 1);
        __syncthreads();
    }
    for (int im = 2 * threadIdx.x + 1; im < a.m / 2 * 2; im += 2 * blockDim.x)
        decide(im);
}

}  // namespace

template <class real>
bool bipartiteFlips(const BGFlipArgs<real> &a, hipStream_t stream) {
    SQ_THROW_IF(a.N <= 0 || a.m <= 0 || a.Nw * 32 < a.N, "bipartite flips: bad row of %d spins in %d words", a.N, a.Nw);
    if (a.sa || a.m > (a.m % 2 ? kMaxFusedSlicesOdd : kMaxFusedSlicesEven) || (long long)a.N * a.m > kMaxFusedSpins)
        return false;
    const int threads = std::min(roundUp(a.m * kSites, kWave), kMaxThreads);
    bgFlipsKernel<real><<<divru(a.N, kSites), threads, (size_t)a.m * 4, stream>>>(a);
    HIP_CHECK(hipGetLastError());
    return true;
}

template bool bipartiteFlips<float>(const BGFlipArgs<float> &, hipStream_t);
template bool bipartiteFlips<double>(const BGFlipArgs<double> &, hipStream_t);

template <class real>
void bipartiteFlipPhase(const BGFlipArgs<real> &a, int nSlices, hipStream_t stream) {
    if (nSlices <= 0)
        return;
    SQ_THROW_IF(a.N <= 0 || a.Nw * 32 < a.N || a.Nw % 2 != 0, "bipartite flip: bad row of %d spins in %d words", a.N,
                a.Nw);
    SQ_THROW_IF(a.slice0 < 0 || a.slice0 + (nSlices - 1) * a.sliceStep >= a.m, "bipartite flip: slices out of range");
    dim3 grid((unsigned)divru(a.N, kWave), (unsigned)nSlices);
    bgFlipKernel<real><<<grid, kWave, 0, stream>>>(a);
    HIP_CHECK(hipGetLastError());
}

template void bipartiteFlipPhase<float>(const BGFlipArgs<float> &, int, hipStream_t);
template void bipartiteFlipPhase<double>(const BGFlipArgs<double> &, int, hipStream_t);

}  // namespace sqaod_rocm
