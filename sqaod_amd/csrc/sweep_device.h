/*
 * What the sweep kernels share (dense_sweep.hip, dense_sweep_team.hip): device
 * scope loads and stores, LDS DMA from inline assembly with explicit waits, row
 * additions to LDS-resident fields.  Included inside an anonymous namespace's
 * users only; everything here is device code.
 */
#pragma once

#include "common.h"
#include "kernels.h"
#include "sq_expf.h"

#include <type_traits>

namespace sqaod_rocm {

namespace {

constexpr int kWave = 64;
constexpr size_t kExpTabBytes = 32 * sizeof(uint64_t); /* LDS copy of the exp table */

__device__ __forceinline__ uint32_t loadShared32(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void storeShared32(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void waveSync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ int firstLane(unsigned long long mask) {
    return mask ? (int)__builtin_ctzll(mask) : kWave;
}

/* lane l's float (l wave-uniform) */
__device__ __forceinline__ float readLaneF(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

/* A wave-uniform int, marked so: control values the compiler cannot prove
 * uniform (they pass through loops with ballot-dependent exits) would
 * otherwise live in VGPRs and turn every branch on them into exec masking. */
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

/* LDS DMA issued from inline assembly: lane i's 4 (16) bytes from src land at
 * ldsDst + 4i (16i).  The compiler sees neither the op nor its LDS write, so
 * it adds no memory waits for it (for the builtin form it waits for every
 * outstanding DMA before any later LDS access, which serialises the batch
 * loop); every read of a DMA destination follows an explicit vmWait instead.
 * Ops the compiler does not count only make its own waits stricter (vmcnt
 * retires in issue order), never weaker.  M0 carries the LDS address; nothing
 * else in the sweep kernels uses M0.  kCoherent: the cache policy of a relaxed
 * atomic load at agent scope (decisions published by other waves). */
/* the M0 clobber below is deliberate (clang warns about any M0 clobber) */
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ uint32_t ldsAddress(const void *p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p);
}
template <bool kCoherent>
__device__ __forceinline__ void dmaDword(const void *src, uint32_t lds) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(lds);
    if constexpr (kCoherent)
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off sc1" ::"v"(src), "s"(m) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(m) : "memory", "m0");
}
__device__ __forceinline__ void dmaDwordx4(const void *src, uint32_t lds) {
    const uint32_t m = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m) : "memory", "m0");
}
/* n consecutive 1 KiB DMA ops (16 B per lane): op i reads the wave-uniform src + i
 * KiB and lands at LDS byte address lds + i KiB.  The ops' immediate offset
 * counts for both addresses, so groups of four take one M0 write and one scalar
 * base: half the instructions of a 64-bit lane address and an M0 step per op
 * (a wait state after the M0 write before the DMA reads it). */
__device__ __forceinline__ void dmaRunx4(const unsigned char *src, uint32_t lds, int n) {
    const uint32_t at = (threadIdx.x & (kWave - 1)) * 16;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)src);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uintptr_t)src >> 32));
    const unsigned long long base = (unsigned long long)hi << 32 | lo;
    int i = 0;
    for (; i + 4 <= n; i += 4) { /* n is wave-uniform: a scalar loop */
        const uint32_t m = __builtin_amdgcn_readfirstlane(lds + (uint32_t)i * 1024u);
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
                     "global_load_lds_dwordx4 %0, %1\n\t"
                     "global_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                     "global_load_lds_dwordx4 %0, %1 offset:2048\n\t"
                     "global_load_lds_dwordx4 %0, %1 offset:3072" ::"v"(at),
                     "s"(base + (unsigned long long)i * 1024), "s"(m)
                     : "memory", "m0");
    }
    for (; i < n; ++i)
        dmaDwordx4(src + (size_t)i * 1024 + at, lds + (uint32_t)i * 1024u);
}
#pragma clang diagnostic pop

/* wait until at most C vector-memory ops are outstanding */
template <int C>
__device__ __forceinline__ void vmWaitImm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C) : "memory");
}
template <int LO, int HI>
__device__ __forceinline__ void vmWaitRange(int c) {
    if constexpr (LO == HI) {
        vmWaitImm<LO>();
    } else {
        constexpr int MID = (LO + HI + 1) / 2;
        if (c >= MID)
            vmWaitRange<MID, HI>(c);
        else
            vmWaitRange<LO, MID - 1>(c);
    }
}
/* vmcnt(c) for a wave-uniform c (counts above 63 wait for 63) */
__device__ __forceinline__ void vmWait(int c) {
    c = __builtin_amdgcn_readfirstlane(c);
    if (c == 1) /* the common case: only a decision store since */
        vmWaitImm<1>();
    else
        vmWaitRange<0, 63>(c < 63 ? c : 63);
}
/* this wave's LDS reads have returned (before a DMA overwrites what they read) */
__device__ __forceinline__ void ldsWait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

/* Copy kEntries entries of ES bytes, from entry e0 of src, into LDS at lds by
 * DMA, skipping entries >= limit (their LDS words keep old contents). */
template <int ES, bool kCoherent, int kEntries>
__device__ __forceinline__ void dmaEntries(const void *src, uint32_t lds, int e0, int limit) {
    const int lane = threadIdx.x & (kWave - 1);
    constexpr int kOps = kEntries * ES / (4 * kWave);
    const uint32_t *s = reinterpret_cast<const uint32_t *>(src) + lane;
    if (e0 + kEntries <= limit) {
#pragma unroll
        for (int j = 0; j < kOps; ++j)
            dmaDword<kCoherent>(s + j * kWave, lds + j * kWave * 4);
    } else {
#pragma unroll
        for (int j = 0; j < kOps; ++j)
            if (e0 + (j * kWave + lane) * 4 / ES < limit)
                dmaDword<kCoherent>(s + j * kWave, lds + j * kWave * 4);
    }
}

__device__ __forceinline__ int slicePos(int y, int m) {
    int nEven = (m + 1) / 2;
    return (y & 1) ? nEven + (y >> 1) : (y >> 1);
}

template <class real>
__device__ __forceinline__ void ldsLoad4(const real *p, real v[4]) {
    if constexpr (sizeof(real) == 4) {
        float4 t = *reinterpret_cast<const float4 *>(p);
        v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
    } else {
        double2 t0 = *reinterpret_cast<const double2 *>(p);
        double2 t1 = *reinterpret_cast<const double2 *>(p + 2);
        v[0] = t0.x; v[1] = t0.y; v[2] = t1.x; v[3] = t1.y;
    }
}

template <class real>
__device__ __forceinline__ void ldsStore4(real *p, const real v[4]) {
    if constexpr (sizeof(real) == 4) {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
        *reinterpret_cast<double2 *>(p) = make_double2(v[0], v[1]);
        *reinterpret_cast<double2 *>(p + 2) = make_double2(v[2], v[3]);
    }
}

template <class real>
struct Expo;
template <>
struct Expo<float> {
    /* the CPU annealer's expf(-dE*beta), bit-identical (sq_expf.h) */
    __device__ static float eval(float v, const uint64_t *tab) { return sq_expf_tab(v, tab); }
};
template <>
struct Expo<double> {
    __device__ static double eval(double v, const uint64_t *) { return exp(v); }
};

/* 4 e4m3 bytes -> floats (exact), gfx950's OCP FP8 conversion */
__device__ __forceinline__ void fp8x4ToFloat(uint32_t w, float v[4]) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
    const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    v[0] = lo.x; v[1] = lo.y; v[2] = hi.x; v[3] = hi.y;
}

/* f + d * v for a field update: d is -+2 (fp8 rows: -+2 times the row's
 * power-of-two scale) and v a J element, so d * v is exact and one fused
 * multiply-add rounds exactly as the separate multiply and add do. */
__device__ __forceinline__ float addScaled(float f, float d, float v) { return __builtin_fmaf(d, v, f); }
__device__ __forceinline__ double addScaled(double f, double d, double v) { return __builtin_fma(d, v, f); }

/* F[b0 ..] += d * sb[b0 ..] for R consecutive 256-element slices: all their
 * LDS reads are issued before the first write, so the round trips overlap.
 * FP8: sb holds e4m3 bytes. */
template <class real, bool FP8, int R>
__device__ __forceinline__ void addStagedSlices(real *F, const real *sb, real d, int b0, int lane) {
#pragma clang fp contract(off)
    const uint8_t *sb8 = reinterpret_cast<const uint8_t *>(sb);
    (void)sb8;
    real fv[R][4], sv[R][4];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = b0 + r * kWave * 4 + lane * 4;
        ldsLoad4(F + j, fv[r]);
        if constexpr (FP8)
            fp8x4ToFloat(*reinterpret_cast<const uint32_t *>(sb8 + j), sv[r]);
        else
            ldsLoad4(sb + j, sv[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = b0 + r * kWave * 4 + lane * 4;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            fv[r][t] = addScaled(fv[r][t], d, sv[r][t]);
        ldsStore4(F + j, fv[r]);
    }
}

/* F += d * (staged row sb): rounds of kR 256-element slices, then single
 * slices for the rest (Np is a multiple of 256).  The rounds carry no
 * per-slice bounds checks, so their reads go out back to back. */
template <class real, bool FP8, int kR = 4>
__device__ __forceinline__ void addStagedRow(real *F, const real *sb, real d, int Np, int lane) {
    int b0 = 0;
    /* b0 and the bounds are wave-uniform: scalar loops */
    for (; b0 + kR * kWave * 4 <= Np; b0 += kR * kWave * 4)
        addStagedSlices<real, FP8, kR>(F, sb, d, b0, lane);
    for (; b0 < Np; b0 += kWave * 4)
        addStagedSlices<real, FP8, 1>(F, sb, d, b0, lane);
}

}  // namespace

}  // namespace sqaod_rocm
