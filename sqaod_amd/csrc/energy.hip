/*
 * FP64 energy recompute for the annealers, evaluated in double from the
 * stored real J and h, with a fixed reduction order so the result does not
 * depend on scheduling:
 *   dense     E_y = -c - sum_i q_yi (h_i + sum_j J_ij q_yj)
 *             (DGFuncs::calculate_E, sqaodc/cpu/SharedFormulas.cpp:69-83);
 *   bipartite E_y = -c - h0.q0_y - sum_i q1_yi (h1_i + sum_j J_ij q0_yj)
 *             (BGFuncs::calculate_E, SharedFormulas.cpp:184-202).
 * Both are sums over "outer" spins of (h + B^T . inner spins): the partial
 * kernel takes the two spin sets separately.  Also the Trotter coupling
 * sum_y q_y . q_(y+1)%m of getSystemE (CPUDenseGraphAnnealer.cpp:236-240).
 */
#include "common.h"
#include "kernels.h"

namespace sqaod_rocm {

namespace {

constexpr int kCols = 256;
constexpr int kYTile = 16;

/* partial[y][bx] = sum over outer spins i in block bx's 256 columns (i < nOut)
 * of qo_yi (h_i + sum_{j<K} B[j][i] qi_yj); B row-major with stride ldB. */
template <class real>
__global__ __launch_bounds__(kCols) void energyPartialKernel(const real *B, int K, int ldB, const real *h,
                                                             const uint32_t *Qin, int NwIn, const uint32_t *Qout,
                                                             int NwOut, int nOut, int m, double *partial) {
    /* block (bx, by): columns i in [bx*256, +256), slices [by*16, +16) */
    __shared__ uint32_t qs[kYTile];
    __shared__ double red[kYTile][kCols / 64];
    const int i = blockIdx.x * kCols + threadIdx.x;
    const int y0 = blockIdx.y * kYTile;
    double acc[kYTile];
#pragma unroll
    for (int t = 0; t < kYTile; ++t)
        acc[t] = 0.;
    for (int j0 = 0; j0 < K; j0 += 32) {
        if (threadIdx.x < kYTile)
            qs[threadIdx.x] = (y0 + (int)threadIdx.x < m) ? Qin[(long long)(y0 + threadIdx.x) * NwIn + (j0 >> 5)] : 0u;
        __syncthreads();
        uint32_t qw[kYTile];
#pragma unroll
        for (int t = 0; t < kYTile; ++t)
            qw[t] = qs[t];
        const int jn = (K - j0) < 32 ? (K - j0) : 32;
        for (int jj = 0; jj < jn; ++jj) {
            /* sum_j B_ji q_j read down column i (coalesced) */
            const double v = (double)B[(long long)(j0 + jj) * ldB + i];
#pragma unroll
            for (int t = 0; t < kYTile; ++t)
                acc[t] += ((qw[t] >> jj) & 1u) ? v : -v;
        }
        __syncthreads();
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const bool colOk = i < nOut;
    const double hi = colOk ? (double)h[i] : 0.;
#pragma unroll
    for (int t = 0; t < kYTile; ++t) {
        double v = 0.;
        if (colOk && y0 + t < m) {
            const bool qp = (Qout[(long long)(y0 + t) * NwOut + (i >> 5)] >> (i & 31)) & 1u;
            const double s = hi + acc[t];
            v = qp ? s : -s;
        }
        /* wave reduction in a fixed butterfly order */
        for (int off = 32; off > 0; off >>= 1)
            v += __shfl_xor(v, off);
        if (lane == 0)
            red[t][wv] = v;
    }
    __syncthreads();
    if (threadIdx.x < kYTile) {
        const int t = threadIdx.x;
        if (y0 + t < m) {
            double s = ((red[t][0] + red[t][1]) + (red[t][2] + red[t][3]));
            partial[(long long)(y0 + t) * gridDim.x + blockIdx.x] = s;
        }
    }
}

/* E[y] = -c - (sum of partial0[y][:]) - (sum of partial1[y][:]) */
__global__ void energyFinalKernel(const double *partial0, int nPart0, const double *partial1, int nPart1, int m,
                                  double c, double *E) {
    int y = blockIdx.x * blockDim.x + threadIdx.x;
    if (y >= m)
        return;
    double s = 0.;
    for (int b = 0; b < nPart0; ++b)
        s += partial0[(long long)y * nPart0 + b];
    double s1 = 0.;
    for (int b = 0; b < nPart1; ++b)
        s1 += partial1[(long long)y * nPart1 + b];
    E[y] = -c - s - s1;
}

__global__ void spinDotSumKernel(const uint32_t *Qbits, int N, int m, int Nw, double *out) {
    /* one block; q_y . q_y' = N - 2 popcount(bits_y xor bits_y') (padding bits are 0 in both) */
    __shared__ long long red[256];
    long long acc = 0;
    for (long long idx = threadIdx.x; idx < (long long)m * Nw; idx += blockDim.x) {
        int y = (int)(idx / Nw), w = (int)(idx % Nw);
        int y1 = (y + 1) % m;
        acc += __popc(Qbits[(long long)y * Nw + w] ^ Qbits[(long long)y1 * Nw + w]);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        out[0] = (double)((long long)N * m - 2 * red[0]);
}

}  // namespace

template <class real>
void energyFP64(const real *d_J, const real *d_h, double c, const uint32_t *d_Qbits, int N, int Np, int m, int Nw,
                double *d_partial, double *d_E, hipStream_t stream) {
    dim3 grid(Np / kCols, divru(m, kYTile));
    energyPartialKernel<real><<<grid, kCols, 0, stream>>>(d_J, N, Np, d_h, d_Qbits, Nw, d_Qbits, Nw, N, m, d_partial);
    HIP_CHECK(hipGetLastError());
    energyFinalKernel<<<divru(m, 64), 64, 0, stream>>>(d_partial, (int)grid.x, nullptr, 0, m, c, d_E);
    HIP_CHECK(hipGetLastError());
}

template <class real>
void energyBipartiteFP64(const real *d_JT, const real *d_h0, const real *d_h1, double c, const uint32_t *d_Q0,
                         const uint32_t *d_Q1, int N0, int N1, int N0p, int N1p, int m, double *d_partial,
                         double *d_E, hipStream_t stream) {
    SQ_THROW_IF(N0p % kCols != 0 || N1p % kCols != 0, "bipartite energy: padded sizes must be multiples of %d", kCols);
    const int N0w = N0p / 32, N1w = N1p / 32;
    /* sum_i q1_i (h1_i + sum_j J_ij q0_j) = sum_i q1_i (h1_i + sum_j JT_ji q0_j) */
    dim3 g1(N1p / kCols, divru(m, kYTile));
    double *p1 = d_partial, *p0 = d_partial + (size_t)m * g1.x;
    energyPartialKernel<real><<<g1, kCols, 0, stream>>>(d_JT, N0, N1p, d_h1, d_Q0, N0w, d_Q1, N1w, N1, m, p1);
    HIP_CHECK(hipGetLastError());
    /* h0 . q0: the same kernel with an empty inner sum */
    dim3 g0(N0p / kCols, divru(m, kYTile));
    energyPartialKernel<real><<<g0, kCols, 0, stream>>>(d_JT, 0, N1p, d_h0, d_Q0, N0w, d_Q0, N0w, N0, m, p0);
    HIP_CHECK(hipGetLastError());
    energyFinalKernel<<<divru(m, 64), 64, 0, stream>>>(p1, (int)g1.x, p0, (int)g0.x, m, c, d_E);
    HIP_CHECK(hipGetLastError());
}

void spinDotSum(const uint32_t *d_Qbits, int N, int m, int Nw, double *d_out, hipStream_t stream) {
    spinDotSumKernel<<<1, 256, 0, stream>>>(d_Qbits, N, m, Nw, d_out);
    HIP_CHECK(hipGetLastError());
}

template void energyFP64<float>(const float *, const float *, double, const uint32_t *, int, int, int, int, double *,
                                double *, hipStream_t);
template void energyFP64<double>(const double *, const double *, double, const uint32_t *, int, int, int, int,
                                 double *, double *, hipStream_t);
template void energyBipartiteFP64<float>(const float *, const float *, const float *, double, const uint32_t *,
                                         const uint32_t *, int, int, int, int, int, double *, double *, hipStream_t);
template void energyBipartiteFP64<double>(const double *, const double *, const double *, double, const uint32_t *,
                                          const uint32_t *, int, int, int, int, int, double *, double *, hipStream_t);

}  // namespace sqaod_rocm

/* ---------------- system energy (dense getSystemE) ---------------- */

namespace sqaod_rocm {

namespace {

template <class real>
__global__ void systemEnergyKernel(const double *E, int m, real sgnE, const double *spinDot, int sqa, real coef,
                                   real sgnOut, real *out) {
    real s = (real)0.;
    for (int y = 0; y < m; ++y)
        s += sgnE * (real)E[y];
    s = s / (real)m;
    if (sqa)
        s -= (real)spinDot[0] * coef;
    out[0] = s * sgnOut;
}

}  // namespace

template <class real>
void systemEnergy(const double *d_E, int m, real sgnE, const double *d_spinDot, int sqa, real coef, real sgnOut,
                  real *d_out, hipStream_t stream) {
    systemEnergyKernel<real><<<1, 1, 0, stream>>>(d_E, m, sgnE, d_spinDot, sqa, coef, sgnOut, d_out);
    HIP_CHECK(hipGetLastError());
}

template void systemEnergy<float>(const double *, int, float, const double *, int, float, float, float *,
                                  hipStream_t);
template void systemEnergy<double>(const double *, int, double, const double *, int, double, double, double *,
                                   hipStream_t);

}  // namespace sqaod_rocm

/* ---------------- batched bilinear forms (the formulas objects) ---------------- */

namespace sqaod_rocm {

namespace {

constexpr int kQfThreads = 256;
constexpr int kSymTile = 32; /* of the symmetry check */
constexpr int kQfTile = 32; /* rows of V, rows of A and columns of both in a tile */

/* E[o] = cst + sgn (sum_j lin0[j] v[j] + sum_i u[i] (lin1[i] + sum_j A[i][j] v[j])),
 * u = U[iu[o]] (nu entries), v = V[iv[o]] (nv entries), int8 vectors; FP64
 * accumulation, fixed reduction order.
 *
 * Two launches.  quadGemmKernel forms G[b][i] = sum_j A[i][j] V[b][j] on
 * v_mfma_f64_16x16x4_f64 (a block: a 32 x 32 tile of G, a 16 x 16 tile a wave,
 * A and V staged through LDS as doubles, the next tile's loads in flight) and
 * either multiplies by u and sums over its 16 rows of A (one output per row of
 * V: partial[b][i / 16]) or stores lin1[i] + G[b][i] (all pairs).
 * quadFormKernel adds those up per output.  A then is read nV / 32 times, whole
 * lines at a time, where one block per output read all of it column by column
 * for each output; all pairs cost nu nv nV + nu nOut operations instead of
 * nu nv nOut.
 *
 * An element of A that is not finite must count only where its v and u are not
 * zero, which a product with zero does not give: such an A (or a stored sum
 * that is not finite) is flagged and quadFormKernel evaluates the outputs term
 * by term.  So it does where nu nv <= kQfDirect, in one launch: a whole call on
 * 100 pairs of float vectors takes 43 us against 45 for 20 x 20 that way, 50
 * against 51 for 40 x 50, and 46 against 44 for 64 x 64.  (All pairs of many
 * vectors would gain by the two launches sooner: 100 x 100 pairs of 20 x 20,
 * 75 against 68 us.)
 * Measured, 1000 x 1000 floats and 500 vectors: 39.9 + 5.7 us against 702 us
 * for the one-launch form; bound by the round trip of a tile's loads (the
 * products alone take 14 us at the 71 TFLOP/s a large FP64 product reaches). */
constexpr long long kQfDirect = 4096;

typedef double f64x4 __attribute__((ext_vector_type(4)));

template <class real>
__global__ __launch_bounds__(kQfThreads) void quadGemmKernel(QuadFormArgs<real> a, double *work, int *flags) {
    /* tile rows padded to 33 doubles: 16 lanes reading one column meet 16 bank pairs */
    __shared__ double sA[2][kQfTile][kQfTile + 1], sV[2][kQfTile][kQfTile + 1];
    __shared__ int sFlag;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    const int i0 = blockIdx.x * kQfTile, b0 = blockIdx.y * kQfTile;
    const int wb = (w >> 1) * 16, wi = (w & 1) * 16; /* the wave's tile */
    const int lr = threadIdx.x / kQfTile, lc = threadIdx.x % kQfTile;
    constexpr int kPer = kQfTile * kQfTile / kQfThreads;
    bool finite = true;
    real ra[kPer];
    int8_t rv[kPer];
    auto fetch = [&](int j0) {
        const int j = j0 + lc;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int r = lr + k * (kQfTile / kPer);
            ra[k] = (i0 + r < a.nu && j < a.nv) ? a.A[(size_t)(i0 + r) * a.nv + j] : (real)0;
            rv[k] = (b0 + r < a.nV && j < a.nv) ? a.V[(size_t)(b0 + r) * a.nv + j] : (int8_t)0;
        }
    };
    if (threadIdx.x == 0)
        sFlag = 0;
    f64x4 acc = {0., 0., 0., 0.};
    fetch(0);
    int buf = 0;
    for (int j0 = 0; j0 < a.nv; j0 += kQfTile, buf ^= 1) {
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int r = lr + k * (kQfTile / kPer);
            sA[buf][r][lc] = (double)ra[k];
            sV[buf][r][lc] = (double)rv[k];
            finite = finite && isfinite(ra[k]);
        }
        __syncthreads(); /* one a tile: the other buffer was read before the last one */
        if (j0 + kQfTile < a.nv)
            fetch(j0 + kQfTile);
#pragma unroll
        for (int t = 0; t < kQfTile / 4; ++t)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(sV[buf][wb + c][4 * t + g], sA[buf][wi + c][4 * t + g], acc, 0,
                                                       0, 0);
    }
    /* register r: row b0 + wb + 4 r + g of V, row i of A */
    const int i = i0 + wi + c;
    const double l1 = (a.lin1 && i < a.nu) ? (double)a.lin1[i] : 0.;
    if (a.twoD) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int b = b0 + wb + 4 * r + g;
            const double v = l1 + acc[r];
            if (b < a.nV && i < a.nu) {
                work[(size_t)b * a.nu + i] = v;
                finite = finite && isfinite(v);
            }
        }
    } else {
        const int nPart = (a.nu + 15) / 16;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int b = b0 + wb + 4 * r + g;
            const int u = (b < a.nV && i < a.nu) ? a.U[(size_t)b * a.nu + i] : 0;
            double v = u ? (double)u * (l1 + acc[r]) : 0.;
#pragma unroll
            for (int off = 8; off > 0; off >>= 1)
                v += __shfl_xor(v, off);
            if (c == 0 && b < a.nV && i < a.nu)
                work[(size_t)b * nPart + (i0 + wi) / 16] = v;
        }
    }
    if (!finite)
        sFlag = 1;
    __syncthreads();
    if (threadIdx.x == 0)
        flags[blockIdx.y * gridDim.x + blockIdx.x] = sFlag;
}

/* One block per output.  work == nullptr: term by term. */
template <class real>
__global__ __launch_bounds__(kQfThreads) void quadFormKernel(QuadFormArgs<real> a, const double *work, const int *flags,
                                                             int nFlags) {
    __shared__ double red[kQfThreads];
    const int o = blockIdx.x;
    const int bu = a.twoD ? o / a.nV : o;
    const int bv = a.twoD ? o % a.nV : o;
    const int8_t *u = a.U + (size_t)bu * a.nu;
    const int8_t *v = a.V + (size_t)bv * a.nv;
    int direct = work == nullptr;
    if (!direct) {
        for (int f = threadIdx.x; f < nFlags; f += kQfThreads)
            direct |= flags[f];
        direct = __syncthreads_or(direct);
    }
    double s = 0.;
    if (direct) {
        for (int i = threadIdx.x; i < a.nu; i += kQfThreads) {
            if (u[i] == 0)
                continue;
            double r = a.lin1 ? (double)a.lin1[i] : 0.;
            const real *Ai = a.A + (size_t)i * a.nv;
            for (int j = 0; j < a.nv; ++j)
                if (v[j])
                    r += (double)Ai[j] * (double)v[j];
            s += (double)u[i] * r;
        }
    } else if (a.twoD) {
        for (int i = threadIdx.x; i < a.nu; i += kQfThreads)
            s += (double)u[i] * work[(size_t)bv * a.nu + i];
    } else {
        const int nPart = (a.nu + 15) / 16;
        for (int p = threadIdx.x; p < nPart; p += kQfThreads)
            s += work[(size_t)o * nPart + p];
    }
    if (a.lin0)
        for (int j = threadIdx.x; j < a.nv; j += kQfThreads)
            s += (double)a.lin0[j] * (double)v[j];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = kQfThreads / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        a.E[o] = (real)(a.cst + a.sgn * red[0]);
}

/* Sets *asymmetric where A != A^T in any element (NaN differs from itself, as in
 * a comparison on the host): a block compares a pair of tiles on either side
 * of the diagonal, one of them turned in LDS, so both are read by rows.
 * It reads A once.  Energies of 16 float states, the comparison on the host /
 * here: 772 / 280 us at N = 1000, 2674 / 623 at N = 2000. */
template <class real>
__global__ __launch_bounds__(kQfThreads) void symmetricKernel(const real *A, int N, int *asymmetric) {
    __shared__ real turned[kSymTile][kSymTile + 1];
    /* pair p of the lower triangle of tiles: row ti, column tj <= ti */
    const long long p = blockIdx.x;
    int ti = (int)((sqrt(8. * (double)p + 1.) - 1.) / 2.);
    while ((long long)(ti + 1) * (ti + 2) / 2 <= p)
        ++ti;
    while ((long long)ti * (ti + 1) / 2 > p)
        --ti;
    const int tj = (int)(p - (long long)ti * (ti + 1) / 2);
    const int col = threadIdx.x % kSymTile, row0 = threadIdx.x / kSymTile;
    constexpr int kRows = kQfThreads / kSymTile;
    real a[kSymTile / kRows];
#pragma unroll
    for (int r = 0; r < kSymTile / kRows; ++r) {
        const int row = row0 + r * kRows;
        const int ia = ti * kSymTile + row, ja = tj * kSymTile + col;
        a[r] = ia < N && ja < N ? A[(long long)ia * N + ja] : real(0.);
        const int ib = tj * kSymTile + row, jb = ti * kSymTile + col;
        turned[col][row] = ib < N && jb < N ? A[(long long)ib * N + jb] : real(0.);
    }
    __syncthreads();
    bool differs = false;
#pragma unroll
    for (int r = 0; r < kSymTile / kRows; ++r)
        differs = differs || !(a[r] == turned[row0 + r * kRows][col]);
    if (differs)
        __hip_atomic_store(asymmetric, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

int quadFormBlocks(int nu, int nV) { return divru(nu, kQfTile) * divru(nV, kQfTile); }

}  // namespace

size_t quadFormWorkBytes(int nu, int nv, int nV, bool twoD) {
    const size_t sums = (size_t)nV * (size_t)(twoD ? nu : divru(nu, 16));
    /* beyond the grid's rows, or 2 GiB of sums: term by term as well */
    if ((long long)nu * nv <= kQfDirect || divru(nV, kQfTile) > 65535 || sums > ((size_t)1 << 28))
        return 0;
    return sums * sizeof(double) + (size_t)quadFormBlocks(nu, nV) * sizeof(int);
}

template <class real>
void quadForm(const QuadFormArgs<real> &a, int nOut, void *d_work, size_t workBytes, hipStream_t stream) {
    if (nOut <= 0)
        return;
    SQ_THROW_IF(a.nu <= 0 || a.nv <= 0 || a.nV <= 0, "bilinear form: empty vectors");
    const size_t need = quadFormWorkBytes(a.nu, a.nv, a.nV, a.twoD != 0);
    SQ_THROW_IF(workBytes < need, "bilinear form: workspace of %zu of %zu bytes", workBytes, need);
    double *work = need ? (double *)d_work : nullptr;
    const int nBlocks = need ? quadFormBlocks(a.nu, a.nV) : 0;
    int *flags = (int *)((char *)d_work + need - (size_t)nBlocks * sizeof(int));
    if (work) {
        const dim3 grid((unsigned)divru(a.nu, kQfTile), (unsigned)divru(a.nV, kQfTile));
        quadGemmKernel<real><<<grid, kQfThreads, 0, stream>>>(a, work, flags);
        HIP_CHECK(hipGetLastError());
    }
    quadFormKernel<real><<<nOut, kQfThreads, 0, stream>>>(a, work, flags, nBlocks);
    HIP_CHECK(hipGetLastError());
}

template void quadForm<float>(const QuadFormArgs<float> &, int, void *, size_t, hipStream_t);
template void quadForm<double>(const QuadFormArgs<double> &, int, void *, size_t, hipStream_t);

template <class real>
void symmetricCheck(const real *d_A, int N, int *d_asymmetric, hipStream_t stream) {
    const long long tiles = divru(N, kSymTile), pairs = tiles * (tiles + 1) / 2;
    SQ_THROW_IF(N <= 0 || pairs > 0x7fffffff, "symmetry check: bad size %d", N);
    HIP_CHECK(hipMemsetAsync(d_asymmetric, 0, sizeof(int), stream));
    symmetricKernel<real><<<(unsigned)pairs, kQfThreads, 0, stream>>>(d_A, N, d_asymmetric);
    HIP_CHECK(hipGetLastError());
}

template void symmetricCheck<float>(const float *, int, int *, hipStream_t);
template void symmetricCheck<double>(const double *, int, int *, hipStream_t);

}  // namespace sqaod_rocm
