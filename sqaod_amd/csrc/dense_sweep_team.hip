/*
 * Dense-graph SQA sweep by a team of four waves per Trotter slice: one
 * annealOneStep with the semantics of dense_sweep.hip's kernels (the serial
 * coloring annealer's, sqaodc/cpu/CPUDenseGraphAnnealer.cpp:250-301, or the SA
 * annealer's, :341-371) and their results bit for bit: local fields in LDS,
 * speculative batches of 64 attempts that end at the first accepted flip,
 * waits only on serially earlier attempts of the neighbour slices.
 *
 * A sweep of low acceptance is bound by the instructions of one wave per
 * batch, most of them not about the batch's own outcome: registering the
 * neighbours' undecided attempts in a table, replaying their decisions,
 * exponentials, row additions.  Here the batch's wave does only what needs the
 * state of the moment:
 *
 *   sweeper  decides and commits the batches.
 *   rows     adds the J rows of committed flips to the fields (F += -+2 J[x][:])
 *            while the sweeper goes on; the sweeper's next batch adds the last
 *            row's elements, streamed into LDS meanwhile, to its own 64 fields.
 *   scout    prepares the attempts ahead of the sweeper, a chunk of 64 at a
 *            time, from what does not depend on any decision: the site; the
 *            least x = -dE beta that is accepted for the uniform
 *            (sq_exp_above; float only); and for each neighbour slice how far
 *            back its last and second to last attempt on the same site lie
 *            (a table of the last two attempts by site, by hash where N is
 *            large: a collision only makes a lane wait).
 *   watcher  reads the neighbours' published decisions over and over and tells
 *            the sweeper how far each is decided and which attempts flipped.
 *
 * Trotter coupling.  A slice publishes its decisions 16 to a word, with the
 * number decided and the sweep's tag, so that a neighbour's next 512 attempts
 * are one 128-byte read (of LDS, within a workgroup).  The sweeper keeps a mirror
 * of each neighbour's spins as of the attempts that precede its batch.  A lane
 * whose site no undecided or not yet mirrored attempt touches reads the spin
 * from the mirror; one such attempt: it decides under both outcomes and waits
 * only if they differ; more than one: it waits.
 *
 * Measured (us a sweep; one wave per slice with a second one for the rows /
 * this kernel), steps 3-19 and 20-204 of a 205-step schedule on integer
 * couplings: N=4096, m=256 float 430 / 231 and 243 / 109; N=1200, m=300 float
 * 131 / 101 and 90 / 54; N=128, m=32 float 56 / 44 and 50 / 19; N=500, m=125
 * double 83 / 43 and 63 / 30.  What bounds it now is the chain of a batch in the
 * sweeper: about 2300 cycles at N=4096, of which 600 are the decision itself and
 * 500 the commit, each operation waiting for the one before.
 */
#include "sweep_device.h"

namespace sqaod_rocm {

namespace {

constexpr int kTeamWaves = 4;
constexpr int kTeamMaxSlices = 4;
constexpr int kRing = 256;      /* prepared attempts, entry e at e % kRing */
constexpr int kNbRing = 1024;   /* the neighbours' sites, entry e at e % kNbRing */
constexpr int kMaxBack = 255;   /* how far back of its position a lane may look */
constexpr int kPerWord = 16;    /* decisions per published word */
constexpr int kWinWords = 32;   /* words of a neighbour's window */
constexpr int kFlipRing = 1024; /* a neighbour's flips not yet mirrored (attempts of kNbRing at most) */
constexpr int kExactTable = 1024; /* sizes up to which a chunk's shared slots are resolved */

/* a published word: tag (11 bits, never 0) | number decided (5 bits) | flips */
__host__ __device__ constexpr uint32_t teamTag(uint32_t tag) { return tag % kTeamTagPeriod + 1; }
__device__ __forceinline__ uint32_t packWord(uint32_t tag, int n, uint32_t flips) {
    return tag << 21 | (uint32_t)n << 16 | flips;
}
__device__ __forceinline__ int decidedIn(uint32_t word, uint32_t tag) {
    return (word >> 21) == tag ? (int)((word >> 16) & 31u) : 0;
}

/* words of a slice's own copy in LDS: a window read may run past the last */
__host__ __device__ inline int ownWords(int N) { return roundUp(divru(N, kPerWord) + kWinWords, 4); }

/* slots of the tables by site: a power of two, one per site up to 4096 */
int siteTableSize(int N) {
    int t = 256;
    while (t < N && t < 4096)
        t <<= 1;
    return t;
}
constexpr int kMinHashed = 1024; /* fewer slots where LDS is short */

/* A slice's LDS region: byte offsets, each a multiple of 16. */
struct TeamRegion {
    int F, stage, bits, table, masks, nbSites, ringS, ringT, ringC, flips, own, ctl, bytes;
};
template <class real>
__host__ __device__ inline TeamRegion teamRegion(int N, int Np, int tableN, int S) {
    TeamRegion r;
    const int row = Np * (int)sizeof(real);
    r.F = 0;
    r.stage = r.F + row;                 /* two rows */
    r.bits = r.stage + 2 * row;          /* own spins, the two mirrors */
    r.table = r.bits + 3 * (Np / 32) * 4;
    r.masks = r.table + 2 * tableN * 4;
    r.nbSites = r.masks + (N <= kExactTable ? tableN * 8 : 0);
    r.ringS = r.nbSites + 2 * kNbRing * 2;
    r.ringT = r.ringS + kRing * 4;
    r.ringC = r.ringT + kRing * (int)sizeof(real);
    r.flips = r.ringC + kRing * 4;
    r.own = r.flips + 2 * kFlipRing * 2;
    r.ctl = r.own + (S > 1 ? ownWords(N) * 4 : 0); /* for the slices of its workgroup */
    r.bytes = r.ctl + 64;
    return r;
}

/* control words (each written by one wave): the rows that the sweeper has handed
 * to the rows wave and those added to F; whether the last two rows handed over
 * have the factor -2; the chunks the scout has prepared; the sweeper's position;
 * per neighbour the attempts decided and the flips listed up to there */
enum { kCtlRows = 0, kCtlDone = 1, kCtlSign = 2, kCtlReady = 4, kCtlPos = 5, kCtlDecided = 6, kCtlFlips = 8, kCtlWords = 10 };
constexpr uint32_t kEnd = 0x7fffffff; /* rows, position: the sweeper has ended */

/* Relaxed LDS accesses with compiler barriers on both sides: a wave's LDS
 * operations execute in issue order, so what was written before such a store
 * is seen after such a load. */
__device__ __forceinline__ uint32_t ldsLoad(const uint32_t *p) {
    asm volatile("" ::: "memory");
    const uint32_t v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
    return v;
}
__device__ __forceinline__ void ldsStore(uint32_t *p, uint32_t v) {
    asm volatile("" ::: "memory");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ uint32_t ctlLoad(const uint32_t *p) {
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)ldsLoad(p));
}
__device__ __forceinline__ void ctlStore(uint32_t *p, uint32_t v) {
    if ((threadIdx.x & (kWave - 1)) == 0)
        ldsStore(p, v);
}

/* The slice's neighbours in the ring of slices and, for each, whether its
 * attempt of the same iteration precedes this slice's (even slices go first). */
struct Neighbours {
    int n[2], delta[2];
};
__device__ __forceinline__ Neighbours neighboursOf(int y, int m) {
    Neighbours b;
    b.n[0] = (y == 0) ? m - 1 : y - 1;
    b.n[1] = (y == m - 1) ? 0 : y + 1;
    const int pos = slicePos(y, m);
    b.delta[0] = slicePos(b.n[0], m) < pos ? 1 : 0;
    b.delta[1] = slicePos(b.n[1], m) < pos ? 1 : 0;
    return b;
}

/* The rows wave: adds the staged rows handed over to F, with the same operation
 * per element as the sweeper's correction of its own fields.  Row i is in stage
 * buffer i % 2. */
template <class real>
__device__ __forceinline__ void rowsLoop(int Np, unsigned char *region, const TeamRegion &r) {
    const int lane = threadIdx.x & (kWave - 1);
    real *const F = reinterpret_cast<real *>(region + r.F);
    const real *const stage = reinterpret_cast<const real *>(region + r.stage);
    uint32_t *const ctl = reinterpret_cast<uint32_t *>(region + r.ctl);
    for (uint32_t i = 0;; ++i) {
        uint32_t rows;
        while ((rows = ctlLoad(ctl + kCtlRows)) == i)
            __builtin_amdgcn_s_sleep(1);
        if (rows == kEnd)
            break;
        const bool negative = ctlLoad(ctl + kCtlSign + (i & 1u)) != 0;
        addStagedRow<real, false, 4>(F, stage + (size_t)(i & 1u) * Np, negative ? (real)-2. : (real)2., Np, lane);
        ldsWait(); /* the field stores are done */
        ctlStore(ctl + kCtlDone, i + 1);
    }
}

/* The scout: chunk by chunk, at most three chunks ahead of the sweeper's. */
template <class real>
__device__ __forceinline__ void scoutLoop(const SweepArgs<real> &a, int y, const uint64_t *expTab, unsigned char *region,
                          const TeamRegion &r, int tableN) {
    const int N = a.N, lane = threadIdx.x & (kWave - 1);
    const int nChunks = divru(N, kWave);
    const Neighbours nb = neighboursOf(y, a.m);
    uint32_t *const table = reinterpret_cast<uint32_t *>(region + r.table);
    unsigned long long *const masks = reinterpret_cast<unsigned long long *>(region + r.masks);
    uint16_t *const nbSites = reinterpret_cast<uint16_t *>(region + r.nbSites);
    uint32_t *const ringS = reinterpret_cast<uint32_t *>(region + r.ringS);
    real *const ringT = reinterpret_cast<real *>(region + r.ringT);
    uint32_t *const ringC = reinterpret_cast<uint32_t *>(region + r.ringC);
    uint32_t *const ctl = reinterpret_cast<uint32_t *>(region + r.ctl);
    const uint32_t mask = (uint32_t)tableN - 1u;
    const uint32_t *Xo = a.X + (long long)y * N, *X0 = a.X + (long long)nb.n[0] * N, *X1 = a.X + (long long)nb.n[1] * N;
    const real *Uo = a.U + (long long)y * N;
    uint32_t s = 0, xn[2] = {0, 0};
    real u = 0;
    auto fetch = [&](int c) {
        const int e = c * kWave + lane, ee = e < N ? e : N - 1;
        s = Xo[ee];
        u = Uo[ee];
        if (!a.sa) {
            xn[0] = X0[ee];
            xn[1] = X1[ee];
        }
    };
    fetch(0);
    for (int c = 0; c < nChunks; ++c) {
        const int e = c * kWave + lane;
        const uint32_t si = s, xi[2] = {xn[0], xn[1]};
        const real ui = u;
        if (c + 1 < nChunks)
            fetch(c + 1); /* in flight while this chunk is prepared */
        real t = ui;
        if constexpr (sizeof(real) == 4)
            t = sq_exp_above(ui, expTab);
        uint32_t code = 0;
        if (c >= kRing / kWave) /* the entries this chunk replaces have been read */
            while (ctlLoad(ctl + kCtlPos) < (uint32_t)(c - (kRing / kWave - 1)) * kWave)
                __builtin_amdgcn_s_sleep(2);
        if (!a.sa) {
            /* table[nb][site]: the neighbour's last and second to last attempt
             * there, each as index + 1 (0: none), last << 16 | second.  Where
             * several of the chunk's attempts share a slot, both become the
             * chunk's end, i.e. are taken for undecided longer than needed; in
             * a small table, where that is no exception, a mask of the chunk's
             * attempts by slot tells the last two that precede. */
            const uint32_t before = (uint32_t)c * kWave, end = before + kWave;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                uint32_t *const own = table + b * tableN + (si & mask), *const his = table + b * tableN + (xi[b] & mask);
                const uint32_t o = ldsLoad(own), h = ldsLoad(his);
                const uint32_t bound = (uint32_t)(e + nb.delta[b]); /* index + 1 of the last that precedes */
                uint32_t p1, p2;
                if (N <= kExactTable) {
                    unsigned long long *const hisM = masks + (xi[b] & mask), *const ownM = masks + (si & mask);
                    if (e < N)
                        atomicOr(hisM, 1ull << lane);
                    waveSync();
                    /* the last two of: the chunk's attempts in m, then old */
                    auto lastTwo = [&](unsigned long long m, uint32_t old, uint32_t &l1, uint32_t &l2) {
                        const int j1 = 63 - __builtin_clzll(m | 1ull);
                        const unsigned long long m2 = m & ~(1ull << j1);
                        const int j2 = 63 - __builtin_clzll(m2 | 1ull);
                        l1 = m ? before + (uint32_t)j1 + 1u : old >> 16;
                        l2 = !m ? old & 0xffffu : m2 ? before + (uint32_t)j2 + 1u : old >> 16;
                    };
                    const unsigned long long mh = *hisM;
                    const int n = (int)(bound - before); /* 0 .. 64 of the chunk's attempts precede */
                    const unsigned long long mo = n >= kWave ? *ownM : *ownM & ((1ull << n) - 1ull);
                    uint32_t q1, q2;
                    lastTwo(mo, o, p1, p2);
                    lastTwo(mh, h, q1, q2);
                    waveSync();
                    if (e < N) {
                        *hisM = 0ull;
                        ldsStore(his, q1 << 16 | q2); /* the same from all that share the slot */
                    }
                    waveSync();
                } else {
                    const uint32_t mine = (uint32_t)(e + 1) << 16 | h >> 16;
                    if (e < N)
                        ldsStore(his, mine);
                    const uint32_t w = ldsLoad(his);
                    if (e < N && w != mine)
                        ldsStore(his, end << 16 | end);
                    const uint32_t v = ldsLoad(own);
                    p1 = v >> 16;
                    p2 = v & 0xffffu;
                    if (p1 > before) {
                        if (p2 > before) {
                            p1 = p2 = bound;
                        } else if (p1 > bound) {
                            p1 = o >> 16;
                            p2 = o & 0xffffu;
                        }
                    }
                }
                const uint32_t d1 = p1 ? bound - p1 + 1u : 0u, d2 = p2 ? bound - p2 + 1u : 0u;
                code |= (d1 <= (uint32_t)kMaxBack ? d1 : 0u) << (16 * b) |
                        (d2 <= (uint32_t)kMaxBack ? d2 : 0u) << (16 * b + 8);
                nbSites[b * kNbRing + (e & (kNbRing - 1))] = (uint16_t)xi[b];
            }
        }
        const int slot = e & (kRing - 1);
        ringS[slot] = si;
        ringT[slot] = t;
        ringC[slot] = code;
        ldsWait();
        ctlStore(ctl + kCtlReady, (uint32_t)(c + 1));
    }
}

/* The watcher of slice y.  ownAt0, 1: the byte offset from `lds` of a neighbour's
 * words when its slice is in this workgroup, else -1.  Lanes 0-31 look at
 * neighbour 0's window, lanes 32-63 at neighbour 1's. */
template <class real>
__device__ __forceinline__ void watcherLoop(const SweepArgs<real> &a, int y, unsigned char *lds, unsigned char *region,
                            const TeamRegion &r, int ownAt0, int ownAt1) {
    const int lane = threadIdx.x & (kWave - 1), half = lane >> 5, word = lane & (kWinWords - 1);
    const Neighbours nb = neighboursOf(y, a.m);
    uint16_t *const list = reinterpret_cast<uint16_t *>(region + r.flips) + half * kFlipRing;
    uint32_t *const ctl = reinterpret_cast<uint32_t *>(region + r.ctl);
    const uint32_t tag = teamTag(a.tag);
    const uint32_t *const P = a.P + (long long)(half ? nb.n[1] : nb.n[0]) * a.ldP + word;
    const int own = half ? ownAt1 : ownAt0;
    int seen = 0;        /* of the lane's half: decided attempts already listed */
    uint32_t nFlips = 0; /* and flips listed */
    for (;;) {
        if (ctlLoad(ctl + kCtlPos) == kEnd)
            return;
        const int ready = (int)ctlLoad(ctl + kCtlReady) * kWave; /* sites known up to there */
        const int first = seen / kPerWord;
        uint32_t w;
        if (own >= 0)
            w = ldsLoad(reinterpret_cast<const uint32_t *>(lds + own) + first + word);
        else
            w = loadShared32(P + first);
        const int cnt = decidedIn(w, tag);
        const uint32_t partial = (uint32_t)(__ballot(cnt < kPerWord) >> (32 * half));
        const int j = partial ? __builtin_ctz(partial) : kWinWords;
        const int more = __shfl(cnt, 32 * half + (j & (kWinWords - 1)));
        int upTo = (first + j) * kPerWord + (partial ? more : 0);
        upTo = upTo < ready ? upTo : ready;
        const bool moved = upTo > seen;
        if (!__ballot(moved))
            continue;
        /* the flips among [seen, upTo), in order */
        const int e0 = (first + word) * kPerWord;
        int lo = seen - e0, hi = upTo - e0;
        lo = lo < 0 ? 0 : lo > kPerWord ? kPerWord : lo;
        hi = hi < 0 ? 0 : hi > kPerWord ? kPerWord : hi;
        uint32_t flips = hi > lo ? w & ((1u << hi) - 1u) & ~((1u << lo) - 1u) : 0u;
        for (;;) {
            const unsigned long long any = __ballot(flips != 0u);
            if (!any)
                break;
            const uint32_t mine = (uint32_t)(any >> (32 * half));
            if (mine && word == __builtin_ctz(mine)) { /* one flip of each half */
                list[nFlips & (kFlipRing - 1)] = (uint16_t)(e0 + __builtin_ctz(flips));
                flips &= flips - 1u;
            }
            nFlips += mine ? 1u : 0u;
        }
        seen = moved ? upTo : seen;
        /* the list before its length before the position it reaches to */
        if (word == 0) {
            ldsStore(ctl + kCtlFlips + half, nFlips);
            ldsStore(ctl + kCtlDecided + half, (uint32_t)seen);
        }
    }
}

/* A wave-uniform value kept in a vector register: the sweeper has many and the
 * scalar registers are few. */
template <class T>
__device__ __forceinline__ T inVector(T v) {
    asm volatile("" : "+v"(v));
    return v;
}

/* A pointer to device memory that was itself loaded, for which the compiler would
 * not know. */
template <class T>
__device__ __forceinline__ T *inGlobal(T *p) {
    return (T *)(__attribute__((address_space(1))) T *)p;
}

/* The sweeper of slice y. */
template <class real>
__device__ __forceinline__ void sweeperLoop(const SweepArgs<real> &a, const int y, const uint64_t *expTab, const real *hS,
                            unsigned char *region, const TeamRegion &r) {
#pragma clang fp contract(off)
    const int N = a.N, Np = a.Np, m = a.m, Nw = a.Nw;
    const int lane = threadIdx.x & (kWave - 1);
    const int half = lane >> 5; /* the neighbour whose flips this lane mirrors */
    real *const F = reinterpret_cast<real *>(region + r.F);
    uint32_t *const Qb = reinterpret_cast<uint32_t *>(region + r.bits);
    uint32_t *const mirror = Qb + Nw; /* [2][Nw] */
    const uint16_t *const list = reinterpret_cast<const uint16_t *>(region + r.flips) + half * kFlipRing;
    const uint16_t *const nbSites = reinterpret_cast<const uint16_t *>(region + r.nbSites) + half * kNbRing;
    const uint32_t *const ringS = reinterpret_cast<const uint32_t *>(region + r.ringS);
    const real *const ringT = reinterpret_cast<const real *>(region + r.ringT);
    const uint32_t *const ringC = reinterpret_cast<const uint32_t *>(region + r.ringC);
    uint32_t *const own = reinterpret_cast<uint32_t *>(region + r.own);
    uint32_t *const ctl = reinterpret_cast<uint32_t *>(region + r.ctl);
    const real *const stage = reinterpret_cast<const real *>(region + r.stage);
    const uint32_t stageL = ldsAddress(stage);
    const uint32_t rowBytes = (uint32_t)Np * (uint32_t)sizeof(real);
    const uint32_t tag = teamTag(a.tag);
    const Neighbours nb = neighboursOf(y, m);
    uint32_t *const P = a.P + (long long)y * a.ldP;
    const real twoDivM = inVector(a.twoDivM), coef = inVector(a.coef), perDE = inVector(a.sa ? a.invKT : a.beta);
    int k = 0, ready = 0;
    int R[2] = {0, 0};  /* the mirror holds the neighbour's attempts before R */
    uint32_t mirrored = 0; /* of the lane's half: flips in the mirror */
    uint32_t open = 0;  /* flips of the published word that is not full */
    uint32_t nFlips = 0, nBatches = 0, nBlocked = 0;
    int spins = 0;
    bool aborted = false;
    /* the last flip's row: until a batch after it commits, the batches add its
     * elements themselves; then the rows wave adds it to F */
    bool rowPending = false;
    uint32_t rows = 0, added = 0; /* handed over, known to be in F */
    real rowD = 0;

    while (k < N) {
        const int need = divru(k + kWave < N ? k + kWave : N, kWave);
        while (ready < need)
            ready = (int)ctlLoad(ctl + kCtlReady);
        /* lanes past the last attempt: their slots may never have been written */
        const uint32_t s = k + lane < N ? ringS[(k + lane) & (kRing - 1)] : 0u;
        const real t = ringT[(k + lane) & (kRing - 1)];
        const uint32_t code = ringC[(k + lane) & (kRing - 1)];
        const uint32_t qw = Qb[s >> 5];
        const real hx = hS[s];
        int limit = uni(N - k);

        /* neighbours: how far each is decided, its flips into the mirror */
        bool pend0 = false, pend1 = false, several = false;
        if (!a.sa) {
            /* the decided positions first, then the flips listed: at least up to them */
            const uint32_t decided = ldsLoad(ctl + kCtlDecided + half), listed = ldsLoad(ctl + kCtlFlips + half);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int A = __builtin_amdgcn_readlane((int)decided, 32 * b), Kk = k + nb.delta[b];
                const int upTo = A < Kk ? A : Kk;
                R[b] = uni(upTo > R[b] ? upTo : R[b]);
                const int lim = kMaxBack + 1 - (Kk - R[b]);
                limit = uni(lim < limit ? lim : limit);
            }
            if (__ballot(listed != mirrored)) {
                const uint32_t before = (uint32_t)(half ? R[1] : R[0]);
                for (;;) { /* 32 of each neighbour's at a time, in order */
                    const uint32_t at = mirrored + (uint32_t)(lane & 31);
                    const uint32_t e = list[at & (kFlipRing - 1)];
                    const bool mine = (int)(listed - at) > 0 && e < before;
                    if (mine) {
                        const uint32_t x = nbSites[e & (kNbRing - 1)];
                        atomicXor(&mirror[half * Nw + (x >> 5)], 1u << (x & 31u));
                    }
                    const unsigned long long done = __ballot(mine);
                    const uint32_t n = (uint32_t)__popc((uint32_t)(done >> (32 * half)));
                    mirrored += n;
                    if (!__ballot(n == 32u))
                        break;
                }
            }
            /* attempts on the lane's site in [R, its position): distance <= back */
            const uint32_t back0 = (uint32_t)(lane + k + nb.delta[0] - R[0]);
            const uint32_t back1 = (uint32_t)(lane + k + nb.delta[1] - R[1]);
            pend0 = (code & 255u) - 1u < back0;
            pend1 = ((code >> 16) & 255u) - 1u < back1;
            several = (pend0 && pend1) || ((code >> 8) & 255u) - 1u < back0 || (code >> 24) - 1u < back1;
            waveSync();
        }

        /* evaluate attempt k + lane speculatively */
        const bool valid = lane < limit;
        const bool qpos = (qw >> (s & 31)) & 1u;
        const real q = qpos ? (real)1 : (real)-1;
        real nsum = 0, nsumAlt = 0;
        if (!a.sa) {
            const real nv0 = ((mirror[s >> 5] >> (s & 31)) & 1u) ? (real)1 : (real)-1;
            const real nv1 = ((mirror[Nw + (s >> 5)] >> (s & 31)) & 1u) ? (real)1 : (real)-1;
            nsum = nv0 + nv1;
            nsumAlt = pend0 ? -nv0 + nv1 : nv0 - nv1;
        }
        while (added != rows)
            added = ctlLoad(ctl + kCtlDone);
        real f = F[s];
        if (rowPending) {
            vmWaitImm<0>();
            f = addScaled(f, rowD, stage[(size_t)(rows & 1u) * Np + s]);
        }
        auto decideWith = [&](real ns) {
            /* the reference's operation order; accepted when the threshold, 1
             * for dE < 0 and exp(x) otherwise, exceeds the uniform */
            real dE;
            if (!a.sa) {
                /* CPUDenseGraphAnnealer.cpp:258-262 */
                dE = twoDivM * q * (hx + (real)2. * f);
                dE -= q * ns * coef;
            } else {
                /* :348-349 */
                dE = (real)2. * q * (hx + (real)2. * f);
            }
            const real x = -dE * perDE;
            if constexpr (sizeof(real) == 4) {
                /* t: the least accepted x, NaN (never accepted) for a uniform of 1 */
                return dE < (real)0. ? t == t : x >= t;
            } else {
                const real e = Expo<real>::eval(x, expTab);
                return (dE < (real)0. ? (real)1. : e) > t;
            }
        };
        const bool acc = decideWith(nsum);
        bool blocked = several;
        if (__ballot(pend0 || pend1))
            blocked = blocked || ((pend0 || pend1) && decideWith(nsumAlt) != acc);
        const int firstStop = uni(__builtin_ffsll((long long)__ballot(!valid || blocked)) - 1);
        const int firstAcc = uni(__builtin_ffsll((long long)__ballot(valid && !blocked && acc)) - 1);
        const int stop = firstStop < 0 ? kWave : firstStop;
        const bool flip = firstAcc >= 0 && firstAcc < stop;
        const int c = flip ? firstAcc + 1 : stop;

        if (c == 0) {
            /* attempt k waits for a neighbour's serially earlier attempt: the
             * last on its site or, beyond kMaxBack, the first undecided one */
            ++nBlocked;
            const uint32_t code0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)code);
            int waitNb = -1, waitE = 0;
#pragma unroll
            for (int b = 1; b >= 0; --b) {
                const int Kk = k + nb.delta[b], back = Kk - R[b];
                const int d = (int)((code0 >> (16 * b)) & 255u);
                if (back > kMaxBack) {
                    waitNb = b;
                    waitE = R[b];
                } else if (d != 0 && d <= back) {
                    waitNb = b;
                    waitE = Kk - d;
                }
            }
            if (waitNb >= 0) {
                while ((int)ctlLoad(ctl + kCtlDecided + waitNb) <= waitE) {
                    if (++spins > a.spinLimit)
                        break;
                    if (spins < 256)
                        __builtin_amdgcn_s_sleep(1);
                    else
                        __builtin_amdgcn_s_sleep(16);
                }
            }
            if (++spins > a.spinLimit) {
                atomicExch(a.abortFlag, 1);
                if (a.abortHost) /* a vector store, system scope: the host reads it after the step */
                    __hip_atomic_store(a.abortHost, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                aborted = true;
                break;
            }
            if ((spins & 63) == 0 && __hip_atomic_load(a.abortFlag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                aborted = true;
                break;
            }
            waveSync();
            continue;
        }
        spins = 0;
        ++nBatches;

        /* publish the committed decisions: the words of attempts k .. k+c-1 */
        {
            const int g0 = k / kPerWord, g1 = (k + c - 1) / kPerWord;
            const int at = k + c - 1; /* the flip, if there is one */
            const uint32_t bit = flip ? 1u << (at % kPerWord) : 0u;
            const int g = g0 + lane;
            const int n = k + c - g * kPerWord;
            uint32_t flips = lane == 0 ? open : 0u;
            flips |= g == g1 ? bit : 0u;
            if (!a.sa && g <= g1) { /* lane 0 always: one op */
                const uint32_t w = packWord(tag, n < kPerWord ? n : kPerWord, flips);
                storeShared32(P + g, w);
                if (r.ctl != r.own)
                    ldsStore(own + g, w);
            }
            open = (g1 == g0 ? open : 0u) | bit;
            if ((k + c) % kPerWord == 0)
                open = 0u;
        }

        if (rowPending) { /* it has landed, and this batch's fields have been read */
            ctlStore(ctl + kCtlSign + (rows & 1u), rowD < (real)0. ? 1u : 0u);
            ctlStore(ctl + kCtlRows, ++rows);
            rowPending = false;
        }
        if (flip) {
            ++nFlips;
            const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)s, firstAcc);
            const bool qx = (__ballot(qpos) >> firstAcc) & 1ull;
            /* F[y][:] += -2 q_x J[x][:] (J symmetric): the row streams into the
             * other buffer than the one the rows wave may be reading (the one
             * before that is in F: this batch's fields waited for it) */
            dmaRunx4(reinterpret_cast<const unsigned char *>(a.J + (long long)x * Np), stageL + (rows & 1u) * rowBytes,
                     (int)(rowBytes / (kWave * 16)));
            rowD = qx ? (real)-2. : (real)2.;
            if (lane == firstAcc)
                atomicXor(&Qb[x >> 5], 1u << (x & 31));
            rowPending = true;
        }
        k = uni(k + c);
        ctlStore(ctl + kCtlPos, (uint32_t)k);
        waveSync();
    }

    /* nothing may land in this region after the wave leaves it */
    vmWaitImm<0>();
    ctlStore(ctl + kCtlPos, kEnd); /* the watcher ends; an aborted sweep's scout runs out */
    if (rowPending) { /* landed by now */
        ctlStore(ctl + kCtlSign + (rows & 1u), rowD < (real)0. ? 1u : 0u);
        ctlStore(ctl + kCtlRows, ++rows);
    }
    while (ctlLoad(ctl + kCtlDone) != rows)
        ;
    ctlStore(ctl + kCtlRows, kEnd);
    /* the arguments, read anew: kept from the start, they would take scalar
     * registers from the loop (double then spills some: 33.2 us a sweep against
     * 32.7 at N=500, m=125) */
    const auto *e = (const __attribute__((address_space(4))) SweepArgs<real> *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(e));
    uint32_t *const Qout = inGlobal(e->Qout) + (long long)y * Nw;
    if (!aborted) {
        real *const Fout = inGlobal(e->F) + (long long)y * Np;
#pragma unroll 4
        for (int b = 0; b < Np; b += kWave * 4) {
            real v[4];
            ldsLoad4(F + b + lane * 4, v);
            ldsStore4(Fout + b + lane * 4, v); /* a plain vector store, here to global */
        }
        for (int b = 0; b < Nw; b += kWave)
            if (b + lane < Nw)
                Qout[b + lane] = Qb[b + lane];
    } else { /* the slice keeps its spins */
        const uint32_t *const Qin = inGlobal(e->Qbits) + (long long)y * Nw;
        for (int b = lane; b < Nw; b += kWave)
            Qout[b] = Qin[b];
    }
    unsigned long long *const counters = inGlobal(e->counters);
    if (lane == 0 && counters) {
        atomicAdd(&counters[0], (unsigned long long)nFlips);
        atomicAdd(&counters[1], (unsigned long long)nBatches);
        atomicAdd(&counters[2], (unsigned long long)nBlocked);
    }
}

template <class real>
__global__ __launch_bounds__(kTeamWaves *kTeamMaxSlices *kWave) void denseSweepTeamKernel(SweepArgs<real> a, int S,
                                                                                         int xcdRemap, int tableN) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int wave = uni(threadIdx.x / kWave), lane = threadIdx.x & (kWave - 1);
    /* consecutive slices on the same XCD (blocks are dispatched round-robin
     * over the 8 XCDs) */
    int b = blockIdx.x;
    if (xcdRemap)
        b = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    const int role = wave / S, i = wave % S; /* the sweepers first: a SIMD each */
    const int y = b * S + i;
    const TeamRegion r = teamRegion<real>(a.N, a.Np, tableN, S);
    uint64_t *const expTab = reinterpret_cast<uint64_t *>(lds);
    real *const hS = reinterpret_cast<real *>(lds + kExpTabBytes);
    unsigned char *const regions = lds + kExpTabBytes + (size_t)a.Np * sizeof(real);
    unsigned char *const region = regions + (size_t)r.bytes * i;
    uint32_t *const ctl = reinterpret_cast<uint32_t *>(region + r.ctl);
    const bool live = y < a.m;

    /* start-up state: h and the fields by DMA, spin bits and mirrors */
    if (threadIdx.x < 32)
        expTab[threadIdx.x] = sq_exp2_tab32[threadIdx.x];
    const int rowBytes = a.Np * (int)sizeof(real);
    {
        const unsigned char *src = reinterpret_cast<const unsigned char *>(a.h);
        const uint32_t hL = ldsAddress(hS);
        for (int j0 = wave * kWave * 16; j0 < rowBytes; j0 += kTeamWaves * S * kWave * 16)
            dmaDwordx4(src + j0 + lane * 16, hL + j0);
    }
    if (live && role == 0) {
        const unsigned char *src = reinterpret_cast<const unsigned char *>(a.F + (long long)y * a.Np);
        const uint32_t FL = ldsAddress(region + r.F);
        for (int j0 = 0; j0 < rowBytes; j0 += kWave * 16)
            dmaDwordx4(src + j0 + lane * 16, FL + j0);
        if (lane < kCtlWords)
            ctl[lane] = 0;
    } else if (live && role == 1) {
        const Neighbours nb = neighboursOf(y, a.m);
        const uint32_t QbL = ldsAddress(region + r.bits);
        const int Nw = a.Nw;
        for (int w = 0; w < Nw; w += kWave) {
            dmaEntries<4, false, kWave>(a.Qbits + (long long)y * Nw + w, QbL + w * 4, w, Nw);
            dmaEntries<4, false, kWave>(a.Qbits + (long long)nb.n[0] * Nw + w, QbL + (Nw + w) * 4, w, Nw);
            dmaEntries<4, false, kWave>(a.Qbits + (long long)nb.n[1] * Nw + w, QbL + (2 * Nw + w) * 4, w, Nw);
        }
    } else if (live && role == 2) {
        uint4 *const table = reinterpret_cast<uint4 *>(region + r.table);
        for (int j = lane; j < (r.nbSites - r.table) / 16; j += kWave) /* and the masks */
            table[j] = uint4{0u, 0u, 0u, 0u};
    } else if (live) {
        uint32_t *const own = reinterpret_cast<uint32_t *>(region + r.own);
        for (int j = lane; j < (r.ctl - r.own) / 4; j += kWave)
            own[j] = 0u;
    }
    vmWaitImm<0>();
    __syncthreads();
    if (!live)
        return;
    if (role == 1) {
        rowsLoop<real>(a.Np, region, r);
    } else if (role == 2) {
        scoutLoop<real>(a, y, expTab, region, r, tableN);
    } else if (role == 3) {
        if (a.sa)
            return;
        const Neighbours nb = neighboursOf(y, a.m);
        /* (with S = 1 no neighbour is in the block: denseSweepTeam's m > 1) */
        auto ownAt = [&](int n) { return n / S == b ? (int)(regions - lds) + r.bytes * (n - b * S) + r.own : -1; };
        watcherLoop<real>(a, y, lds, region, r, ownAt(nb.n[0]), ownAt(nb.n[1]));
    } else {
        sweeperLoop<real>(a, y, expTab, hS, region, r);
    }
}

}  // namespace

int teamWordStride(int N) { return roundUp(divru(N, kPerWord) + kWinWords, kWave); }

static size_t teamLdsBytes(int N, int Np, int tableN, int S, size_t realSize) {
    const size_t region = realSize == 8 ? teamRegion<double>(N, Np, tableN, S).bytes : teamRegion<float>(N, Np, tableN, S).bytes;
    return kExpTabBytes + (size_t)Np * realSize + region * S;
}

/* Slots of the tables by site for S slices a block, 0 where it does not fit.
 * Fewer slots than sites only for one slice, where LDS demands it: with hashed
 * tables many lanes wait for attempts on other sites (N=4096, m=256, two slices
 * a block on 1024 slots: 175 us a sweep against 110 us for one slice on 4096). */
static int teamTable(int N, int Np, int S, size_t realSize, size_t maxLds) {
    for (int t = siteTableSize(N);; t >>= 1) {
        if (N < 65000 && teamLdsBytes(N, Np, t, S, realSize) <= maxLds)
            return t;
        if (S > 1 || N <= kExactTable || t <= kMinHashed)
            return 0;
    }
}

int denseSweepTeamSlices(int N, int Np, int m, size_t realSize, int asked, int numCUs, size_t maxLds) {
    if (asked > 0) {
        const int tableN = asked <= kTeamMaxSlices ? teamTable(N, Np, asked, realSize, maxLds) : 0;
        if (tableN == 0)
            return 0;
        /* a team takes more LDS than one wave: 256 of them at N=4096 where 512
         * slices of the one-wave sweep fit */
        const int nBlocks = divru(m, asked);
        const void *fn = realSize == 8 ? (const void *)denseSweepTeamKernel<double> : (const void *)denseSweepTeamKernel<float>;
        const size_t lds = teamLdsBytes(N, Np, tableN, asked, realSize);
        return nBlocks <= numCUs || fitsAtOnce(fn, kTeamWaves * asked * kWave, lds, nBlocks, numCUs) ? asked : 0;
    }
    /* as many slices as LDS holds: they read each other's decisions there, in a
     * quarter of the time it takes over device memory (N=1200, m=300: 53.6 us a
     * sweep with three, 55.0 with two, 56.3 with one on twice the blocks there
     * are CUs for) */
    int S = m < kTeamMaxSlices ? m : kTeamMaxSlices;
    while (S > 1 && !teamTable(N, Np, S, realSize, maxLds))
        --S;
    return teamTable(N, Np, S, realSize, maxLds) && divru(m, S) <= numCUs ? S : 0;
}

template <class real>
void denseSweepTeam(const SweepArgs<real> &args, int slicesPerBlock, size_t maxLds, bool allowDirect, int numCUs,
                    hipStream_t stream) {
    SQ_THROW_IF(args.Np % 256 != 0 || args.Nw * 32 != args.Np || args.N > args.Np || args.N >= 65000,
                "team sweep: bad row of %d sites in %d", args.N, args.Np);
    SQ_THROW_IF(slicesPerBlock < 1 || slicesPerBlock > kTeamMaxSlices, "slices per block out of range (1..%d)",
                kTeamMaxSlices);
    SQ_THROW_IF(args.m == 1 && !args.sa, "team sweep: a slice that is its own neighbour");
    SQ_THROW_IF(!args.Qout || args.Qout == args.Qbits, "the sweep needs a second spin buffer");
    SQ_THROW_IF(!args.P || args.ldP < teamWordStride(args.N), "team sweep: no decision words");
    const int nBlocks = divru(args.m, slicesPerBlock);
    int xcdRemap = (nBlocks % 8 == 0 && nBlocks >= 16) ? 1 : 0;
    int tableN = teamTable(args.N, args.Np, slicesPerBlock, sizeof(real), maxLds);
    SQ_THROW_IF(tableN == 0, "team sweep: N=%d does not fit in LDS", args.N);
    SweepArgs<real> a = args;
    void *kargs[] = {(void *)&a, (void *)&slicesPerBlock, (void *)&xcdRemap, (void *)&tableN};
    launchSweep((void *)denseSweepTeamKernel<real>, nBlocks, kTeamWaves * slicesPerBlock * kWave,
                teamLdsBytes(args.N, args.Np, tableN, slicesPerBlock, sizeof(real)), kargs, allowDirect, numCUs,
                stream);
}

template void denseSweepTeam<float>(const SweepArgs<float> &, int, size_t, bool, int, hipStream_t);
template void denseSweepTeam<double>(const SweepArgs<double> &, int, size_t, bool, int, hipStream_t);

}  // namespace sqaod_rocm
