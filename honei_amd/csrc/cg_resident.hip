// cg_resident.hip -- CG and Jacobi-preconditioned CG iterations that stay on
// the chip: one launch runs thousands of iterations.
//
// An iteration enqueued launch by launch costs three (up to 65,536 rows) or
// five kernels of 4-8 us and the gaps between them, whatever the system's
// size; the work itself (a few hundred KB to a few tens of MB out of L2 /
// MALL) is far less.  Here every thread keeps its rows' matrix entries,
// column offsets and the direction's values at those columns in registers,
// with x, r and the own direction value beside them; the only data that
// cross work-groups are the residual (CG) or z = dinv .* r (PCG), published
// once per iteration and gathered at the row's columns (the direction there
// is then updated in registers: the same expression of the same operands as
// its owner forms), and the partial sums of the two reductions.
//
// Work-groups meet at each reduction: each posts its partials, one word a
// sum, and reads everyone's until no word is empty, so a reduction and the
// barrier are one exchange; the published vector is gathered while the second
// one is under way, each value read again until it is there.  All data exchanged inside the launch are
// agent-scope accesses.
//
// What bounds it: the two exchanges (a store and a load through memory, about
// 1.7 us each across XCDs) and, above some 100,000 rows, the gather's
// requests.  FP64, 9 entries per row, per iteration, CG / PCG-Jacobi, against
// the launches: 65^2 rows 4.2 / 4.7 us (15.6 / 16.9), 129^2 4.8 / 5.3 (17.3 /
// 18.6), 361^2 5.9 / 6.1 (22.9 / 23.9), 513^2 11.5 / 12.1 (26.6 / 28.0), 720^2
// 14.2 / 14.9 (35.6 / 37.6).
//
// Bits: the sums are those of the launch-by-launch kernels, term for term
// (k_cg_spmv_dot's partial per 256 rows, the update's per-thread chain over
// its grid-stride elements and block_sum, sum_partials' tree), so x, the
// iteration count and the defect do not depend on the path.
//
// Waits are bounded: a work-group that sees no progress for too long sets
// sc->aborted and leaves, the others follow; x is written to scratch and
// copied to the caller's vector only when no work-group did, so the caller can
// run the launches instead.  A lease bounds the work-groups of all such
// launches of a process on a device by its compute units, so its own solves
// cannot keep each other out.  Other processes' can: each then holds part of
// the chip and waits for the rest of its own.  So the first exchange of a
// launch, after which every work-group is known to be on the chip, waits
// kArriveTicks only.  Four processes with twelve solves each on 522,729 rows
// (5.5 ms a solve alone): 0.3 to 0.4 s, launches only 0.4 to 0.5; the long wait there
// too: 5.4 s.

#include <atomic>

#include "solvers.hh"

#include "ell_device.hh"
#include "solver_device.hh"

#pragma clang fp contract(off)

namespace honei {
namespace hipx {
namespace {

constexpr int kThreads = 512, kWaves = kThreads / kWave;
constexpr int kChunk = 256;            // rows per SpMV partial
constexpr int kGroupChunks = 8;        // chunks of one update partial (2048 rows)
constexpr int kWidth = 9;              // stored entries per row at most
constexpr int64_t kMaxChunks = 2048;   // partials two rounds of 1024 threads sum
constexpr int64_t kFourRows = 65536, kTwoRows = 262144;   // four / two work-groups per group up to here
// wall_clock64 ticks (100 MHz): 2 ms for the work-groups of a launch to arrive
// (some 50 us where nothing is in their way), 1 s for any other wait
constexpr uint64_t kArriveTicks = 200000ull, kWaitTicks = 100000000ull;

// What crosses work-groups is empty (a signalling NaN, which no addition or
// product returns; results that are NaN travel as quiet ones) until its owner
// posts it, so a reader needs no other sign that it is there.  Words of sums
// and published vectors have two sets each, used by even and odd iterations;
// an owner empties the set of the next iteration when it knows that everyone
// has read it, and before its own next post that others wait for.
constexpr uint64_t kEmpty = 0x7ff0000000000001ull;
template <typename V> struct EmptyOf;
template <> struct EmptyOf<double> {
    typedef uint64_t Bits;
    static constexpr Bits value = kEmpty;
};
template <> struct EmptyOf<float> {
    typedef uint32_t Bits;
    static constexpr Bits value = 0x7f800001u;
};
constexpr int64_t kWordsA = 4 * kMaxChunks, kWordsB = 2 * 4 * (kMaxChunks / kGroupChunks);
constexpr int64_t kWords = 2 * (kWordsA + kWordsB);

template <typename T> __device__ inline T agent_load(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T> __device__ inline void agent_store(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The value where it is used: keeps what is derived from it (64-bit addresses,
// lane masks: two registers each) from being formed once before the loop.
template <typename T> __device__ inline T here(T v) {
    asm volatile("" : "+v"(v));
    return v;
}
template <typename V> __device__ inline typename EmptyOf<V>::Bits agent_load_bits(const V *base, uint32_t byte_off) {
    return agent_load((const typename EmptyOf<V>::Bits *)((const char *)base + byte_off));
}
template <typename V>
__device__ inline void agent_store_bits(V *base, uint32_t byte_off, typename EmptyOf<V>::Bits v) {
    agent_store((typename EmptyOf<V>::Bits *)((char *)base + byte_off), v);
}

__device__ inline void post(uint64_t *w, double v) { agent_store(w, __builtin_bit_cast(uint64_t, v)); }

// t0: 0 at the first call of a wait
__device__ inline bool in_time(uint64_t &t0, uint64_t ticks) {
    const uint64_t now = wall_clock64();
    if (t0 == 0) t0 = now;
    return now - t0 <= ticks;
}

// The N words w[0], w[step], ... once all are posted; false when the wait
// runs out.  Neighbouring lanes read neighbouring words: a poll of a
// wavefront is N requests of 512 bytes.
template <int N>
__device__ inline bool take(const uint64_t *w, int step, double (&v)[N], uint64_t ticks) {
    uint64_t t0 = 0, q[N];
    for (uint32_t spin = 0;; ++spin) {
        bool all = true;
#pragma unroll
        for (int i = 0; i < N; ++i) q[i] = agent_load(w + i * step);
#pragma unroll
        for (int i = 0; i < N; ++i) all = all && q[i] != kEmpty;
        if (all) break;
        if ((spin & 255u) == 255u && !in_time(t0, ticks)) return false;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = __builtin_bit_cast(double, q[i]);
    return true;
}

// block_sum's combination of a 256-thread work-group's wave sums from the
// words posted for it: one (the sum), two (waves 0 + 2, 1 + 3), four
__device__ inline double combine(const double (&w)[1]) { return w[0]; }
__device__ inline double combine(const double (&w)[2]) { return w[0] + w[1]; }
__device__ inline double combine(const double (&w)[4]) { return (w[0] + w[2]) + (w[1] + w[3]); }

__device__ inline double first_lane(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// block_sum's second stage over up to 16 wave sums, in every thread
__device__ inline double tree16(const double *red, int lane) {
    return first_lane(wave_sum(lane < 16 ? red[lane] : 0.0));
}

template <typename VT> __device__ inline typename VecOf<VT>::type stored(const VT *Ax, int64_t s) {
    if constexpr (sizeof(VT) == 2)
        return bf16_to_float(Ax[s].bits);
    else
        return Ax[s];
}

// Group b (2048 rows): chunks b + k g2, k < 8 -- the rows whose squares one
// update partial sums (thread t of it: row t of each chunk, in order of k).
// Q = 4 / R work-groups share a group, R rows per thread: work-group h of
// them serves the 64-row quarters h, h + Q, .. of every chunk.  Few rows per
// thread put small systems on more CUs, each with fewer gathers to wait for;
// many keep the words of a sum few.  Wave w serves (chunk, quarter) pairs
// w + 8 j.
template <typename VT, bool PCG, int R>
__global__ __launch_bounds__(kThreads) void k_cg_resident(EllView A, const typename VecOf<VT>::type *dinv,
                                                          const typename VecOf<VT>::type *xin,
                                                          typename VecOf<VT>::type *xs, typename VecOf<VT>::type *pv,
                                                          typename VecOf<VT>::type *rv,
                                                          typename VecOf<VT>::type *pub0,
                                                          typename VecOf<VT>::type *pub1, CGScalars *sc,
                                                          uint64_t *words, int nchunks, int g2, int it_begin,
                                                          int it_end, uint64_t arrive) {
    typedef typename VecOf<VT>::type V;
    typedef typename EmptyOf<V>::Bits Bits;
    constexpr int Q = 4 / R, NRED = PCG ? 2 : 1;
    // gather while the sum is under way (the values wanted: 18 registers a row)
    constexpr bool kEarly = R <= 2;
    __shared__ double red_a[16], red_b[NRED][16], sq[NRED][kGroupChunks][64 * R], wsum[kGroupChunks][R],
        bsum[NRED][R];
    __shared__ int bad;
    // another work-group may set aborted meanwhile: read it once
    if (sc->done || block_uniform_flag(&sc->aborted)) return;
    const int tid = threadIdx.x, lane = tid % kWave, w = tid / kWave;
    const int b = blockIdx.x / Q, h = blockIdx.x % Q;
    const VT *Ax = (const VT *)A.Ax;
    const V e = eps_of<V>();

    // x, r and dinv of the own rows: touched once per iteration, in LDS (a
    // thread's own words) so that four rows' entries fit the registers
    __shared__ V xl[R][kThreads], rl[R][kThreads], dl[PCG ? R : 1][kThreads];
    V a[R][kWidth], pc[R][kWidth], po[R];
    uint32_t off[R][kWidth], own[R];
    int len[R];
#pragma unroll
    for (int j = 0; j < R; ++j) {
        const int pr = w + kWaves * j, k = pr / R, quarter = h + Q * (pr % R);
        const int64_t c = b + (int64_t)k * g2, row = c * kChunk + quarter * kWave + lane;
        const bool live = c < nchunks && row < A.rows;
        const int64_t rr = live ? row : 0;
        len[j] = live ? (int)A.Arl[rr] : -1;
        own[j] = (uint32_t)rr * (uint32_t)sizeof(V);
#pragma unroll
        for (int t = 0; t < kWidth; ++t) {
            const bool in = t < len[j];
            const int64_t s = rr + (int64_t)(in ? t : 0) * A.stride;
            off[j][t] = in ? (uint32_t)A.Aj[s] * (uint32_t)sizeof(V) : own[j];
            a[j][t] = in ? stored<VT>(Ax, s) : V(0);
        }
#pragma unroll
        for (int t = 0; t < kWidth; ++t) pc[j][t] = *(const V *)((const char *)pv + off[j][t]);
        xl[j][tid] = xin[rr];
        rl[j][tid] = rv[rr];
        po[j] = pv[rr];
        if constexpr (PCG) dl[j][tid] = dinv[rr];
        if (live) agent_store_bits((it_begin & 1) ? pub1 : pub0, own[j], EmptyOf<V>::value);
    }
    // word of (chunk c, work-group h): h nchunks + the index of the SpMV
    // work-group that serves c; of (sum m, work-group h, group b)
    auto word_a = [&](int i, int part) { return words + (i & 1) * kWordsA + part * nchunks; };
    auto word_b = [&](int i, int part) { return words + 2 * kWordsA + (i & 1) * kWordsB + part * g2; };
    const bool poster = tid < kGroupChunks && b + tid * g2 < nchunks;   // thread k posts chunk b + k g2
    const int my_a = poster ? (int)xcd_unblock(b + tid * g2, nchunks) : 0;
    if (tid == 0) bad = 0;
    if (tid < 16) {
        red_a[tid] = 0.0;
#pragma unroll
        for (int m = 0; m < NRED; ++m) red_b[m][tid] = 0.0;
    }
    const V initial = (V)sc->initial, eps_rel = (V)sc->eps_rel;
    const int max_iters = sc->max_iters;
    V alpha = (V)sc->alpha, factor = V(0), current = V(0);   // alpha: |r|^2 (CG), r.z (PCG)
    bool stop = false, conv = false, ok = arrive != 0;   // 0: give up at the first wait
    int it = it_begin;
    __syncthreads();
    while (true) {
        // v = A p, partial p.v per chunk
        V v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
            V s = V(0);
            const int n = here(len[j]);
#pragma unroll
            for (int t = 0; t < kWidth; ++t) s = t < n ? s + a[j][t] * pc[j][t] : s;
            v[j] = s;
            const double ws = wave_sum(len[j] >= 0 ? (double)s * (double)po[j] : 0.0);
            const int pr = w + kWaves * j;
            if (lane == 0) wsum[pr / R][pr % R] = ws;
        }
        __builtin_amdgcn_s_waitcnt(0);   // everything emptied is out
        __syncthreads();
        if (poster) {
            double q[R];
#pragma unroll
            for (int i = 0; i < R; ++i) q[i] = wsum[tid][i];
            post(word_a(it, h) + my_a, combine(q));
        }
        // everyone's partials: sum_partials over the SpMV work-groups
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            if (m * kThreads >= nchunks) break;
            double acc = 0.0;
            for (int i = tid + m * kThreads; i < nchunks; i += 1024) {
                double q[Q];
#pragma unroll
                for (int u = 0; u < Q; ++u) q[u] = 0.0;
                if (ok) ok = take(word_a(it, 0) + i, nchunks, q, it == it_begin ? arrive : kWaitTicks);
                acc += combine(q);
            }
            acc = wave_sum(acc);
            if (lane == 0) red_a[w + m * kWaves] = acc;
        }
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) break;
        const V dv = (V)tree16(red_a, lane);
        V lambda;
        if constexpr (PCG)
            lambda = ((dv < 0 ? -dv : dv) >= e) ? alpha / dv : alpha / e;
        else
            lambda = alpha / ((dv < 0 ? -dv : dv) > e ? dv : e);
        const V mlambda = -lambda;
        // x += lambda p, r -= lambda v; publish r (z); squares.  Everyone has
        // posted A, so the previous iteration's published values are read.
        V *const pub = (it & 1) ? pub1 : pub0, *const pub_next = (it & 1) ? pub0 : pub1;
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int pr = w + kWaves * j, k = pr / R, col = (pr % R) * kWave + lane;
            double s0 = 0.0, s1 = 0.0;
            if (len[j] >= 0) {
                xl[j][tid] += po[j] * lambda;
                const V ri = rl[j][tid] + v[j] * mlambda;
                rl[j][tid] = ri;
                V zi = ri;
                if constexpr (PCG) zi = dl[j][tid] * ri;
                const uint32_t o = here(own[j]);
                agent_store_bits(pub, o, __builtin_bit_cast(Bits, zi));
                agent_store_bits(pub_next, o, EmptyOf<V>::value);
                s0 = (double)zi * (double)ri;
                s1 = (double)ri * (double)ri;
            }
            sq[0][k][col] = s0;
            if constexpr (PCG) sq[1][k][col] = s1;
        }
        if constexpr (!kEarly) __builtin_amdgcn_s_waitcnt(0);   // published before B is posted
        __syncthreads();
        if (tid < 64 * R) {
#pragma unroll
            for (int m = 0; m < NRED; ++m) {
                double acc = 0.0;
#pragma unroll
                for (int k = 0; k < kGroupChunks; ++k) acc += sq[m][k][tid];
                acc = wave_sum(acc);
                if constexpr (R == 1) {
                    if (lane == 0) post(word_b(it, m * Q + h) + b, acc);
                } else {
                    if (lane == 0) bsum[m][w] = acc;
                }
            }
        }
        if constexpr (R > 1) {
            __syncthreads();
            if (tid < NRED) {
                double q[R];
#pragma unroll
                for (int i = 0; i < R; ++i) q[i] = bsum[tid][i];
                post(word_b(it, tid * Q + h) + b, combine(q));
            }
        }
        // the sum, and meanwhile the published values at the rows' columns
        Bits g[kEarly ? R : 1][kWidth];
        auto ask = [&](int j, int u) {
#pragma unroll
            for (int t = 0; t < kWidth; ++t) g[u][t] = agent_load_bits(pub, here(off[j][t]));
        };
        {
            uint64_t q[NRED * Q], t0 = 0;
#pragma unroll
            for (int i = 0; i < NRED * Q; ++i) q[i] = 0;
            bool need = tid < g2, want = kEarly;
            if constexpr (kEarly) {
#pragma unroll
                for (int j = 0; j < R; ++j) ask(j, j);
            }
            for (uint32_t spin = 0; ok && (need || want); ++spin) {
                if (need) {
#pragma unroll
                    for (int i = 0; i < NRED * Q; ++i) q[i] = agent_load(word_b(it, 0) + tid + i * g2);
                }
                if constexpr (kEarly) {
                    // only what is missing is read again
                    want = false;
#pragma unroll
                    for (int j = 0; j < R; ++j)
#pragma unroll
                        for (int t = 0; t < kWidth; ++t)
                            if (len[j] >= 0 && g[j][t] == EmptyOf<V>::value) {
                                g[j][t] = agent_load_bits(pub, here(off[j][t]));
                                want = true;
                            }
                }
                if (need) {
                    need = false;
#pragma unroll
                    for (int i = 0; i < NRED * Q; ++i) need = need || q[i] == kEmpty;
                }
                if ((spin & 255u) == 255u) ok = in_time(t0, kWaitTicks) && !agent_load(&sc->aborted);
            }
            if (w * kWave < g2) {
#pragma unroll
                for (int m = 0; m < NRED; ++m) {
                    double f[Q];
#pragma unroll
                    for (int u = 0; u < Q; ++u) f[u] = __builtin_bit_cast(double, q[m * Q + u]);
                    const double sum = wave_sum(0.0 + combine(f));
                    if (lane == 0) red_b[m][w] = sum;
                }
            }
        }
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) break;
        const V alpha_old = alpha;
        alpha = (V)tree16(red_b[0], lane);
        // everyone has posted B: the words of A(it) and of the previous B are read
        if (tid < NRED) agent_store(word_b(it + 1, tid * Q + h) + b, kEmpty);
        if (poster) agent_store(word_a(it, h) + my_a, kEmpty);
        ++it;
        if constexpr (PCG) {
            factor = ((alpha_old < 0 ? -alpha_old : alpha_old) >= e) ? alpha / alpha_old : alpha / e;
            current = sqrt((V)tree16(red_b[NRED - 1], lane));
            conv = current < initial * eps_rel;
            stop = conv || it >= max_iters;
        } else {
            factor = alpha / ((alpha_old < 0 ? -alpha_old : alpha_old) > e ? alpha_old : e);
            current = sqrt(alpha);
            stop = current < eps_rel * initial || current < eps_rel || it >= max_iters;
        }
        if (stop) break;
        // the direction at the own row and at the row's columns
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int u = kEarly ? j : 0;
            if constexpr (!kEarly) ask(j, u);
#pragma unroll
            for (int t = 0; t < kWidth; ++t) {
                const V f = pc[j][t] * factor, gv = __builtin_bit_cast(V, g[u][t]);
                if constexpr (PCG)
                    pc[j][t] = gv + f;
                else
                    pc[j][t] = f + gv;
            }
            const V f = po[j] * factor;
            if constexpr (PCG)
                po[j] = dl[j][tid] * rl[j][tid] + f;
            else
                po[j] = f + rl[j][tid];
        }
        if (it >= it_end) break;
    }
    if (bad) {
        if (tid == 0) agent_store(&sc->aborted, 1);
        return;
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        if (len[j] < 0) continue;
        *(V *)((char *)xs + own[j]) = xl[j][tid];
        *(V *)((char *)pv + own[j]) = po[j];
        *(V *)((char *)rv + own[j]) = rl[j][tid];
    }
    if (blockIdx.x == 0 && tid == 0) {
        sc->carry[it & 1] = (double)alpha;
        sc->alpha = (double)alpha;
        sc->talpha = (double)factor;
        sc->iters = it;
        sc->current = (double)current;
        if (PCG) sc->converged = conv ? 1 : 0;
        if (stop) sc->done = 1;
    }
}

// x = xs once the solve is over and no work-group gave up
template <typename V>
__global__ __launch_bounds__(256) void k_cg_commit(V *x, const V *xs, int64_t n, const CGScalars *sc) {
    if (!sc->done || sc->aborted) return;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        x[i] = xs[i];
}

constexpr int kMaxDevices = 64;
std::atomic<int> g_leased[kMaxDevices];

int groups(int64_t rows) { return (int)((rows + kChunk * kGroupChunks - 1) / (kChunk * kGroupChunks)); }
int split(int64_t rows) { return rows <= kFourRows ? 4 : (rows <= kTwoRows ? 2 : 1); }

__global__ __launch_bounds__(256) void k_empty_words(uint64_t *w, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) w[i] = kEmpty;
}

template <typename VT, bool PCG>
hipError_t launch(const EllView &A, const void *dinv, const void *xin, void *x, void *xs, void *p, void *r, void *pub0,
                  void *pub1, CGScalars *sc, uint64_t *words, int it_begin, int it_end, uint64_t arrive, hipStream_t s) {
    typedef typename VecOf<VT>::type V;
    const int nchunks = (int)((A.rows + kChunk - 1) / kChunk), g2 = groups(A.rows);
#define RUN(R)                                                                                                  \
    hipLaunchKernelGGL((k_cg_resident<VT, PCG, R>), dim3(g2 * (4 / R)), dim3(kThreads), 0, s, A, (const V *)dinv, \
                       (const V *)xin, (V *)xs, (V *)p, (V *)r, (V *)pub0, (V *)pub1, sc, words, nchunks, g2, it_begin, it_end, \
                       arrive)
    switch (split(A.rows)) {
        case 4: RUN(1); break;
        case 2: RUN(2); break;
        default: RUN(4);
    }
#undef RUN
    const int64_t g = (A.rows + 1023) / 1024;
    hipLaunchKernelGGL((k_cg_commit<V>), dim3((unsigned)g), dim3(256), 0, s, (V *)x, (const V *)xs, A.rows,
                       (const CGScalars *)sc);
    return hipGetLastError();
}

}  // namespace

// T = 1 matrices of at most 9 stored entries per row whose rows two rounds of
// partials cover; anything else goes launch by launch.
bool cg_resident_fits(const EllView &A) {
    return A.threads == 1 && A.index_words == 1 && A.ncpr >= 1 && A.ncpr <= kWidth && A.rows >= 1 &&
           A.rows <= kMaxChunks * kChunk;
}

// Iterations from which a resident launch pays for bringing the rows in: up to
// one (two / three) launch by launch against resident, us a call, FP64: 65^2
// rows 66 / 69 (82 / 72), 385^2 75 / 80 (97 / 85), 513^2 79 / 95 (104 / 106),
// 720^2 92 / 100 (128 / 114); bf16: 513^2 72 / 98 (94 / 108; 115 / 118), 720^2
// 76 / 105 (102 / 116; 128 / 127).
size_t cg_resident_from(const EllView &A) { return A.rows > kTwoRows && A.vtype != VT_F64 ? 3 : 2; }

ResidentLease::ResidentLease(const EllView &A, const ReduceSlots &slots) {
    if (!cg_resident_fits(A) || (int64_t)slots.capacity * 4 < kWords) return;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return;
    const int need = groups(A.rows) * split(A.rows);
    if (g_leased[dev].fetch_add(need) + need > cus) {
        g_leased[dev].fetch_sub(need);
        return;
    }
    dev_ = dev;
    count_ = need;
}
ResidentLease::~ResidentLease() {
    if (count_) g_leased[dev_].fetch_sub(count_);
}

hipError_t cg_resident(const EllView &A, const void *dinv, const void *xin, void *x, void *xs, void *p, void *r,
                       void *pub0, void *pub1, CGScalars *sc, const ReduceSlots &sl, int it_begin, int it_end,
                       bool give_up, hipStream_t s) {
    const uint64_t arrive = give_up ? 0 : kArriveTicks;
    uint64_t *words = (uint64_t *)sl.partials;
    if (it_begin == 0)
        hipLaunchKernelGGL(k_empty_words, dim3((kWords + 255) / 256), dim3(256), 0, s, words, (int)kWords);
#define RES(VT)                                                                                              \
    return dinv ? launch<VT, true>(A, dinv, xin, x, xs, p, r, pub0, pub1, sc, words, it_begin, it_end, arrive, s)             \
                : launch<VT, false>(A, dinv, xin, x, xs, p, r, pub0, pub1, sc, words, it_begin, it_end, arrive, s)
    switch (A.vtype) {
        case VT_F32: RES(float);
        case VT_F64: RES(double);
        case VT_BF16: RES(bf16);
    }
#undef RES
    return hipErrorInvalidValue;
}

}  // namespace hipx
}  // namespace honei
