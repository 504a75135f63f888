// coarse_kernels.hip -- the coarse end of a V-cycle on Q1 hierarchies in one
// launch, one work-group per system: levels 1..top (33^2 nodes in FP64, 65^2
// otherwise, at most), from the restricted defect of the level above (or the
// system's own right-hand side) to the correction it prolongs.
//
// Launch by launch these levels cost three launches each of 3-5 us in which
// almost nothing runs.  Here vectors live in LDS, and each interior node's
// weights, dinv and rhs with the thread that owns it, in registers (of the
// levels that one wavefront runs: in LDS between their phases).  Weights come
// from the cell coefficients (or are the constant stencil), so no matrix is
// read; every global load of a system is issued before the first use.  Nodes
// go row by row over the lanes, so a stencil is one LDS address and fixed
// offsets, without a test for the boundary: below the finest level the
// boundary's right-hand side and correction are 0 and it stays 0 in LDS; the
// finest level's is a node of its own for a few threads.  Levels up to 9^2 and
// the 3^2 CG run in one wavefront, without barriers; the CG's sums and products
// are register moves between its nine lanes.
//
// What bounds it: FP64 arithmetic of the weights (a fifth), VALU issue of the
// 65^2 phases (a third), and the chain of short phases below.  One system of
// 257^2 nodes 18.9 us (constant operator 14.5); 16 bf16 systems of levels
// 5..8 19.8; 256 systems of up to 513^2 nodes 23.7.  (With a thread's four nodes of 65^2
// sixteen rows apart, so that they share neither cells nor staged rows: 20.5,
// 16.1, 22.4, 25.8; with flat node numbers, five a thread, and weights in LDS
// below 33^2: 26.5 for the first; an earlier launch for levels 1..4 alone: 32.)
// Distinct weights read instead of formed: 21.8 against 20.9.
//
// Sums and roundings are those of the level-by-level launches: rows in column
// order, boundary rows 0 + 1 x, transfers as k_b_restrict_rows /
// prolong_value, the CG as coarse_cg_block.

#include "batch.hh"

#include "q1_device.hh"
#include "solver_device.hh"
#include "transfer_device.hh"

#pragma clang fp contract(off)

namespace honei {
namespace hipx {
namespace {

constexpr int kThreads = 1024, kWaves = kThreads / kWave;
constexpr int kWaveTop = 3;    // levels up to here run in wavefront 0

__host__ __device__ constexpr int side_at(int l) { return (1 << l) + 1; }
__host__ __device__ constexpr int nodes_at(int l) { return side_at(l) * side_at(l); }
// LDS, in elements: the coarsest solution, then two vectors per level; behind
// them what lanes without a node may read (never used)
__host__ __device__ constexpr int vec_at(int l) {
    int o = nodes_at(1);
    for (int k = 2; k < l; ++k) o += 2 * nodes_at(k);
    return o;
}
constexpr int kTail = 160;
__host__ __device__ constexpr int lds_elements(int top) { return (vec_at(top + 1) + kTail + 3) / 4 * 4; }

// Interior nodes over threads: a wavefront takes `rows` grid rows of `cols`
// columns (a power of two, one more than the level's interior); a thread has
// np nodes, one above the other (np > 1: rows = 1).  So a node's stencil is one
// address and fixed offsets, and a thread's nodes share staged rows and cells.
template <int L> struct Lv {
    static constexpr int side = side_at(L), n = nodes_at(L);
    static constexpr bool wave = L <= kWaveTop;
    static constexpr int cols = 1 << L < kWave ? 1 << L : kWave, rows = kWave / cols;
    static constexpr int waves = (1 << L) / rows < 1 ? 1 : ((1 << L) / rows < kWaves ? (1 << L) / rows : kWaves);
    static constexpr int np = ((1 << L) + waves * rows - 1) / (waves * rows);
    static_assert((1 << L) <= cols && (np == 1 || rows == 1), "one lane per column");
};

// what a thread keeps of its interior nodes: in registers; of the wavefront's
// levels in LDS, in registers only while the level runs
template <typename V, int NP> struct Regs {
    V w[NP][9], di[NP], rh[NP];
};
// ... and what that is made from, as loaded (rhs used on the finest level only)
template <typename V, int NP> struct Raw {
    double c[NP + 1][2];
    V di[NP], rh[NP];
};
constexpr int kKeep = 11 * kWave;   // LDS elements of one of the wavefront's levels


// The lane as a phase sees it: positions, masks and addresses formed from it
// are formed in the phase again (a few instructions) instead of being kept in
// registers from one phase to the others.
__device__ inline int fresh(int t) {
    asm volatile("" : "+v"(t));
    return t;
}

template <int L> __device__ inline void level_sync() {
    if constexpr (Lv<L>::wave) {
        // LDS accesses of one wavefront complete in order; the compiler keeps it too
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

template <typename V> __device__ inline V lane_value(V v, int lane) {
    if constexpr (sizeof(V) == 4) {
        return __builtin_bit_cast(V, __builtin_amdgcn_readlane(__builtin_bit_cast(uint32_t, v), lane));
    } else {
        const uint64_t b = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), lane);
        return __builtin_bit_cast(V, (uint64_t)lo | ((uint64_t)hi << 32));
    }
}

// Node 0 of this thread on level L: grid position and LDS index; node q is q
// rows further.
template <int L> struct Pos {
    int r, c, id;
    bool mine;   // the wavefront takes part
    __device__ inline Pos(int lane_, int wv) {
        const int lane = fresh(lane_);
        r = 1 + wv * Lv<L>::rows * Lv<L>::np + lane / Lv<L>::cols;
        c = 1 + lane % Lv<L>::cols;
        id = r * Lv<L>::side + c;
        mine = wv < Lv<L>::waves;
    }
    __device__ inline bool live(int q) const {
        return c < Lv<L>::side - 1 && r + q < Lv<L>::side - 1;
    }
};

template <typename VT, bool COEF, int TOP> struct Cycle {
    typedef typename VecOf<VT>::type V;
    V *mem;
    int lane, wv;    // of this thread
    bool odd_pre;    // an odd number of sweeps follows the first two: the iterate ends in the second vector
    const CoarseCycle &cc;
    // the finest level's boundary node of this thread (id < 0: none); on the
    // other levels the boundary stays 0: right-hand side and correction are
    int bid;
    V bdi, brh;

    template <int L> __device__ inline V *iterate() const { return mem + vec_at(L) + (odd_pre ? Lv<L>::n : 0); }
    template <int L> __device__ inline V *other() const { return mem + vec_at(L) + (odd_pre ? 0 : Lv<L>::n); }
    // where the level's result is after the up-leg
    template <int L> __device__ inline const V *result() const {
        if constexpr (L == 1) return mem;
        return (cc.n_post & 1) ? iterate<L>() : other<L>();
    }

    // cells, dinv and rhs of the thread's nodes as wavefront v of the level's
    template <int L> __device__ inline void fetch(Raw<V, Lv<L>::np> &raw, int64_t g, int v) const {
        constexpr int S = Lv<L>::side;
        const CoarseLevel &cl = cc.lv[L];
        const Pos<L> p(lane, v);
        if (!p.mine) return;
        const V *dinv = (const V *)cl.dinv + g * cl.vld, *rhs = (const V *)cl.rhs + g * cl.vld;
        const double *kap = cl.kappa + g * cl.kld;
        // a lane without a node: the last interior one's
        const int c = min(p.c, S - 2);
        if constexpr (COEF) {
#pragma unroll
            for (int k = 0; k <= Lv<L>::np; ++k) {
                const double *cs = kap + (min(p.r - 1 + k, S - 2) * (S - 1) + c - 1);
                raw.c[k][0] = cs[0];
                raw.c[k][1] = cs[1];
            }
        }
#pragma unroll
        for (int q = 0; q < Lv<L>::np; ++q) {
            const int r = min(p.r + q, S - 2);
            raw.di[q] = dinv[r * S + c];
            raw.rh[q] = rhs[r * S + c];
        }
    }
    // weights; on the finest level the first operand dinv .* rhs
    template <int L>
    __device__ inline void settle(Regs<V, Lv<L>::np> &reg, const Raw<V, Lv<L>::np> &raw, bool top, int v) const {
        const Pos<L> p(lane, v);
        if (!p.mine) return;
        if constexpr (COEF) q1_column_weights<VT, Lv<L>::np, V>(raw.c, reg.w);
#pragma unroll
        for (int q = 0; q < Lv<L>::np; ++q) {
            reg.di[q] = raw.di[q];
            reg.rh[q] = raw.rh[q];
            if (top && p.live(q))
                (mem + vec_at(L) + Lv<L>::n)[p.id + q * Lv<L>::side] = raw.di[q] * raw.rh[q];
        }
    }

    // the wavefront's levels: put away and taken back by their lanes
    template <int L> __device__ inline V *kept() const { return mem + lds_elements(TOP) + (L - 2) * kKeep + lane; }
    template <int L> __device__ inline void put(const Regs<V, Lv<L>::np> &reg) const {
        V *k = kept<L>();
        if constexpr (COEF) {
#pragma unroll
            for (int i = 0; i < 9; ++i) k[i * kWave] = reg.w[0][i];
        }
        k[9 * kWave] = reg.di[0];
        k[10 * kWave] = reg.rh[0];
    }
    template <int L> __device__ inline void get(Regs<V, Lv<L>::np> &reg) const {
        const V *k = kept<L>();
        if constexpr (COEF) {
#pragma unroll
            for (int i = 0; i < 9; ++i) reg.w[0][i] = k[i * kWave];
        }
        reg.di[0] = k[9 * kWave];
        reg.rh[0] = k[10 * kWave];
    }

    // DEFECT: dst = rhs - A src; else a Jacobi sweep (from zero: src = dinv .* rhs)
    template <int L, bool DEFECT> __device__ inline void sweep(const V *src, V *dst, const Regs<V, Lv<L>::np> &reg, bool top) const {
        constexpr int S = Lv<L>::side;
        const Pos<L> p(lane, wv);
        if (p.mine) {
            src += p.id - S - 1;
            V x[3][3], w[9];
            if constexpr (!COEF) q1_constant_weights<VT, V>(w);
#pragma unroll
            for (int k = 0; k < Lv<L>::np + 2; ++k) {   // staged row k: above node k - 2
#pragma unroll
                for (int j = 0; j < 3; ++j) x[k % 3][j] = src[k * S + j];
                if (k < 2) continue;
                const int q = k - 2;
                V s = V(0);
#pragma unroll
                for (int i = 0; i < 9; ++i) s = s + (COEF ? reg.w[q][i] : w[i]) * x[(q + i / 3) % 3][i % 3];
                const V d = reg.rh[q] - s;
                if (p.live(q)) dst[p.id + q * S] = DEFECT ? d : x[(q + 1) % 3][1] + d * reg.di[q];
            }
            src -= p.id - S - 1;
        }
        if (top && bid >= 0) {
            const V x = src[bid], d = brh - (V(0) + V(1) * x);
            dst[bid] = DEFECT ? d : x + d * bdi;
        }
    }

    // the right-hand side of level C from the defect of the finer one (its
    // border is Dirichlet: 0), value(q, s) taking node q's
    template <int C, typename F> __device__ inline void restrict_to(F &&value) const {
        constexpr int SF = Lv<C + 1>::side;
        const Pos<C> p(lane, wv);
        if (!p.mine) return;
        const V *f = other<C + 1>() + 2 * p.r * SF + 2 * p.c;
#pragma unroll
        for (int q = 0; q < Lv<C>::np; ++q) {
            const V *f0 = f + q * 2 * SF, *fm = f0 - SF, *fp = f0 + SF;
            const int d = p.c - (p.r + q);
            const V h = V(0.5), qq = V(0.25);
            const V A_ = h * fm[0], B_ = h * fp[0], C_ = h * f0[1], D_ = h * f0[-1];
            const V E_ = qq * fp[1], F_ = qq * fp[-1], G_ = qq * fm[1], H_ = qq * fm[-1];
            V s = f0[0];
            s = d <= -1 ? s + D_ : s;
            s = d <= -2 ? s + C_ : s;
            s = s + A_;
            s = d == -1 ? s + C_ : s;
            s = d == 0 ? s + D_ : s;
            s = s + G_;
            s = s + H_;
            s = s + B_;
            s = d == 0 ? s + C_ : s;
            s = d == 1 ? s + D_ : s;
            s = s + E_;
            s = s + F_;
            s = d >= 2 ? s + D_ : s;
            s = d >= 1 ? s + C_ : s;
            value(q, s);
        }
    }
    template <int C> __device__ inline void restrict_to_level(Regs<V, Lv<C>::np> &reg) const {
        const Pos<C> p(lane, wv);
        restrict_to<C>([&](int q, V s) {
            reg.rh[q] = s;
            if (p.live(q)) (mem + vec_at(C) + Lv<C>::n)[p.id + q * Lv<C>::side] = reg.di[q] * s;
        });
    }

    // from the level's rhs and first operand to its defect
    template <int L> __device__ inline void down(const Regs<V, Lv<L>::np> &reg, bool top) const {
        V *x = mem + vec_at(L), *y = x + Lv<L>::n;
        sweep<L, false>(y, x, reg, top);
        level_sync<L>();
        for (int k = 2; k < cc.n_pre; ++k) {
            sweep<L, false>((k & 1) ? y : x, (k & 1) ? x : y, reg, top);
            level_sync<L>();
        }
        sweep<L, true>(iterate<L>(), other<L>(), reg, top);
        level_sync<L>();
    }

    template <int L> __device__ inline void up(const Regs<V, Lv<L>::np> &reg, bool top) const {
        constexpr int nc = Lv<L - 1>::side;
        V *a = other<L>(), *b = iterate<L>();
        const V *xc = result<L - 1>();
        const Pos<L> p(lane, wv);
        if (p.mine) {
#pragma unroll
            for (int q = 0; q < Lv<L>::np; ++q) {
                const int r = p.r + q, c = p.c, id = p.id + q * Lv<L>::side;
                const V *c0 = xc + (r >> 1) * nc + (c >> 1), *c1 = xc + ((r + 1) >> 1) * nc + (c >> 1);
                const int dc = c & 1;
                const V t0 = c0[0], t1 = c0[dc], t2 = c1[0], t3 = c1[dc];
                const V h = V(0.5), qq = V(0.25);
                const V f_rc = ((V(0) + t0 * qq + t1 * qq) + t2 * qq) + t3 * qq;
                const V f_c = (V(0) + t0 * h) + t1 * h, f_r = (V(0) + t0 * h) + t2 * h;
                const V f = (r & 1) ? ((c & 1) ? f_rc : f_r) : ((c & 1) ? f_c : t0);
                const V v = b[id] + f * V(1);
                if (p.live(q)) a[id] = v;
            }
        }
        if (top && bid >= 0) a[bid] = b[bid] + V(0) * V(1);
        level_sync<L>();
        for (int k = 0; k < cc.n_post; ++k) {
            sweep<L, false>((k & 1) ? b : a, (k & 1) ? a : b, reg, top);
            level_sync<L>();
        }
    }

    // coarse_cg_block on the 3 x 3 grid by wavefront 0, lane = node; rhs: the
    // centre's (the border's is 0), w: the centre row (the others are 0 + 1 x)
    __device__ inline void coarse_cg(V centre, const V (&w)[9]) const {
        const int t = lane;
        const bool in = t < 9;
        const V rhs = t == 4 ? centre : V(0);
        const V e = eps_of<V>();
        auto mul = [&](V v) {
            V s = V(0);
#pragma unroll
            for (int k = 0; k < 9; ++k) s += w[k] * lane_value(v, k);
            return t == 4 ? s : V(0) + V(1) * v;
        };
        auto sum = [&](V a, V b) {
            const double s = wave_sum(in ? (double)a * (double)b : 0.0);
            return (V)lane_value(s, 0);
        };
        auto ratio = [&](V up_, V low_) { return (low_ < 0 ? -low_ : low_) >= e ? V(up_ / low_) : V(up_ / e); };
        V x = V(0), gr = mul(x) - rhs, u = gr * V(-1.);
        V norm_x = sum(x, x), norm_x_last = V(norm_x - V(1));
        for (int it = 0; (double)(norm_x - norm_x_last) > cc.konv && it < cc.max_iters; ++it) {
            V upper = sum(gr, gr);
            V en = mul(u);
            V lower = sum(en, u);
            const V f1 = ratio(upper, lower);
            en = u * f1 + x;
            lower = upper;
            gr = mul(en) - rhs;
            upper = sum(gr, gr);
            const V f2 = ratio(upper, lower);
            u = u * f2 - gr;
            x = en;
            norm_x_last = norm_x;
            norm_x = sum(x, x);
        }
        if (in) mem[t] = x;
    }
};

template <typename VT, bool COEF, int TOP>
__global__ __launch_bounds__(kThreads) void k_coarse_cycle(CoarseCycle cc, BWork w) {
    typedef typename VecOf<VT>::type V;
    __shared__ __attribute__((aligned(16))) V mem[lds_elements(TOP) + 2 * kKeep + 12];
    const int64_t a0 = w.bounds[w.lo], na = w.bounds[w.hi] - w.bounds[w.lo];
    const int t = threadIdx.x, lane = t % kWave, wv = __builtin_amdgcn_readfirstlane(t / kWave);
    for (int64_t a = blockIdx.x; a < na; a += gridDim.x) {
        const int64_t g = w.list[a0 + a];
        int top = cc.top;
        while (top > 2 && g >= cc.lv[top].cap) --top;   // systems whose finest level is lower
        Cycle<VT, COEF, TOP> c{mem, lane, wv, (cc.n_pre & 1) != 0, cc, -1, V(0), V(0)};
        const CoarseLevel &cl = cc.lv[top];
        // every global load of the system before the first use (initialised:
        // else what a branch leaves unset lives on from system to system)
        Raw<V, Lv<TOP >= 6 ? 6 : 5>::np> f6{};
        Raw<V, 1> f5{}, f4{}, fw{};
        if constexpr (TOP >= 6) {
            if (top >= 6) c.template fetch<6>(f6, g, wv);
        }
        if (top >= 5) c.template fetch<5>(f5, g, wv);
        if (top >= 4) c.template fetch<4>(f4, g, wv);
        // wavefronts 1 and 2 make wavefront 0's levels, 3 the centre row of level 1
        if (wv == 1 && top >= 3) c.template fetch<3>(fw, g, 0);
        if (wv == 2) c.template fetch<2>(fw, g, 0);
        if constexpr (COEF) {
            if (wv == 3) {
                const double *k = cc.lv[1].kappa + g * cc.lv[1].kld;
#pragma unroll
                for (int i = 0; i < 4; ++i) fw.c[0][i] = k[i];
            }
        }
        // the finest level's boundary: bottom, top, left, right without corners twice
        const int e = (1 << top), side = e + 1;
        if (t < 4 * e) {
            const int k = t & (e - 1), part = t >> top;
            c.bid = part == 0 ? k : (part == 1 ? e * side + k + 1 : (part == 2 ? (k + 1) * side : k * side + e));
            c.bdi = ((const V *)cl.dinv + g * cl.vld)[c.bid];
            c.brh = ((const V *)cl.rhs + g * cl.vld)[c.bid];
        }
        for (int i = t; i < lds_elements(TOP) / 4; i += kThreads) {
            V *m = mem + 4 * i;
            m[0] = m[1] = m[2] = m[3] = V(0);
        }
        __syncthreads();
        if (wv >= 1 && wv <= 3) {
            Regs<V, 1> rw{};
            if (wv == 1 && top >= 3) {
                c.template settle<3>(rw, fw, top == 3, 0);
                c.template put<3>(rw);
            }
            if (wv == 2) {
                c.template settle<2>(rw, fw, top == 2, 0);
                c.template put<2>(rw);
            }
            if (wv == 3) {
                if constexpr (COEF)
                    q1_interior_weights_cells<VT, V>(fw.c[0][0], fw.c[0][1], fw.c[0][2], fw.c[0][3], rw.w[0]);
                else
                    q1_constant_weights<VT, V>(rw.w[0]);
#pragma unroll
                for (int k = 0; k < 9; ++k) mem[lds_elements(TOP) + 2 * kKeep + k] = rw.w[0][k];
            }
        }
        Regs<V, Lv<TOP >= 6 ? 6 : 5>::np> r6{};
        Regs<V, 1> r5{}, r4{};
        if (top >= 4) c.template settle<4>(r4, f4, top == 4, wv);
        if (top >= 5) c.template settle<5>(r5, f5, top == 5, wv);
        if constexpr (TOP >= 6) {
            if (top >= 6) c.template settle<6>(r6, f6, top == 6, wv);
        }
        if (c.bid >= 0) mem[cl.at + cl.n + c.bid] = c.bdi * c.brh;
        __syncthreads();
        if constexpr (TOP >= 6) {
            if (top >= 6) {
                c.template down<6>(r6, top == 6);
                c.template restrict_to_level<5>(r5);
                __syncthreads();
            }
        }
        if (top >= 5) {
            c.template down<5>(r5, top == 5);
            c.template restrict_to_level<4>(r4);
            __syncthreads();
        }
        if (top >= 4) c.template down<4>(r4, top == 4);
        if (wv == 0) {
            if (top >= 3) {
                Regs<V, 1> r3{};
                c.template get<3>(r3);
                if (top >= 4) {
                    c.template restrict_to_level<3>(r3);
                    c.template put<3>(r3);
                    level_sync<3>();
                }
                c.template down<3>(r3, top == 3);
            }
            {
                Regs<V, 1> r2{};
                c.template get<2>(r2);
                if (top >= 3) {
                    c.template restrict_to_level<2>(r2);
                    level_sync<2>();
                }
                c.template down<2>(r2, top == 2);
                V centre = V(0), w1[9];
                c.template restrict_to<1>([&](int, V s) { centre = s; });
#pragma unroll
                for (int k = 0; k < 9; ++k) w1[k] = mem[lds_elements(TOP) + 2 * kKeep + k];
                c.coarse_cg(lane_value(centre, 0), w1);
                level_sync<1>();
                c.template up<2>(r2, top == 2);
            }
            if (top >= 3) {
                Regs<V, 1> r3{};
                c.template get<3>(r3);
                c.template up<3>(r3, top == 3);
            }
        }
        __syncthreads();
        if (top >= 4) c.template up<4>(r4, top == 4);
        if (top >= 5) c.template up<5>(r5, top == 5);
        if constexpr (TOP >= 6) {
            if (top >= 6) c.template up<6>(r6, top == 6);
        }
        // the finest level's result
        V *out = (V *)cl.x + g * cl.vld;
        const V *src = mem + cl.at + (((cc.n_pre ^ cc.n_post) & 1) ? 0 : cl.n);
        for (int i = t; i < cl.n; i += kThreads) out[i] = src[i];
        __syncthreads();
    }
}

}  // namespace

int64_t coarse_top(ValueType vt) { return vt == VT_F64 ? 5 : 6; }

hipError_t b_coarse_cycle(ValueType vt, const CoarseCycle &cc, const BWork &w, int64_t max_slots, hipStream_t s) {
    if (max_slots <= 0) return hipSuccess;
    if (cc.top < 2 || cc.top > coarse_top(vt) || cc.n_pre < 2 || cc.n_post < 0) return hipErrorInvalidValue;
    CoarseCycle c = cc;
    const bool coef = cc.lv[1].kappa != nullptr;
    for (int l = 1; l <= cc.top; ++l) {
        c.lv[l].n = nodes_at(l);
        c.lv[l].at = vec_at(l);
        if (!cc.lv[l].dinv || cc.lv[l].vld < nodes_at(l) || (l > 1 && cc.lv[l].cap > cc.lv[l - 1].cap) ||
            (cc.lv[l].kappa != nullptr) != coef || (coef && cc.lv[l].kld < (int64_t(1) << (2 * l))))
            return hipErrorInvalidValue;
    }
    const dim3 grid((unsigned)(max_slots < 2048 ? max_slots : 2048)), block(kThreads);
#define CYCLE(VT, TOP)                                                                       \
    do {                                                                                     \
        if (coef)                                                                            \
            hipLaunchKernelGGL((k_coarse_cycle<VT, true, TOP>), grid, block, 0, s, c, w);    \
        else                                                                                 \
            hipLaunchKernelGGL((k_coarse_cycle<VT, false, TOP>), grid, block, 0, s, c, w);   \
    } while (0)
    if (vt == VT_F32)
        CYCLE(float, 6);
    else if (vt == VT_BF16)
        CYCLE(bf16, 6);
    else if (vt == VT_F64)
        CYCLE(double, 5);
    else
        return hipErrorInvalidValue;
#undef CYCLE
    return hipGetLastError();
}

}  // namespace hipx
}  // namespace honei
