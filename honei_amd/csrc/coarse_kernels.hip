// coarse_kernels.hip -- the coarse end of a V-cycle on Q1 hierarchies in one
// launch, one work-group per system: levels 1..top (33^2 nodes in FP64, 65^2
// otherwise, at most), from the restricted defect of the level above (or the
// system's own right-hand side) to the correction it prolongs.
//
// Launch by launch these levels cost three launches each of 3-5 us in which
// almost nothing runs.  Here vectors live in LDS and a node's weights with
// the thread that owns the node: in registers from 33^2 nodes up (five nodes
// a thread at 65^2), in LDS below.  Weights come from the cell coefficients
// (or are the constant stencil), so no matrix is read.  Levels up to 9^2 and
// the 3^2 CG run in one wavefront, without barriers; the CG's four sums and
// two products per iteration are register moves between its nine lanes.  What
// bounds it is the chain of phases (six per level, each an LDS round trip
// and 18 dependent roundings per node) and the CG.
//
// 18 systems, levels 1..6: 23 us against 28-30 us for levels 1..4 in the
// earlier one-launch form and six launches for levels 5 and 6; one system of
// 257^2 nodes 26 us against 32 us and six launches.  256 systems of up to
// 513^2 nodes: 26 us against 38 us and six launches.  Five nodes a thread with
// positions kept across phases spilled 170 registers (45 us): `fresh`.
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

constexpr int kThreads = 1024;
constexpr int kWaveTop = 3;    // levels up to here run in wavefront 0
constexpr int kRegFrom = 5;    // levels from here keep weights, dinv and rhs in registers

__host__ __device__ constexpr int side_at(int l) { return (1 << l) + 1; }
__host__ __device__ constexpr int nodes_at(int l) { return side_at(l) * side_at(l); }
// LDS, in elements: two vectors per level, then nine weights, dinv and rhs of
// the levels below kRegFrom
__host__ __device__ constexpr int vec_at(int l) {
    int o = 0;
    for (int k = 1; k < l; ++k) o += 2 * nodes_at(k);
    return o;
}
__host__ __device__ constexpr int low_at(int l, int top) {
    int o = vec_at(top + 1);
    for (int k = 1; k < l; ++k) o += 11 * nodes_at(k);
    return o;
}
__host__ __device__ constexpr int lds_elements(int top) { return low_at(kRegFrom < top + 1 ? kRegFrom : top + 1, top); }

template <int L> struct Lv {
    static constexpr int side = side_at(L), n = nodes_at(L);
    static constexpr bool wave = L <= kWaveTop, regs = L >= kRegFrom;
    static constexpr int threads = wave ? kWave : kThreads;
    static constexpr int np = (n + threads - 1) / threads;   // nodes per thread
};

// what a thread keeps of its nodes of a register level
template <typename V, int L> struct Regs {
    V w[Lv<L>::np][9], di[Lv<L>::np], rh[Lv<L>::np];
};

// Node q of this thread on level L (clamped to the last one) and the interior
// node whose stencil fits its position.
template <int L> struct Node {
    int id, base;
    bool live, bnd;
    __device__ inline Node(int t, int q) {
        constexpr int S = Lv<L>::side;
        const int i = t + q * Lv<L>::threads;
        live = i < Lv<L>::n;
        id = live ? i : Lv<L>::n - 1;
        const int r = id / S, c = id - r * S;
        bnd = r == 0 || c == 0 || r == S - 1 || c == S - 1;
        const int ir = r < 1 ? 1 : (r > S - 2 ? S - 2 : r), ic = c < 1 ? 1 : (c > S - 2 ? S - 2 : c);
        base = ir * S + ic;
    }
};

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

// The thread index as a phase sees it: positions, masks and addresses formed
// from it are formed in the phase again (a few instructions) instead of being
// kept in registers from one phase to the others.
__device__ inline int fresh(int t) {
    asm volatile("" : "+v"(t));
    return t;
}

template <typename VT, bool COEF, int TOP> struct Cycle {
    typedef typename VecOf<VT>::type V;
    V *mem;
    int t;           // thread of the work-group
    bool odd_pre;    // an odd number of sweeps follows the first two: the iterate ends in the second vector
    const CoarseCycle &cc;

    template <int L> __device__ inline V *iterate() const { return mem + vec_at(L) + (odd_pre ? Lv<L>::n : 0); }
    template <int L> __device__ inline V *other() const { return mem + vec_at(L) + (odd_pre ? 0 : Lv<L>::n); }
    template <int L> __device__ inline V *low() const { return mem + low_at(L, TOP); }
    // where the level's result is after the up-leg
    template <int L> __device__ inline const V *result() const {
        if constexpr (L == 1) return mem + vec_at(1);
        return (cc.n_post & 1) ? iterate<L>() : other<L>();
    }

    // weights and dinv of the level's nodes; top: its right-hand side too
    template <int L, typename R> __device__ inline void load(R &reg, int64_t g, bool top) const {
        const CoarseLevel &cl = cc.lv[L];
        const V *dinv = (const V *)cl.dinv + g * cl.vld, *rhs = (const V *)cl.rhs + g * cl.vld;
        constexpr int S = Lv<L>::side, NP = Lv<L>::regs ? Lv<L>::np : 1;
        const int t = fresh(this->t);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const int i = t + q * kThreads;
            if (!Lv<L>::regs && i >= Lv<L>::n) break;
            const int id = i < Lv<L>::n ? i : Lv<L>::n - 1, r = id / S, c = id - r * S;
            V w[9];
            if constexpr (COEF) {
                const int ir = r < 1 ? 1 : (r > S - 2 ? S - 2 : r), ic = c < 1 ? 1 : (c > S - 2 ? S - 2 : c);
                const double *cs = cl.kappa + g * cl.kld + ((ir - 1) * (S - 1) + ic - 1), *cs2 = cs + (S - 1);
                q1_interior_weights_cells<VT, V>(cs[0], cs[1], cs2[0], cs2[1], w);
            } else {
                q1_constant_weights<VT, V>(w);
            }
            const V di = dinv[id], rh = top ? rhs[id] : V(0);
            if constexpr (Lv<L>::regs) {
#pragma unroll
                for (int k = 0; k < 9; ++k) reg.w[q][k] = w[k];
                reg.di[q] = di;
                reg.rh[q] = rh;
            } else {
                V *lo = low<L>();
#pragma unroll
                for (int k = 0; k < 9; ++k) lo[k * Lv<L>::n + id] = w[k];
                lo[9 * Lv<L>::n + id] = di;
                lo[10 * Lv<L>::n + id] = rh;
            }
            if (L > 1 && top && i < Lv<L>::n) (mem + vec_at(L) + Lv<L>::n)[id] = di * rh;
        }
    }

    // DEFECT: dst = rhs - A src; else a Jacobi sweep (from zero: src = dinv .* rhs)
    template <int L, bool DEFECT, typename R>
    __device__ inline void sweep(const V *src, V *dst, const R &reg) const {
        constexpr int S = Lv<L>::side;
        const int t = fresh(this->t);
#pragma unroll
        for (int q = 0; q < Lv<L>::np; ++q) {
            const Node<L> nd(t, q);
            V x[9], s = V(0), di, rh;
#pragma unroll
            for (int k = 0; k < 9; ++k) x[k] = src[k == 4 ? nd.id : nd.base + (k / 3 - 1) * S + (k % 3 - 1)];
            if constexpr (Lv<L>::regs) {
                if constexpr (COEF) {
#pragma unroll
                    for (int k = 0; k < 9; ++k) s = s + reg.w[q][k] * x[k];
                }
                di = reg.di[q];
                rh = reg.rh[q];
            } else {
                const V *lo = low<L>() + nd.id;
                if constexpr (COEF) {
#pragma unroll
                    for (int k = 0; k < 9; ++k) s = s + lo[k * Lv<L>::n] * x[k];
                }
                di = lo[9 * Lv<L>::n];
                rh = lo[10 * Lv<L>::n];
            }
            if constexpr (!COEF) {
                V w[9];
                q1_constant_weights<VT, V>(w);
#pragma unroll
                for (int k = 0; k < 9; ++k) s = s + w[k] * x[k];
            }
            s = nd.bnd ? V(0) + V(1) * x[4] : s;
            const V d = rh - s;
            if (nd.live) dst[nd.id] = DEFECT ? d : x[4] + d * di;
        }
    }

    // the right-hand side of level L - 1 from the defect of level L, and its
    // first operand dinv .* rhs
    template <int L, typename R> __device__ inline void restrict_to_coarser(R &reg) const {
        constexpr int C = L - 1, S = Lv<L>::side, m = Lv<C>::side - 1;
        const V *f = other<L>();
        const int t = fresh(this->t);
#pragma unroll
        for (int q = 0; q < Lv<C>::np; ++q) {
            const Node<C> nd(t, q);
            const int ir = nd.base / Lv<C>::side, ic = nd.base - ir * Lv<C>::side;
            const int d = ic - ir;
            const V *f0 = f + 2 * ir * S + 2 * ic, *fm = f0 - S, *fp = f0 + S;
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
            s = nd.bnd ? V(0) : s;
            static_assert(m >= 2, "coarse grids have an interior");
            V di;
            if constexpr (Lv<C>::regs) {
                reg.rh[q] = s;
                di = reg.di[q];
            } else {
                V *lo = low<C>() + nd.id;
                if (nd.live) lo[10 * Lv<C>::n] = s;
                di = lo[9 * Lv<C>::n];
            }
            if (C > 1 && nd.live) (mem + vec_at(C) + Lv<C>::n)[nd.id] = di * s;
        }
    }

    // from the level's rhs and first operand to the coarser level's
    template <int L, typename R, typename RC> __device__ inline void down(const R &reg, RC &rc) const {
        V *x = mem + vec_at(L), *y = x + Lv<L>::n;
        sweep<L, false>(y, x, reg);
        level_sync<L>();
        for (int k = 2; k < cc.n_pre; ++k) {
            sweep<L, false>((k & 1) ? y : x, (k & 1) ? x : y, reg);
            level_sync<L>();
        }
        sweep<L, true>(iterate<L>(), other<L>(), reg);
        level_sync<L>();
        if constexpr (Lv<L - 1>::wave == Lv<L>::wave) {
            restrict_to_coarser<L>(rc);
            level_sync<L>();
        }
    }

    template <int L, typename R> __device__ inline void up(const R &reg) const {
        constexpr int S = Lv<L>::side, nc = Lv<L - 1>::side;
        V *a = other<L>(), *b = iterate<L>();
        const V *xc = result<L - 1>();
        const int t = fresh(this->t);
#pragma unroll
        for (int q = 0; q < Lv<L>::np; ++q) {
            const Node<L> nd(t, q);
            const int r = nd.id / S, c = nd.id - r * S;
            const int rlo = r >> 1, rhi = (r + 1) >> 1, clo = c >> 1, chi = (c + 1) >> 1;
            const V t0 = xc[rlo * nc + clo], t1 = xc[rlo * nc + chi], t2 = xc[rhi * nc + clo], t3 = xc[rhi * nc + chi];
            const V h = V(0.5), qq = V(0.25);
            const V f_rc = ((V(0) + t0 * qq + t1 * qq) + t2 * qq) + t3 * qq;
            const V f_c = (V(0) + t0 * h) + t1 * h, f_r = (V(0) + t0 * h) + t2 * h;
            V f = (r & 1) ? ((c & 1) ? f_rc : f_r) : ((c & 1) ? f_c : t0);
            f = nd.bnd ? V(0) : f;
            const V v = b[nd.id] + f * V(1);
            if (nd.live) a[nd.id] = v;
        }
        level_sync<L>();
        for (int k = 0; k < cc.n_post; ++k) {
            sweep<L, false>((k & 1) ? b : a, (k & 1) ? a : b, reg);
            level_sync<L>();
        }
    }

    // coarse_cg_block on the 3 x 3 grid by wavefront 0, lane = node
    __device__ inline void coarse_cg() const {
        const bool in = t < 9;
        const V *lo = low<1>();
        V w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = lo[k * 9 + 4];   // the centre row; the others are 0 + 1 x
        const V rhs = in ? lo[90 + t] : V(0);
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
        if (in) (mem + vec_at(1))[t] = x;
    }
};

struct None {};

template <typename VT, bool COEF, int TOP>
__global__ __launch_bounds__(kThreads) void k_coarse_cycle(CoarseCycle cc, BWork w) {
    typedef typename VecOf<VT>::type V;
    __shared__ V mem[lds_elements(TOP)];
    const int64_t a0 = w.bounds[w.lo], na = w.bounds[w.hi] - w.bounds[w.lo];
    const int t = threadIdx.x;
    for (int64_t a = blockIdx.x; a < na; a += gridDim.x) {
        const int64_t g = w.list[a0 + a];
        int top = cc.top;
        while (top > 1 && g >= cc.lv[top].cap) --top;   // systems whose finest level is lower
        const Cycle<VT, COEF, TOP> c{mem, t, (cc.n_pre & 1) != 0, cc};
        None no;
        Regs<V, 5> r5;
        Regs<V, TOP >= 6 ? 6 : 5> r6;
        if constexpr (TOP >= 6) {
            if (top >= 6) c.template load<6>(r6, g, top == 6);
        }
        if (top >= 5) c.template load<5>(r5, g, top == 5);
        if (top >= 4) c.template load<4>(no, g, top == 4);
        if (top >= 3) c.template load<3>(no, g, top == 3);
        if (top >= 2) c.template load<2>(no, g, top == 2);
        c.template load<1>(no, g, top == 1);
        __syncthreads();
        if constexpr (TOP >= 6) {
            if (top >= 6) c.template down<6>(r6, r5);
        }
        if (top >= 5) c.template down<5>(r5, no);
        if (top >= 4) c.template down<4>(no, no);
        if (t < kWave) {
            if (top >= 4) {
                c.template restrict_to_coarser<4>(no);
                level_sync<3>();
            }
            if (top >= 3) c.template down<3>(no, no);
            if (top >= 2) c.template down<2>(no, no);
            c.coarse_cg();
            level_sync<1>();
            if (top >= 2) c.template up<2>(no);
            if (top >= 3) c.template up<3>(no);
        }
        __syncthreads();
        if (top >= 4) c.template up<4>(no);
        if (top >= 5) c.template up<5>(r5);
        if constexpr (TOP >= 6) {
            if (top >= 6) c.template up<6>(r6);
        }
        // the finest level's result
        const CoarseLevel &cl = cc.lv[top];
        V *out = (V *)cl.x + g * cl.vld;
        const int n = cl.n, at = cc.lv[top].at;
        const bool first = top == 1 || (((cc.n_pre ^ cc.n_post) & 1) != 0);
        const V *src = mem + at + (first ? 0 : n);
        for (int i = t; i < n; i += kThreads) out[i] = src[i];
        __syncthreads();
    }
}

}  // namespace

int64_t coarse_top(ValueType vt) { return vt == VT_F64 ? 5 : 6; }

hipError_t b_coarse_cycle(ValueType vt, const CoarseCycle &cc, const BWork &w, int64_t max_slots, hipStream_t s) {
    if (max_slots <= 0) return hipSuccess;
    if (cc.top < 1 || cc.top > coarse_top(vt) || cc.n_pre < 2 || cc.n_post < 0) return hipErrorInvalidValue;
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
