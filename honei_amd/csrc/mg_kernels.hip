// mg_kernels.hip -- FP64 outer iterations of the single-system multigrid
// solvers on device-assembled Q1 hierarchies (MGHierarchy::solve_mixed and
// solve_pcg): matrix-free row sums, reductions fused into the pass that forms
// their operands, scalars on the device.
//
// The outer operator is the Q1 operator of a lexicographic side x side grid,
// so a row's neighbours follow from its position and its weights are the
// constant stencil or a fixed expression of the cell coefficients
// (q1_device.hh): a pass reads 8 bytes per cell (or none) instead of the
// stored row's 108.  Sums keep the order of the launches they replace: rows in
// column order; a defect's norm per 256-row work-group of ell_row_kernel; the
// other dots and norms as k_reduce forms them.

#include "solvers.hh"

#include "q1_device.hh"

#pragma clang fp contract(off)

namespace honei {
namespace hipx {
namespace {

constexpr int kRows = 1024;   // threads of the reducing passes: four columns of k_reduce's 256
constexpr int kLanes = 256;

// Grid position of a row and the offsets of its stencil (a boundary row's
// neighbours: itself, loaded and never used).
struct Q1Pos {
    uint32_t r, c;
    bool bnd;
};
__device__ inline Q1Pos q1_pos(int64_t row, int32_t side) {
    Q1Pos p;
    p.r = (uint32_t)row / (uint32_t)side;
    p.c = (uint32_t)row - p.r * (uint32_t)side;
    p.bnd = p.r == 0 || p.c == 0 || p.r == (uint32_t)side - 1 || p.c == (uint32_t)side - 1;
    return p;
}
// The stored row's sum (q1_row, threads = 1) over the operand value(j); mid
// receives the own value.
template <bool COEF, typename F>
__device__ inline double q1_sum(int64_t row, int32_t side, const double *kappa, F &&value, double &mid) {
    const Q1Pos p = q1_pos(row, side);
    double x[9], w[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) x[k] = value(p.bnd ? row : row + (int64_t)(k / 3 - 1) * side + (k % 3 - 1));
    if constexpr (COEF)
        q1_stored_weights<double, double>(side, p.r, p.c, p.bnd, kappa, w);
    else
        q1_constant_weights<double, double>(w);
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k) s = s + w[k] * x[k];
    mid = x[4];
    return p.bnd ? 0.0 + x[4] : s;
}

// d = b - A x with the partials of ||d||^2; ACC: x = (xold null: 0, else
// xold) + e * *scale first, formed at every neighbour from the same operands
// and stored by its own row into xnew.
template <bool COEF, bool ACC>
__global__ __launch_bounds__(256) void k_mg_defect(int32_t side, int64_t n, const double *kappa, const double *b,
                                                   const double *x, const float *e, const double *scale, double *xnew,
                                                   double *d, double *partials, int64_t nlogical, const int *skip,
                                                   const int *gate) {
    if ((skip && *skip) || (gate && !*gate)) return;
    const int64_t p = xcd_block(blockIdx.x, gridDim.x);
    const int64_t per = nlogical / gridDim.x, rem = nlogical % gridDim.x;
    const int64_t first = p * per + (p < rem ? p : rem), last = first + per + (p < rem ? 1 : 0);
    const double sc = ACC ? *scale : 0.0;
    double nval = 0.0;
    for (int64_t lb = first; lb < last; ++lb) {
        const int64_t row = lb * 256 + threadIdx.x;
        if (row >= n) continue;
        auto value = [&](int64_t j) {
            if constexpr (ACC)
                return (x ? x[j] : 0.0) + (double)e[j] * sc;
            else
                return x[j];
        };
        double own;
        const double s = q1_sum<COEF>(row, side, kappa, value, own);
        const double r = b[row] - s;
        d[row] = r;
        if constexpr (ACC) xnew[row] = own;
        nval += r * r;
    }
    const double v = block_sum(nval);
    if (threadIdx.x == 0) partials[blockIdx.x] = v;
}

// k_reduce's sum over the rows of its work-group `blockIdx.x`, by 1024
// threads: k_reduce's thread t adds rows t + k * stride into accumulator k
// mod 4, here thread (k mod 4, t) does, and the four meet in LDS.  Stores the
// partial.
template <typename F> __device__ inline void reduce_rows(int64_t n, double *partials, F &&term) {
    __shared__ double acc[4][kLanes];
    __shared__ double red[4];
    const int t = threadIdx.x % kLanes, u = threadIdx.x / kLanes;
    const int64_t stride = (int64_t)gridDim.x * kLanes;
    double a = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)kLanes + t + u * stride; i < n; i += 4 * stride) a += term(i);
    acc[u][t] = a;
    __syncthreads();
    if (u == 0) {
        const double v = wave_sum((acc[0][t] + acc[1][t]) + (acc[2][t] + acc[3][t]));
        if (t % kWave == 0) red[t / kWave] = v;
    }
    __syncthreads();
    // block_sum's tree over four wave sums
    if (threadIdx.x == 0) partials[blockIdx.x] = (red[0] + red[2]) + (red[1] + red[3]);
}

template <typename Z> __device__ inline double widen(Z x, double nrm) {
    if constexpr (sizeof(Z) == 4)
        return 0.0 + (double)x * nrm;
    else
        return x * nrm;
}

// partials of r.z, z = |r| x
template <typename Z>
__global__ __launch_bounds__(kRows) void k_mg_rz(const double *r, const Z *x, int64_t n, const MgPcgScalars *sc,
                                                 double *prz) {
    if (sc->halt) return;
    const double nrm = sc->nrm;
    reduce_rows(n, prz, [&](int64_t i) { return r[i] * widen(x[i], nrm); });
}

// beta from the partials of r.z (every work-group the same value), p = z +
// beta p_old, q = A p and, with DOT, the partials of p.q; p is formed at every
// neighbour from the same operands and stored by its own row.
// DOT gives a work-group the 2048 rows of one of k_reduce's partials; while
// those are too few to fill the chip (kSplitRows) a work-group takes 256 rows
// and k_mg_pq forms the sum: 257^2 nodes 4.8 + 3.1 us instead of 13.2.
constexpr int64_t kSplitRows = 524288;   // 256 partials: also what 256 threads sum in k_finish_sum's order
template <bool COEF, typename Z, bool DOT>
__global__ __launch_bounds__(DOT ? kRows : kLanes) void k_mg_dir(int32_t side, int64_t n, const double *kappa,
                                                                 const Z *x, const double *pold, double *pnew,
                                                                 double *q, MgPcgScalars *sc, const double *prz,
                                                                 int64_t nparts, double *ppq) {
    if (sc->halt) return;
    const double rho_prev = sc->rho_prev, nrm = sc->nrm;
    const double rz = sum_partials(prz, nparts, 1, 0);
    const double beta = (rho_prev > 0.0 && rz > 0.0) ? rz / rho_prev : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->rz = rz;
        sc->beta = beta;
        sc->iters += 1;
    }
    auto row = [&](int64_t i) {
        double own;
        auto value = [&](int64_t j) {
            const double z = widen(x[j], nrm);
            return beta == 0.0 ? z : z + pold[j] * beta;
        };
        const double s = q1_sum<COEF>(i, side, kappa, value, own);
        pnew[i] = own;
        q[i] = s;
        return own * s;
    };
    if constexpr (DOT) {
        reduce_rows(n, ppq, row);
    } else {
        const int64_t i = xcd_block(blockIdx.x, gridDim.x) * kLanes + threadIdx.x;
        if (i < n) (void)row(i);
    }
}

__global__ __launch_bounds__(kRows) void k_mg_pq(const double *p, const double *q, int64_t n, const MgPcgScalars *sc,
                                                 double *ppq) {
    if (sc->halt) return;
    reduce_rows(n, ppq, [&](int64_t i) { return p[i] * q[i]; });
}

// alpha from the partials of p.q (breakdown: done), x += alpha p, r -= alpha
// q and the partials of ||r||^2
__global__ __launch_bounds__(kRows) void k_mg_update(double *x, const double *p, double *r, const double *q, int64_t n,
                                                     MgPcgScalars *sc, const double *ppq, int64_t nparts,
                                                     double *pr2) {
    // block 0 of this launch may set halt: read it once per work-group
    if (block_uniform_flag(&sc->halt)) return;
    const double rz = sc->rz;
    const double pq = sum_partials(ppq, nparts, 1, 0);
    if (!(pq > 0.0) || !(rz > 0.0)) {   // breakdown: not converged
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            sc->done = sc->halt = 1;
            sc->work.end = 0;
        }
        return;
    }
    const double alpha = rz / pq, malpha = -alpha;
    reduce_rows(n, pr2, [&](int64_t i) {
        x[i] += p[i] * alpha;
        const double v = r[i] + q[i] * malpha;
        r[i] = v;
        return v * v;
    });
}

// after the update: the iteration's decision from the partials of ||r||^2, the
// same in every thread that has r2; whether the solve goes on, and its norm
__device__ inline bool pcg_goes_on(const MgPcgScalars *sc, double r2, double &nrm, bool &verify) {
    nrm = sqrt(r2);
    verify = nrm < sc->tol * sc->initial;
    return !verify && sc->iters < sc->cap && isfinite(nrm);
}
__device__ inline void pcg_decide(MgPcgScalars &c, double r2, double nrm, bool verify, bool on) {
    c.r2 = r2;
    c.nrm = nrm;
    c.rho_prev = c.rz;
    if (verify)
        c.verify = 1;
    else if (!on)
        c.done = 1;
    c.halt = c.verify | c.done;
    c.work.end = c.halt ? 0 : 1;
}
__global__ __launch_bounds__(1024) void k_mg_check(MgPcgScalars *sc, const double *pr2, int64_t nparts) {
    if (block_uniform_flag(&sc->halt)) return;
    const double r2 = sum_partials(pr2, nparts, 1, 0);
    if (threadIdx.x != 0) return;
    double nrm;
    bool verify;
    const bool on = pcg_goes_on(sc, r2, nrm, verify);
    pcg_decide(*sc, r2, nrm, verify, on);
}

// INIT after the first defect, CONFIRM after the gated true defect (one
// work-group): ||d||^2 from the defect's partials and the decision
__global__ __launch_bounds__(1024) void k_mg_pcg_defect(int init, MgPcgScalars *sc, const double *partials,
                                                        int64_t nparts, double tol, int cap) {
    if (!init && !block_uniform_flag(&sc->verify)) return;
    const double h = sum_partials(partials, nparts, 1, 0);
    if (threadIdx.x != 0) return;
    MgPcgScalars &c = *sc;
    c.verify = 0;
    c.nrm = sqrt(h);
    c.rho_prev = 0.0;   // CONFIRM: drifted, restart from the true residual
    if (init) {
        c.initial = c.nrm;
        c.tol = tol;
        c.iters = 0;
        c.cap = cap;
        c.alpha = c.malpha = c.beta = 0.0;
        c.done = (c.initial > 0.0 && cap > 0 && isfinite(c.nrm)) ? 0 : 1;
    } else {
        c.done = (c.nrm < c.tol * c.initial || !(c.iters < c.cap) || !isfinite(c.nrm)) ? 1 : 0;
    }
    c.halt = c.done;
    c.work = OneSlot{0, 0, c.done ? 0 : 1};
}

// rhs = d * inv in the inner precision
template <typename V>
__global__ __launch_bounds__(256) void k_mg_rhs(V *rhs, const double *d, int64_t n, const double *inv,
                                                const double *nrm, const int *halt) {
    if (*halt) return;
    const double f = inv ? *inv : 1.0 / *nrm;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        rhs[i] = (V)(d[i] * f);
}

// the decision of the iteration before and this one's right-hand side, up to
// kSplitRows rows: every work-group sums the (at most 256) partials and comes
// to the same decision, the first writes it (the others read nothing that it
// changes, but for a halt, which they come to themselves); 257^2 nodes 2.0 and
// 3.9 us in two launches
template <typename V>
__global__ __launch_bounds__(256) void k_mg_check_rhs(V *rhs, const double *d, int64_t n, MgPcgScalars *sc,
                                                      const double *pr2, int64_t nparts) {
    if (block_uniform_flag(&sc->halt)) return;
    const double r2 = sum_partials(pr2, nparts, 1, 0);
    double nrm;
    bool verify;
    const bool on = pcg_goes_on(sc, r2, nrm, verify);
    if (blockIdx.x == 0 && threadIdx.x == 0) pcg_decide(*sc, r2, nrm, verify, on);
    if (!on) return;
    const double f = 1.0 / nrm;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        rhs[i] = (V)(d[i] * f);
}

// the MIXED driver's decision after a defect (one work-group)
__global__ __launch_bounds__(1024) void k_mg_mixed_check(int init, MgMixedScalars *sc, const double *partials,
                                                         int64_t nparts, double tol, int64_t cap) {
    if (!init && block_uniform_flag(&sc->done)) return;
    const double h = sum_partials(partials, nparts, 1, 0);
    if (threadIdx.x != 0) return;
    MgMixedScalars &c = *sc;
    c.norm = sqrt(h);
    if (init) {
        c.initial = c.norm;
        c.scale = c.inv = 1.0;
        c.outer = 0;
        c.done = 0;
        c.work = OneSlot{0, 0, 1};
        return;
    }
    c.outer += 1;
    if (c.norm < tol * c.initial || c.outer >= cap || !isfinite(c.norm)) {
        c.done = 1;
        c.work.end = 0;
    } else {
        c.scale = c.norm;
        c.inv = 1.0 / c.scale;
    }
}

int64_t dot_groups(int64_t n) {   // k_reduce's grid
    const int64_t g = (n + 2047) / 2048;
    return g < 1 ? 1 : (g > 2048 ? 2048 : g);
}
int64_t defect_groups(int64_t n, const ReduceSlots &sl) {
    const int64_t g = (n + 255) / 256;
    return g > sl.capacity ? sl.capacity : g;
}
unsigned stream_groups(int64_t n) {
    const int64_t g = (n + 1023) / 1024;
    return (unsigned)(g < 1 ? 1 : (g > 8192 ? 8192 : g));
}
// partials: the defect's in [0, capacity), then r.z, p.q, |r|^2
double *parts(const ReduceSlots &sl, int k) { return sl.partials + sl.capacity + k * 2048; }

}  // namespace

hipError_t mg_defect(const Q1Outer &o, const double *b, const double *x, const float *e, const double *scale,
                     double *xnew, double *d, const ReduceSlots &sl, const int *skip, const int *gate, hipStream_t s) {
    const int64_t nl = (o.n + 255) / 256;
    const dim3 g((unsigned)defect_groups(o.n, sl)), blk(256);
#define DEFECT(C, A)                                                                                                  \
    hipLaunchKernelGGL((k_mg_defect<C, A>), g, blk, 0, s, o.side, o.n, o.kappa, b, x, e, scale, xnew, d, sl.partials, nl, \
                       skip, gate)
    if (o.kappa) {
        if (e) DEFECT(true, true); else DEFECT(true, false);
    } else {
        if (e) DEFECT(false, true); else DEFECT(false, false);
    }
#undef DEFECT
    return hipGetLastError();
}

hipError_t mg_mixed_check(bool init, MgMixedScalars *sc, int64_t n, const ReduceSlots &sl, double tol, int64_t cap,
                          hipStream_t s) {
    hipLaunchKernelGGL(k_mg_mixed_check, dim3(1), dim3(1024), 0, s, init ? 1 : 0, sc, (const double *)sl.partials,
                       defect_groups(n, sl), tol, cap);
    return hipGetLastError();
}

hipError_t mg_mixed_rhs(float *rhs, const double *d, int64_t n, const MgMixedScalars *sc, hipStream_t s) {
    hipLaunchKernelGGL(k_mg_rhs<float>, dim3(stream_groups(n)), dim3(256), 0, s, rhs, d, n, &sc->inv,
                       (const double *)nullptr, &sc->done);
    return hipGetLastError();
}

hipError_t mg_pcg_defect(bool init, const Q1Outer &o, const double *b, const double *x, double *r, MgPcgScalars *sc,
                         const ReduceSlots &sl, double tol, int cap, hipStream_t s) {
    HX(mg_defect(o, b, x, nullptr, nullptr, nullptr, r, sl, nullptr, init ? nullptr : &sc->verify, s));
    hipLaunchKernelGGL(k_mg_pcg_defect, dim3(1), dim3(1024), 0, s, init ? 1 : 0, sc, (const double *)sl.partials,
                       defect_groups(o.n, sl), tol, cap);
    return hipGetLastError();
}

bool mg_pcg_late_check(int64_t n) { return n <= kSplitRows; }

hipError_t mg_pcg_check_rhs(ValueType inner, void *rhs, const double *r, int64_t n, MgPcgScalars *sc,
                            const ReduceSlots &sl, hipStream_t s) {
    const double *pr2 = parts(sl, 2);
    if (inner == VT_F64)
        hipLaunchKernelGGL(k_mg_check_rhs<double>, dim3(stream_groups(n)), dim3(256), 0, s, (double *)rhs, r, n, sc, pr2,
                           dot_groups(n));
    else
        hipLaunchKernelGGL(k_mg_check_rhs<float>, dim3(stream_groups(n)), dim3(256), 0, s, (float *)rhs, r, n, sc, pr2,
                           dot_groups(n));
    return hipGetLastError();
}

hipError_t mg_pcg_rhs(ValueType inner, void *rhs, const double *r, int64_t n, const MgPcgScalars *sc, hipStream_t s) {
    if (inner == VT_F64)
        hipLaunchKernelGGL(k_mg_rhs<double>, dim3(stream_groups(n)), dim3(256), 0, s, (double *)rhs, r, n,
                           (const double *)nullptr, &sc->nrm, &sc->halt);
    else
        hipLaunchKernelGGL(k_mg_rhs<float>, dim3(stream_groups(n)), dim3(256), 0, s, (float *)rhs, r, n,
                           (const double *)nullptr, &sc->nrm, &sc->halt);
    return hipGetLastError();
}

hipError_t mg_pcg_outer(ValueType inner, const Q1Outer &o, const void *x_top, double *x, double *r, const double *pold,
                        double *pnew, double *q, MgPcgScalars *sc, const ReduceSlots &sl, bool check,
                        hipStream_t s) {
    const int64_t g = dot_groups(o.n);
    const dim3 grid((unsigned)g), blk(kRows);
    double *prz = parts(sl, 0), *ppq = parts(sl, 1), *pr2 = parts(sl, 2);
    const bool split = o.n <= kSplitRows;
    const dim3 rows((unsigned)((o.n + kLanes - 1) / kLanes)), lanes(kLanes);
#define DIR(C, Z)                                                                                                  \
    do {                                                                                                           \
        if (split)                                                                                                 \
            hipLaunchKernelGGL((k_mg_dir<C, Z, false>), rows, lanes, 0, s, o.side, o.n, o.kappa, (const Z *)x_top, \
                               pold, pnew, q, sc, (const double *)prz, g, ppq);                                    \
        else                                                                                                       \
            hipLaunchKernelGGL((k_mg_dir<C, Z, true>), grid, blk, 0, s, o.side, o.n, o.kappa, (const Z *)x_top,    \
                               pold, pnew, q, sc, (const double *)prz, g, ppq);                                    \
    } while (0)
#define OUTER(Z)                                                                                                   \
    do {                                                                                                           \
        hipLaunchKernelGGL(k_mg_rz<Z>, grid, blk, 0, s, (const double *)r, (const Z *)x_top, o.n,                  \
                           (const MgPcgScalars *)sc, prz);                                                         \
        if (o.kappa)                                                                                               \
            DIR(true, Z);                                                                                          \
        else                                                                                                       \
            DIR(false, Z);                                                                                         \
    } while (0)
    if (inner == VT_F64)
        OUTER(double);
    else
        OUTER(float);
#undef OUTER
#undef DIR
    if (split)
        hipLaunchKernelGGL(k_mg_pq, grid, blk, 0, s, (const double *)pnew, (const double *)q, o.n,
                           (const MgPcgScalars *)sc, ppq);
    hipLaunchKernelGGL(k_mg_update, grid, blk, 0, s, x, (const double *)pnew, r, (const double *)q, o.n, sc,
                       (const double *)ppq, g, pr2);
    if (check) hipLaunchKernelGGL(k_mg_check, dim3(1), dim3(1024), 0, s, sc, (const double *)pr2, g);
    return hipGetLastError();
}

}  // namespace hipx
}  // namespace honei
