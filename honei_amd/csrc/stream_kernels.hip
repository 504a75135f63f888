// stream_kernels.hip -- the paired row passes of large Q1 levels, one
// wavefront marching down a column strip.
#include "batch.hh"
#include "q1_device.hh"

namespace honei {
namespace hipx {
namespace {

// The lane to the left's / right's value (lane 0 / lane 63: zero).
template <int CTRL>
__device__ inline float lane_shift(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ inline double lane_shift(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <typename T> __device__ inline T from_west(T v) { return lane_shift<0x138>(v); }
template <typename T> __device__ inline T from_east(T v) { return lane_shift<0x130>(v); }

// A strip is at most kStreamWidth columns (two halo columns each side fill a
// wavefront; the restriction takes one more to the west and ends on an even
// one: two columns fewer).  Segments are long, medium or short: the longest
// of which the running systems give kStreamFill (four wavefronts a SIMD), so
// that a few systems still spread over the chip.  With the rows of the halo
// (four, six with the restriction) a segment is a whole number of rounds of
// six steps, and it starts on an even row.
constexpr int64_t kStreamWidth = 60, kStreamFill = 4096, kStreamBlocks = 4096;
constexpr int kStreamDepth = 3;   // rows in flight

struct StreamGeom {
    int32_t side, width, strips;
    int32_t rows[3], segs[3];   // long, medium and short segments
    int64_t from[2];            // running systems from which the long, the medium ones are taken
};

// Weights of one row of cells (the cell east of the lane's node; the nodes'
// corner and vertical neighbours) and of one row of nodes.
template <typename V> struct CellRow { V corner, across; };
template <typename V> struct NodeRow { V east, diag; };

// The interior row sum of the lane's node: nine terms in column order, below
// (b), own and above (a) rows of x.  A term whose weight and operand both
// belong to the node to the west is formed there and shifted.
template <typename V>
__device__ inline V stencil(const CellRow<V> &b, const NodeRow<V> &n, const CellRow<V> &a, V xb, V x, V xa) {
    V s = V(0);
    s = s + from_west(b.corner * xb);
    s = s + b.across * xb;
    s = s + b.corner * from_east(xb);
    s = s + from_west(n.east * x);
    s = s + n.diag * x;
    s = s + n.east * from_east(x);
    s = s + from_west(a.corner * xa);
    s = s + a.across * xa;
    s = s + a.corner * from_east(xa);
    return s;
}

// k_b_restrict_rows' value of the lane's coarse node (its fine node in this
// lane's column and the middle row), d = coarse column - row, from the defect
// rows below (b), through (m) and above (a) it: the same terms in the same
// order.
template <typename V>
__device__ inline V restrict_value(int d, V b, V m, V a) {
    const V h = V(0.5), q = V(0.25);
    const V C = h * from_east(m), D = h * from_west(m);
    V s = m;
    s = d <= -1 ? s + D : s;
    s = d <= -2 ? s + C : s;
    s = s + h * b;
    s = d == -1 ? s + C : s;
    s = d == 0 ? s + D : s;
    s = s + q * from_east(b);
    s = s + q * from_west(b);
    s = s + h * a;
    s = d == 0 ? s + C : s;
    s = d == 1 ? s + D : s;
    s = s + q * from_east(a);
    s = s + q * from_west(a);
    s = d >= 2 ? s + D : s;
    s = d >= 1 ? s + C : s;
    return s;
}

// k_b_pair's two passes, the same terms in the same order.  A wavefront owns
// `rows` rows by `width` (<= 60) columns of one slot's grid and marches down
// them, one row a step: row r arrives (its operand x formed), row r - 1's
// first-pass value, then row r - 2's second-pass value follow from the last
// three rows, which stay in registers; a node's neighbours to the west and
// east are in the next lanes.  So there is no LDS and no barrier, every
// wavefront runs on its own with D rows' loads in flight, and a weight is
// formed once per cell, edge and node (four divisions a node; nine where
// every node forms its row alone).
// PAIR_PRE writes no defect: when the three defect rows around a coarse row
// are there, its restriction goes out instead (k_b_restrict_rows' terms and
// order).  Only the coarse right-hand side ever reads the defect, so a write
// and a read of it and a launch are saved.  FUSED (PAIR_POST only): with the
// prolongation.
// Bound by memory: 21 (PRE) and 25 bytes a node with weights from the cells,
// and the halo's rows and columns through L2.  51 systems of 513^2 in FP32,
// PRE with the restriction / POST with the prolongation: 89 / 80 us (3.2 /
// 4.2 TB/s) where the tiles of k_b_pair take 117 and 20 for the restriction /
// 118; all levels of 256 systems 159 / 143, tiles 212 and 43 / 223.  One
// system of 1025^2, 513^2, 257^2, 129^2 with the constant operator, PRE: 9.1,
// 5.6, 5.0, 5.5, tiles and restriction 13.8, 9.6, 8.7, 7.9.  Longer segments
// (32 to 68 rows: POST 86) leave the chip less evenly filled, shorter ones
// (8: 85) load more halo; six rows in flight instead of three took 86 (fewer
// wavefronts).  When the last few systems run, short segments take 7 us where
// long ones take 13.
// WM: 1 weights from the cells, 3 the constant operator's.
template <typename VT, int PAIR, int WM, bool FUSED, int D, typename V = typename VecOf<VT>::type>
__global__ __launch_bounds__(256) void k_b_stream(BWork w, StreamGeom g, int64_t vld, const double *kappa, int64_t kld,
                                                  V *out0, const V *xin, const V *rhs, const V *dinv,
                                                  V *xc, int64_t vld_c) {
    constexpr bool RS = PAIR == PAIR_PRE, FP = PAIR == PAIR_POST && FUSED;
    static_assert(!RS || !FUSED, "the prolongation fuses into the post-smoothing pair");
    constexpr int LEAD = RS ? 4 : 2;    // steps before a segment's first row (an even number)
    constexpr int SIDE = RS ? 3 : 2;    // halo columns to the west
    constexpr int U = 6;   // steps per round: a multiple of D, of the three rows kept and of the coarse rows' two
    static_assert(U % D == 0, "ring");
    static_assert(LEAD % 2 == 0, "row parity");
    const int lane = threadIdx.x % kWave;
    const int64_t a0 = w.bounds[w.lo], na = w.bounds[w.hi] - a0;
    const int pick = na >= g.from[0] ? 0 : (na >= g.from[1] ? 1 : 2);
    const int rows = g.rows[pick];
    const uint32_t per = (uint32_t)g.strips * (uint32_t)g.segs[pick];
    const int S = g.side;
    const int64_t total = na * per;
    // every XCD takes one contiguous eighth of the segments, whatever their number
    const int64_t quads = (total + 3) / 4, share = quads / kXcds, more = quads % kXcds;
    const int64_t xcd = blockIdx.x % kXcds, step = (gridDim.x - 1 - xcd) / kXcds + 1;
    const int64_t lo = xcd * share + (xcd < more ? xcd : more), hi = lo + share + (xcd < more ? 1 : 0);
    for (int64_t quad = lo + blockIdx.x / kXcds; quad < hi; quad += step) {
        const int64_t q = quad * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
        if (q >= total) break;
        const uint32_t e = (uint32_t)q / per, rem = (uint32_t)q - e * per;
        const uint32_t seg = rem / (uint32_t)g.strips, strip = rem - seg * (uint32_t)g.strips;
        const int64_t ls = w.list[a0 + e] - w.base;
        const int r0 = (int)seg * rows, r1 = min(S, r0 + rows);
        const int c0 = (int)strip * g.width, c1 = min(S, c0 + g.width);
        const int col = c0 - SIDE + lane;
        const int rlast = __builtin_amdgcn_readfirstlane(min(S - 1, r1 + 1));   // the last row a load asks for
        const bool mine = lane >= SIDE && col < c1;
        const uint32_t cn = (uint32_t)min(max(col, 0), S - 1);    // the lane's node
        const uint32_t cc = (uint32_t)min(max(col, 0), S - 2);    // and cell column (positions outside: never used)
        const bool side_border = cn == 0 || (int)cn == S - 1;
        const V *rs = rhs + ls * vld, *ds = dinv + ls * vld, *xs = xin + ls * vld;
        const double *ks = WM == 1 ? kappa + ls * kld : nullptr;
        V *o0 = out0 + ls * vld;
        // FP: the coarse values left and right of the node's column
        const V *cs = FP ? xc + ls * vld_c : nullptr;
        const int SC = (S >> 1) + 1;
        const uint32_t clo = cn >> 1, chi = (cn + 1) >> 1;
        const uint32_t ct = min(clo, (uint32_t)(SC - 2));

        V di_in = V(0), di_bnd = V(0);
        if constexpr (WM == 3) {
            di_in = dinv[S + 1];
            di_bnd = dinv[0];
        }
        // rows in flight
        V prh[D], pdi[D], pxn[D], pt0[D], pt1[D];
        double pk[D];
        auto load = [&](int r, int i, bool odd) {
            const int rc = min(max(r, 0), rlast);
            const int64_t at = (int64_t)rc * S;
            prh[i] = (rs + at)[cn];
            if constexpr (WM != 3) pdi[i] = (ds + at)[cn];
            if constexpr (PAIR == PAIR_POST) pxn[i] = (xs + at)[cn];
            if constexpr (WM == 1) {
                const int kr = min(max(r - 1, 0), S - 2);   // the cells below the row
                pk[i] = (ks + (int64_t)kr * (S - 1))[cc];
            }
            if constexpr (FP) {
                if (odd) {   // the coarse row above an odd row
                    const V *p = cs + (int64_t)min((rc + 1) >> 1, SC - 1) * SC;
                    pt0[i] = p[ct];
                    pt1[i] = (p + 1)[ct];
                }
            }
        };
#pragma unroll
        for (int i = 0; i < D; ++i) load(r0 - LEAD + i, i, (i & 1) != 0);
        // RS: the last coarse row, on the border, follows one step past the grid
        const int rend = RS && r1 == S ? S + 3 : r1 + 2;
        const int rcoarse = rend - 3;   // the last defect row that completes a coarse row
        V *cr = RS ? xc + ls * vld_c : nullptr;
        V e1 = V(0), e2 = V(0);   // defect rows r - 3, r - 4
        V t0 = V(0), t1 = V(0);   // the coarse row at or below the current row
        if constexpr (FP) {
            const V *p = cs + (int64_t)max((r0 - 2) >> 1, 0) * SC;
            t0 = p[ct];
            t1 = (p + 1)[ct];
        }
        // the last three rows: x, first pass v, rhs, dinv; cells b (one row
        // below), bb (two below) and their weights
        V x1 = V(0), x2 = V(0), v2 = V(0), v3 = V(0), h1 = V(0), h2 = V(0), d1 = V(0), d2 = V(0);
        double k1 = 0.0, across1 = 0.0;
        CellRow<V> cconst{};
        NodeRow<V> nconst{};
        if constexpr (WM == 3) {
            V wv[9];
            q1_constant_weights<VT, V>(wv);
            cconst.corner = wv[0];
            cconst.across = wv[1];
            nconst.east = wv[3];
            nconst.diag = wv[4];
        }
        CellRow<V> c2 = cconst, c3 = cconst;
        NodeRow<V> n2 = nconst;
        auto put = [](double v) {
            V a = (V)v;
            if constexpr (sizeof(VT) == 2) a = bf16_round(a);
            return a;
        };
        for (int base = r0 - LEAD; base < rend; base += U) {
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const int r = base + j, i = j % D;
                const bool odd = (j & 1) != 0;
                // ---- row r arrives ----
                const V h0 = prh[i];
                V d0;
                if constexpr (WM == 3)
                    d0 = (side_border || r <= 0 || r >= S - 1) ? di_bnd : di_in;
                else
                    d0 = pdi[i];
                V x0;
                if constexpr (PAIR == PAIR_PRE) {
                    x0 = d0 * h0;
                } else {
                    x0 = pxn[i];
                    if constexpr (FP) {   // + P xc, as k_b_prolong_rows forms it
                        const V half = V(0.5), q4 = V(0.25);
                        const V tl = clo == ct ? t0 : t1, tr = chi == ct ? t0 : t1;
                        V f;
                        if (odd) {
                            const V u0 = pt0[i], u1 = pt1[i];
                            const V ul = clo == ct ? u0 : u1, ur = chi == ct ? u0 : u1;
                            const V f_rc = ((V(0) + tl * q4 + tr * q4) + ul * q4) + ur * q4;
                            const V f_r = (V(0) + tl * half) + ul * half;
                            f = (cn & 1) ? f_rc : f_r;
                            t0 = u0;
                            t1 = u1;
                        } else {
                            const V f_c = (V(0) + tl * half) + tr * half;
                            f = (cn & 1) ? f_c : tl;
                        }
                        if (side_border || r <= 0 || r >= S - 1) f = V(0);
                        x0 = x0 + f * V(1);
                    }
                }
                // ---- the weights of cell row r - 1 and node row r - 1 ----
                CellRow<V> c1 = cconst;
                NodeRow<V> n1 = nconst;
                if constexpr (WM == 1) {
                    const double k0 = pk[i], kw = from_west(k0);
                    const double pair0 = kw + k0;
                    c1.corner = put(-div3_rn(k0));
                    c1.across = put(-0.5 * div3_rn(pair0));
                    n1.east = put(-0.5 * div3_rn(k1 + k0));
                    n1.diag = put(div3_rn(2.0 * ((across1 + kw) + k0)));
                    k1 = k0;
                    across1 = pair0;
                }
                load(r + D, i, ((j + D) & 1) != 0);
                // ---- row r - 1, first pass ----
                V v1;
                {
                    const int a = r - 1;
                    V sm = stencil(c2, n1, c1, x2, x1, x0);
                    if (side_border || a <= 0 || a >= S - 1) sm = V(0) + V(1) * x1;
                    v1 = x1 + (h1 - sm) * d1;
                    if (PAIR == PAIR_PRE && mine && a >= r0 && a < r1) (o0 + (int64_t)a * S)[cn] = v1;
                }
                // ---- row r - 2, second pass ----
                {
                    const int b = r - 2;
                    V sm = stencil(c3, n2, c2, v3, v2, v1);
                    if (side_border || b <= 0 || b >= S - 1) sm = V(0) + V(1) * v2;
                    const V t = h2 - sm;
                    if constexpr (RS) {
                        if (odd) {   // rows b - 2 .. b around coarse row (b - 1) / 2
                            const int I = (b - 1) / 2;
                            const V f = restrict_value((int)(cn >> 1) - I, e2, e1, t);
                            if (mine && !(cn & 1) && b > r0 && b <= rcoarse)
                                (cr + (int64_t)I * SC)[cn >> 1] =
                                    (side_border || I == 0 || I == SC - 1) ? V(0) : f;
                        }
                        e2 = e1;
                        e1 = t;
                    } else if (mine && b >= r0 && b < r1) {
                        (o0 + (int64_t)b * S)[cn] = v2 + t * d2;
                    }
                }
                x2 = x1;
                x1 = x0;
                v3 = v2;
                v2 = v1;
                h2 = h1;
                h1 = h0;
                d2 = d1;
                d1 = d0;
                c3 = c2;
                c2 = c1;
                n2 = n1;
            }
        }
    }
}

template <typename VT, int PAIR, int WM, bool FUSED>
void stream_launch(dim3 grid, hipStream_t s, const BWork &w, const StreamGeom &g, const BLevel &lv, void *out0,
                   const void *xin, void *xc, int64_t vld_c) {
    using V = typename VecOf<VT>::type;
    hipLaunchKernelGGL((k_b_stream<VT, PAIR, WM, FUSED, kStreamDepth>), grid, dim3(256), 0, s, w, g, lv.vld, lv.kappa,
                       lv.kld, (V *)out0, (const V *)xin, (const V *)lv.rhs, (const V *)lv.dinv, (V *)xc, vld_c);
}

template <typename VT, int WM>
void stream_pair(int pair, dim3 grid, hipStream_t s, const BWork &w, const StreamGeom &g, const BLevel &lv, void *out0,
                 const void *xin, void *xc, int64_t vld_c) {
    if (pair == PAIR_PRE)
        stream_launch<VT, PAIR_PRE, WM, false>(grid, s, w, g, lv, out0, lv.rhs, xc, vld_c);
    else if (xc)
        stream_launch<VT, PAIR_POST, WM, true>(grid, s, w, g, lv, out0, xin, xc, vld_c);
    else
        stream_launch<VT, PAIR_POST, WM, false>(grid, s, w, g, lv, out0, xin, nullptr, 0);
}

// k_b_dir_spmv with weights from the cells, a wavefront marching down each
// tile: row r's p arrives (and is stored), then row r - 1's q = A p from the
// last three rows.  p, q and the tile's p.q are that launch's, the p.q too:
// the tile kernel's thread i holds rows i and i + 16 of the tile, its sixteen
// wavefronts' sums are added as one more wavefront's lanes.  Bound by memory:
// 36 bytes a node, 256 systems of five sizes (17.9 10^6 nodes) 179 -> 127 us
// (5.1 TB/s; 127 to 135 over a solve): no barriers, every wavefront with three
// rows' loads on their way.  That is in an iteration, where the launches before
// leave z and p in the memory-side cache; repeated by itself 151 to 162.
template <typename Z>
__global__ __launch_bounds__(256, 4) void k_b_dir_march(BClassTab tab, BWork w, const SlotScalars *sc) {
    constexpr int T = kPairTileRows, TR = T * kDirNodes, D = 3;   // rows of a tile with its halo, rows in flight
    static_assert(kDirNodes == 2 && kDirRows == TR - 2, "two rows of a tile for each of its partial sums");
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int64_t total = 0;
    for (int c = 0; c < tab.nclass; ++c) total += (int64_t)(w.bounds[c + 1] - w.bounds[c]) * tab.c[c].ntiles;
    const int64_t quads = (total + 3) / 4, share = quads / kXcds, more = quads % kXcds;
    const int64_t xcd = blockIdx.x % kXcds, step = (gridDim.x - 1 - xcd) / kXcds + 1;
    const int64_t lo = xcd * share + (xcd < more ? xcd : more), hi = lo + share + (xcd < more ? 1 : 0);
    for (int64_t quad = lo + blockIdx.x / kXcds; quad < hi; quad += step) {
        int64_t q = quad * 4 + wave;
        if (q >= total) break;
        int c = 0;
        int64_t here;
        while (q >= (here = (int64_t)(w.bounds[c + 1] - w.bounds[c]) * tab.c[c].ntiles)) {
            q -= here;
            ++c;
        }
        const BClassEntry &e = tab.c[c];
        const uint32_t si = (uint32_t)q / (uint32_t)e.ntiles, tile = (uint32_t)q - si * (uint32_t)e.ntiles;
        const uint32_t seg = tile / (uint32_t)e.strips, strip = tile - seg * (uint32_t)e.strips;
        const int64_t g = w.list[w.bounds[c] + (int64_t)si], ls = g - e.first;
        const double beta = sc[g].beta, scale = sc[g].scale;
        const int64_t cur = sc[g].pcur & 1;
        const int S = (int)e.side;
        const int r0 = (int)seg * kDirRows, r1 = min(S, r0 + kDirRows);
        const int c0 = (int)strip * e.tw, c1 = min(S, c0 + e.tw);
        const int col = c0 - 1 + lane;
        const bool mine = lane >= 1 && col < c1;
        const uint32_t cn = (uint32_t)min(max(col, 0), S - 1), cc = (uint32_t)min(max(col, 0), S - 2);
        const bool side_border = cn == 0 || (int)cn == S - 1;
        const double *pold = e.p + ls * e.vld + cur * e.palt;
        double *pnew = e.p + ls * e.vld + (1 - cur) * e.palt, *qs = e.q + ls * e.vld;
        const Z *zs = (const Z *)e.x_top + g * e.vld_top;
        const double *ks = e.kappa + g * e.kld;
        Z pz[D];
        double po[D], pk[D];
        auto load = [&](int r, int i) {
            const int64_t at = (int64_t)min(max(r, 0), min(S - 1, r1)) * S;
            pz[i] = (zs + at)[cn];
            po[i] = (pold + at)[cn];
            pk[i] = (ks + (int64_t)min(max(r - 1, 0), S - 2) * (S - 1))[cc];   // the cells below the row
        };
#pragma unroll
        for (int i = 0; i < D; ++i) load(r0 - 1 + i, i);
        double part[T];
#pragma unroll
        for (int i = 0; i < T; ++i) part[i] = 0.0;
        double x1 = 0.0, x2 = 0.0, k1 = 0.0, across1 = 0.0;
        CellRow<double> c2{};
#pragma unroll
        for (int I = 0; I < TR; ++I) {
            const int r = r0 - 1 + I, i = I % D;
            if (r > r1) continue;   // past a short tile's halo: the same for the whole wavefront
            // ---- row r of p ----
            const double z = (double)pz[i] * scale;
            const double x0 = beta == 0.0 ? z : z + beta * po[i];
            if (mine && r >= r0 && r < r1) (pnew + (int64_t)r * S)[cn] = x0;
            // ---- the weights of row r - 1, as q1_cell_weights forms them ----
            const double k0 = pk[i], kw = from_west(k0), pair0 = kw + k0;
            CellRow<double> c1r;
            NodeRow<double> n1;
            c1r.corner = -div3_rn(k0);
            c1r.across = -0.5 * div3_rn(pair0);
            n1.east = -0.5 * div3_rn(k1 + k0);
            n1.diag = div3_rn(2.0 * ((across1 + kw) + k0));
            k1 = k0;
            across1 = pair0;
            if (I + D < TR) load(r + D, i);
            // ---- row r - 1 of q = A p ----
            if (I >= 2) {
                const int a = r - 1;
                double t = stencil(c2, n1, c1r, x2, x1, x0);
                if (side_border || a == 0 || a == S - 1) t = 0.0 + x1;
                if (mine && a < r1) {
                    (qs + (int64_t)a * S)[cn] = t;
                    part[(I - 1) % T] = part[(I - 1) % T] + x1 * t;
                }
            }
            x2 = x1;
            x1 = x0;
            c2 = c1r;
        }
        double sum = 0.0;
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const double v = wave_sum(part[i]);
            const int vl = __builtin_amdgcn_readfirstlane(__double2loint(v));
            const int vh = __builtin_amdgcn_readfirstlane(__double2hiint(v));
            sum = lane == i ? __hiloint2double(vh, vl) : sum;
        }
        sum = wave_sum(sum);
        if (lane == 0) e.partials[ls * e.pst + tile] = sum;
    }
}

}  // namespace

hipError_t b_dir_march(const BClassTab &tab, const BWork &w, int64_t max_tiles, const SlotScalars *sc, hipStream_t s) {
    const int64_t blocks = (max_tiles + 3) / 4;
    const dim3 grid((uint32_t)(blocks < kStreamBlocks ? blocks : kStreamBlocks));
    if (tab.c[0].top64)
        hipLaunchKernelGGL(k_b_dir_march<double>, grid, dim3(256), 0, s, tab, w, sc);
    else
        hipLaunchKernelGGL(k_b_dir_march<float>, grid, dim3(256), 0, s, tab, w, sc);
    return hipGetLastError();
}

hipError_t b_pair_stream(ValueType vt, int pair, const BLevel &lv, const BWork &w, void *out0, const void *xin,
                         hipStream_t s, int wmode, void *xc, int64_t vld_c) {
    const bool rs = pair == PAIR_PRE;
    StreamGeom g;
    g.side = (int32_t)lv.side;
    const int64_t most = rs ? kStreamWidth - 2 : kStreamWidth;
    g.strips = (int32_t)((lv.side + most - 1) / most);
    g.width = (int32_t)((lv.side + g.strips - 1) / g.strips);
    if (rs) g.width += g.width & 1;
    const int rows[3] = {rs ? 24 : 20, rs ? 12 : 14, rs ? 6 : 8};
    for (int k = 0; k < 3; ++k) {
        g.rows[k] = rows[k];
        g.segs[k] = (int32_t)((lv.side + rows[k] - 1) / rows[k]);
        const int64_t per = (int64_t)g.strips * g.segs[k];
        if (k < 2) g.from[k] = (kStreamFill + per - 1) / per;
    }
    const int64_t units = lv.cap * (int64_t)g.strips * g.segs[2], blocks = (units + 3) / 4;
    if (units < 1) return hipSuccess;
    if (units > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((uint32_t)(blocks < kStreamBlocks ? blocks : kStreamBlocks));
#define STREAM(VT)                                                                    \
    do {                                                                              \
        if (wmode == 3)                                                               \
            stream_pair<VT, 3>(pair, grid, s, w, g, lv, out0, xin, xc, vld_c);  \
        else                                                                          \
            stream_pair<VT, 1>(pair, grid, s, w, g, lv, out0, xin, xc, vld_c);  \
    } while (0)
    if (vt == VT_F32)
        STREAM(float);
    else if (vt == VT_BF16)
        STREAM(bf16);
    else if (vt == VT_F64)
        STREAM(double);
    else
        return hipErrorInvalidValue;
#undef STREAM
    return hipGetLastError();
}

}  // namespace hipx
}  // namespace honei
