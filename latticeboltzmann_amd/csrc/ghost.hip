// Ghost-layer D2Q9 flows: one fused pull step for the reference's Couette,
// Poiseuille, sliding-lid and obstacle-canal scripts
// (simulators/simple_flows/PoiseuilleFlow.py, slidingLid.py;
// simulators/experimantal_flows/obstacle_canal.py).
//
// Those scripts run, per step and on the whole array including its ghost
// layer: [pressure-periodic columns] -> np.roll streaming -> [pressure-periodic
// columns] -> override rules (bounce-back, moving walls, obstacle faces) ->
// moments and collision.  Here one thread owns one node (x, y) and computes
// its post-step populations directly from the previous state:
//
//   P(x, y)  pre-stream value: the state, or on columns 0 and nx-1 the
//            pressure-periodic inlet / outlet value (mode BEFORE_STREAM);
//   G_i(x,y) streamed value P_i(x - cx_i, y - cy_i) (periodic), or on columns
//            0 and nx-1 the inlet / outlet value built from the streamed
//            column (mode AFTER_STREAM);
//   H(x, y)  G with every rule whose target holds (x, y) applied in order; a
//            rule reads G at (x + dx, y + dy) (the host rejects rule tables in
//            which a rule reads what an earlier one writes, so G is what the
//            scripts read too);
//   out      H collided with the scripts' equilibrium.
//
// Interior nodes read their nine populations once (whole rows shifted by at
// most one element, coalesced along y); nodes next to the ghost layer or an
// obstacle read a few more.  Either population layout works; the
// row-interleaved one (the nine channel segments of an x-row adjacent) with
// 512-thread blocks streams about 8 % faster than f[i][k][l] with 256.  Every expression keeps the evaluation order of
// the scripts' numpy code, and the unit is built with -ffp-contract=off, so the
// FP64 and FP32 results are those of the scripts bit for bit.
//
// Runs of several steps (lbm_ghost_run_*) take k_ghost_multi, up to four steps
// per launch on LDS tiles, with the same node code and so the same bits.
//
// Node coordinates in the device functions are unwrapped: a node one period
// outside the grid stands for its periodic image, and only the tests against
// columns 0 / nx-1 and rule targets wrap it.

#include "d2q9_grid.hpp"
#include "lbm_internal.hpp"

#pragma clang fp contract(off)

namespace lbm {
namespace {

constexpr int kGhostBlock = 512;

struct GhostParams {
    int nx, ny;
    int nrules, pbc_mode, flags;
    int reach;  // columns from the inlet / outlet within which its values can matter
    double omega, rho_in, rho_out;
    lbm_ghost_rule rules[LBM_GHOST_MAX_RULES];
};

__device__ __forceinline__ int cx_of(int i) {
    return int(i == 1 || i == 5 || i == 8) - int(i == 3 || i == 6 || i == 7);
}
__device__ __forceinline__ int cy_of(int i) {
    return int(i == 2 || i == 5 || i == 6) - int(i == 4 || i == 7 || i == 8);
}

// rho = sum g (sequential), u = (sum of the + channels - sum of the - channels) / rho
// (PoiseuilleFlow.py:49-53).
template <typename T>
__device__ __forceinline__ void sf_moments(const T g[9], T &rho, T &ux, T &uy) {
    rho = g[0];
#pragma unroll
    for (int i = 1; i < 9; ++i) rho = rho + g[i];
    ux = ((g[1] + g[5]) + g[8]) - ((g[3] + g[6]) + g[7]);
    ux = ux / rho;
    uy = ((g[2] + g[5]) + g[6]) - ((g[4] + g[7]) + g[8]);
    uy = uy / rho;
}

// The scripts' equilibrium (PoiseuilleFlow.py:25-43) with the density factors
// a0 = 2 rho / 9, a1 = rho / 18, a2 = rho / 36 given.
template <typename T>
__device__ __forceinline__ void sf_eq(T a0, T a1, T a2, T ux, T uy, T e[9]) {
    const T p3 = T(3) * (ux + uy);
    const T m3 = T(3) * (ux - uy);
    const T uu = T(3) * (ux * ux + uy * uy);
    const T x6 = T(6) * ux;
    const T y6 = T(6) * uy;
    const T xx9 = T(9) * ux * ux;
    const T yy9 = T(9) * uy * uy;
    const T xy9 = T(9) * ux * uy;
    e[0] = a0 * (T(2) - uu);
    e[1] = a1 * (T(2) + x6 + xx9 - uu);
    e[2] = a1 * (T(2) + y6 + yy9 - uu);
    e[3] = a1 * (T(2) - x6 + xx9 - uu);
    e[4] = a1 * (T(2) - y6 + yy9 - uu);
    e[5] = a2 * (T(1) + p3 + xy9 + uu);
    e[6] = a2 * (T(1) - m3 - xy9 + uu);
    e[7] = a2 * (T(1) - p3 + xy9 + uu);
    e[8] = a2 * (T(1) + m3 - xy9 + uu);
}

// Density factors of an array density (computed in T): 2 rho / 9 and rho / 36
// are rho / 18 times powers of two, so they round to the same digits and one
// division serves all three, unless 2 rho overflows or a quotient is subnormal
// (nodes that cleared walls have drained for thousands of steps) ...
template <typename T>
__device__ __forceinline__ void eq_of_node(T rho, T ux, T uy, T e[9]) {
    constexpr T kLeast = sizeof(T) == 8 ? T(0x1p-1016) : T(0x1p-120), kMost = sizeof(T) == 8 ? T(0x1p1022) : T(0x1p126);
    const T a1 = rho / T(18), m = fabs(rho);
    T a0 = T(4) * a1, a2 = T(0.5) * a1;
    if (__builtin_expect(!(m >= kLeast && m <= kMost), 0)) {
        a0 = T(2) * rho / T(9);
        a2 = rho / T(36);
    }
    sf_eq<T>(a0, a1, a2, ux, uy, e);
}
// ... and of the scalar inlet / outlet density, a Python float: the factors
// are computed in double and then meet the arrays in T.
template <typename T>
__device__ __forceinline__ void eq_of_scalar(double rho, T ux, T uy, T e[9]) {
    sf_eq<T>(T(2.0 * rho / 9.0), T(rho / 18.0), T(rho / 36.0), ux, uy, e);
}

// v[i] and v[i] = x for a wave-uniform channel i, as branches on i, so the
// arrays stay in registers (an indexed access would put them in scratch).
template <typename T>
__device__ __forceinline__ T pick(const T v[9], int i) {
    switch (i) {
    case 1: return v[1];
    case 2: return v[2];
    case 3: return v[3];
    case 4: return v[4];
    case 5: return v[5];
    case 6: return v[6];
    case 7: return v[7];
    case 8: return v[8];
    default: return v[0];
    }
}
template <typename T>
__device__ __forceinline__ void put(T v[9], int i, T x) {
    switch (i) {
    case 0: v[0] = x; break;
    case 1: v[1] = x; break;
    case 2: v[2] = x; break;
    case 3: v[3] = x; break;
    case 4: v[4] = x; break;
    case 5: v[5] = x; break;
    case 6: v[6] = x; break;
    case 7: v[7] = x; break;
    default: v[8] = x; break;
    }
}

// Element (i, x, y) of an nx x ny population array: f[x][i][y] (Rows) or
// f[i][x][y]; the layout is a template parameter so the index folds.
template <bool Rows>
__device__ __forceinline__ int64_t index_of(int i, int x, int y, int nx, int ny) {
    return Rows ? (int64_t(x) * 9 + i) * ny + y : (int64_t(i) * nx + x) * ny + y;
}

// The state in memory; (X, Y) at most one period outside the grid.
template <typename T, bool Rows>
struct Grid {
    using value_type = T;
    const T *s;
    int nx, ny;
    __device__ __forceinline__ T at(int i, int X, int Y) const {
        return s[index_of<Rows>(i, wrap1(X, nx), wrap1(Y, ny), nx, ny)];
    }
};

// A state held in an LDS tile: planes of NA values, rows PITCH wide, whose
// first node is (xlo, ylo).
template <typename T, int PITCH, int NA>
struct Tile {
    using value_type = T;
    const T *s;
    int xlo, ylo;
    __device__ __forceinline__ T at(int i, int X, int Y) const {
        return s[i * NA + (X - xlo) * PITCH + (Y - ylo)];
    }
};

// Inlet (x == 0) or outlet (x == nx-1) populations from the nine values g of
// the opposite interior column (nx-2 or 1): f_eq(rho_b, u) + (g - f_eq(g)),
// summed as eq_b + (g - eq) (BEFORE) or (eq_b + g) - eq (AFTER).
template <typename T, bool After>
__device__ __forceinline__ void pbc_values(const T g[9], double rho_b, T out[9]) {
    T rho, ux, uy, e[9], eb[9];
    sf_moments<T>(g, rho, ux, uy);
    eq_of_node<T>(rho, ux, uy, e);
    eq_of_scalar<T>(rho_b, ux, uy, eb);
#pragma unroll
    for (int i = 0; i < 9; ++i) out[i] = After ? (eb[i] + g[i]) - e[i] : eb[i] + (g[i] - e[i]);
}

// Whether column X (unwrapped) is the inlet or the outlet; then the column whose
// values it is built from (nx-2 or 1) and its density.
__device__ __forceinline__ bool pbc_column(const GhostParams &p, int X, int &Xs, double &rho_b) {
    const int x = wrap1(X, p.nx);
    if (x != 0 && x != p.nx - 1) return false;
    Xs = x == 0 ? X - 2 : X + 2;
    rho_b = x == 0 ? p.rho_in : p.rho_out;
    return true;
}

// Streamed value of channel i at (X, Y), periodic in x and y: the pre-stream
// value at (X - cx_i, Y - cy_i), which on the inlet and outlet columns
// (BEFORE) is built from the opposite column.
template <bool Pbc, typename Gr, typename T = typename Gr::value_type>
__device__ __forceinline__ T pull(const Gr &g, const GhostParams &p, int i, int X, int Y) {
    const int Xp = X - cx_of(i), Yp = Y - cy_of(i);
    int Xs;
    double rho_b;
    if (Pbc && p.pbc_mode == LBM_PBC_BEFORE_STREAM && pbc_column(p, Xp, Xs, rho_b)) {
        T v[9], o[9];
#pragma unroll
        for (int j = 0; j < 9; ++j) v[j] = g.at(j, Xs, Yp);
        pbc_values<T, false>(v, rho_b, o);
        return pick(o, i);
    }
    return g.at(i, Xp, Yp);
}

// The nine streamed values at (X, Y) with the after-stream inlet / outlet
// columns: on those the opposite column's nine values are pulled once and
// make all nine channels.
template <bool Pbc, typename Gr, typename T = typename Gr::value_type>
__device__ __forceinline__ void load_g9(const Gr &g, const GhostParams &p, int X, int Y, T h[9]) {
    int Xs = X;
    double rho_b = 0.0;
    const bool col = Pbc && p.pbc_mode == LBM_PBC_AFTER_STREAM && pbc_column(p, X, Xs, rho_b);
#pragma unroll
    for (int j = 0; j < 9; ++j) h[j] = g.at(j, Xs - cx_of(j), Y - cy_of(j));
    if (Pbc && p.pbc_mode == LBM_PBC_BEFORE_STREAM) {
        // the three channels that come from each inlet or outlet column; unrolled,
        // so that their loads are in flight together (a node of column 0 pulls six:
        // 102 x 52 FP64 10.4 us a step one after another, 8.8 so)
#pragma unroll
        for (int c = -1; c <= 1; ++c) {
            int Xo;
            if (!pbc_column(p, X - c, Xo, rho_b)) continue;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                // channels of cx = -1: 3 6 7, 0: 0 2 4, 1: 1 5 8
                const int j = ((c < 0 ? 0x763 : (c == 0 ? 0x420 : 0x851)) >> (4 * k)) & 15;
                put(h, j, pull<Pbc>(g, p, j, X, Y));
            }
        }
    }
    if (col) {
        T v[9];
#pragma unroll
        for (int j = 0; j < 9; ++j) v[j] = h[j];
        pbc_values<T, true>(v, rho_b, h);
    }
}

// One of them.  Pbc: the flow may have an inlet and outlet.
template <bool Pbc, typename Gr, typename T = typename Gr::value_type>
__device__ __forceinline__ T load_g(const Gr &g, const GhostParams &p, int i, int X, int Y) {
    int Xs;
    double rho_b;
    if (Pbc && p.pbc_mode == LBM_PBC_AFTER_STREAM && pbc_column(p, X, Xs, rho_b)) {
        T v[9], o[9];
#pragma unroll
        for (int j = 0; j < 9; ++j) v[j] = g.at(j, Xs - cx_of(j), Y - cy_of(j));
        pbc_values<T, true>(v, rho_b, o);
        return pick(o, i);
    }
    return pull<Pbc>(g, p, i, X, Y);
}

template <bool Pbc, typename Gr, typename T = typename Gr::value_type>
__device__ __forceinline__ T rule_value(const Gr &g, const GhostParams &p, const lbm_ghost_rule &r,
                                        int X, int Y) {
    if (r.kind == LBM_RULE_ZERO) return T(0);
    const int Xs = X + r.dx, Ys = Y + r.dy;
    T rw = T(0);
    if (r.kind == LBM_RULE_LID_RHO) {
        // 2.0 * (g2 + g5 + g6) + g0 + g1 + g3 at the source node
        // (slidingLid.py:86-87); all loads in flight at once, unless the inlet's
        // and outlet's arithmetic behind each would make seven copies of it
        constexpr int ch[6] = {2, 5, 6, 0, 1, 3};
        T c[6];
        if constexpr (Pbc) {
#pragma unroll 1
            for (int k = 0; k < 6; ++k) {
                const T v = load_g<Pbc>(g, p, (0x310652 >> (4 * k)) & 15, Xs, Ys);
                rw = k == 0 ? v : rw + v;
                if (k == 2) rw = T(2) * rw;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) c[k] = load_g<Pbc>(g, p, ch[k], Xs, Ys);
            rw = T(2) * ((c[0] + c[1]) + c[2]);
            rw = ((rw + c[3]) + c[4]) + c[5];
        }
    }
    const T v = load_g<Pbc>(g, p, r.src_ch, Xs, Ys);
    if (r.kind == LBM_RULE_LID) return v + T(r.coef);
    if (r.kind == LBM_RULE_LID_RHO) return v + T(r.coef) * rw;
    return v;
}

// The nine values of node (x, y) after streaming and the rules (ascending, the
// scripts' order).  x is the same for all lanes, so most rules end at a scalar
// branch.
template <bool Pbc, typename Gr, typename T = typename Gr::value_type>
__device__ __forceinline__ void node_values(const Gr &g, const GhostParams &p, int x, int y, T h[9]) {
    load_g9<Pbc>(g, p, x, y, h);
    for (int r = 0; r < p.nrules; ++r) {
        const lbm_ghost_rule &rule = p.rules[r];
        if (unsigned(x - rule.x0) < unsigned(rule.x1 - rule.x0) &&
            unsigned(y - rule.y0) < unsigned(rule.y1 - rule.y0))
            put(h, rule.ch, rule_value<Pbc>(g, p, rule, x, y));
    }
}

// BGK collision with the scripts' equilibrium, in place: h -= omega (h - f_eq).
template <typename T>
__device__ __forceinline__ void sf_collide(T h[9], T om, T &rho, T &ux, T &uy) {
    T e[9];
    sf_moments<T>(h, rho, ux, uy);
    eq_of_node<T>(rho, ux, uy, e);
#pragma unroll
    for (int i = 0; i < 9; ++i) h[i] = h[i] - om * (h[i] - e[i]);
}

template <typename T, bool Rows, bool Pbc>
__global__ __launch_bounds__(kGhostBlock) void k_ghost_step(const T *__restrict__ src, T *__restrict__ dst,
                                                       const GhostParams p, T *__restrict__ rho_out,
                                                       T *__restrict__ ux_out, T *__restrict__ uy_out) {
    // columns near the inlet and outlet take longest, so their blocks come first
    // (700^2 FP64, built before streaming, 22.9 us a step with them last, 17.2 so)
    const int shifted = Pbc ? int(blockIdx.y) - p.reach : int(blockIdx.y);
    const int x = shifted < 0 ? shifted + p.nx : shifted;
    const int y = blockIdx.x * kGhostBlock + threadIdx.x;
    if (y >= p.ny) return;
    const Grid<T, Rows> g{src, p.nx, p.ny};
    T h[9];
    if (p.flags & LBM_GHOST_COLLIDE_ONLY) {
#pragma unroll
        for (int i = 0; i < 9; ++i) h[i] = g.at(i, x, y);
    } else if (Pbc && (x < p.reach || x >= p.nx - p.reach)) {
        node_values<true>(g, p, x, y, h);
    } else {
        node_values<false>(g, p, x, y, h);
    }
    T rho = T(0), ux = T(0), uy = T(0);
    if (!(p.flags & LBM_GHOST_NO_COLLIDE)) sf_collide<T>(h, T(p.omega), rho, ux, uy);
#pragma unroll
    for (int i = 0; i < 9; ++i) dst[index_of<Rows>(i, x, y, p.nx, p.ny)] = h[i];
    if (rho_out && !(p.flags & LBM_GHOST_NO_COLLIDE)) {
        const int64_t node = int64_t(x) * p.ny + y;
        rho_out[node] = rho;
        ux_out[node] = ux;
        uy_out[node] = uy;
    }
}

// ---------------------------------------------------------------------------
// K steps per launch (2 <= K <= 4), src -> dst, on TR x TC tiles in LDS.
//
// Step j is computed on the tile widened by what the later steps read.  For
// pulls that is one node a step; the inlet / outlet columns (built from three
// columns on the other side) and rules whose source lies further off read
// more, at the columns and rows listed in GhostPlan, so the extents follow
// from a short recurrence per tile.  Step 1 reads memory, the others the LDS
// tile in place (all pulls of a step into registers, a barrier, then the
// results over the old values), the last one writes dst: memory sees each
// population about once per K steps instead of once a step.
//
// Rules, inlet and outlet: each streamed value is pulled by one node, so
// overriding G_ch at (x, y) is the same as overwriting the value that the pull
// reads, P_ch at (x - cx, y - cy), before the pulls.  A tile that meets any
// therefore runs, before the pulls of a step, one item per (rule, target node)
// and per inlet / outlet node, spread over the threads: all items read the
// values as they are, then (after a barrier) write.  The pulls themselves are
// the same bare code everywhere.  (With the rules applied to each node's
// registers in a loop, as the single step does, the serial scalar work of a
// dozen rules per wave and step made a 102 x 52 canal take 37 us per four
// steps.)  In step 1 the items overwrite the pulled values instead.
constexpr int kGhostMaxK = 4;
constexpr int kGhostMaxWide = 16;

// Columns (axis 0) / rows (axis 1), periodic images included, whose nodes read
// state at offsets lo .. hi beyond -1 .. 1 along that axis; over[r]: later
// rules with the same target channel that share target nodes with rule r.
struct GhostPlan {
    int n[2];
    int at[2][kGhostMaxWide], lo[2][kGhostMaxWide], hi[2][kGhostMaxWide];
    uint32_t over[LBM_GHOST_MAX_RULES];
};

// n / w for 0 <= n < 2^14, 1 <= w <= 64, given 1.0f / w.
__device__ __forceinline__ int row_of(int n, float inv_w) { return int((float(n) + 0.5f) * inv_w); }

// Region of a step, columns [xa, xb) and rows [ya, yb), unwrapped.
struct Region {
    int xa, xb, ya, yb;
    __device__ __forceinline__ bool has(int X, int Y, int margin = 0) const {
        return X >= xa - margin && X < xb + margin && Y >= ya - margin && Y < yb + margin;
    }
};

// The items of a thread, found once per tile.
struct GhostItems {
    int rule, X, Y;  // rule item; rule < 0: none, or a later rule overrides it
    int PX, PY;      // inlet / outlet node
    bool pbc;
};

// A thread's items for the step on region `rg`: their values from the state g
// and, once every item has read, the writes over the values that the pulls
// read (Pulled: over the pulled values).  The rules come after the inlet and
// outlet, as in the scripts.
template <typename T, int PITCH, int NA, bool Pulled, bool Pbc, typename Gr>
__device__ __forceinline__ void item_pass(const Gr &g, T *buf, int xlo, int ylo, const GhostParams &p,
                                          const lbm_ghost_rule *rules, const GhostItems &it,
                                          const Region &rg) {
    const bool rule = it.rule >= 0 && rg.has(it.X, it.Y);
    T val = T(0);
    if (rule) val = rule_value<Pbc>(g, p, rules[it.rule], it.X, it.Y);
    if constexpr (Pbc) {
        const bool before = p.pbc_mode == LBM_PBC_BEFORE_STREAM;
        const bool node = it.pbc && rg.has(it.PX, it.PY, before ? 1 : 0);
        T v[9], pv[9];
        if (node) {
            int Xs;
            double rho_b = 0.0;
            (void)pbc_column(p, it.PX, Xs, rho_b);
#pragma unroll
            for (int j = 0; j < 9; ++j)
                v[j] = before ? g.at(j, Xs, it.PY) : g.at(j, Xs - cx_of(j), it.PY - cy_of(j));
            if (before) pbc_values<T, false>(v, rho_b, pv);
            else pbc_values<T, true>(v, rho_b, pv);
        }
        __syncthreads();
        if (node) {
#pragma unroll
            for (int j = 0; j < 9; ++j) {
                // the node that the value reaches (after streaming)
                const int X = before ? it.PX + cx_of(j) : it.PX, Y = before ? it.PY + cy_of(j) : it.PY;
                if (!rg.has(X, Y)) continue;
                const int px = Pulled ? X : X - cx_of(j), py = Pulled ? Y : Y - cy_of(j);
                buf[j * NA + (px - xlo) * PITCH + (py - ylo)] = pv[j];
            }
        }
    }
    __syncthreads();
    if (rule) {
        const int ch = rules[it.rule].ch;
        const int px = Pulled ? it.X : it.X - cx_of(ch), py = Pulled ? it.Y : it.Y - cy_of(ch);
        buf[ch * NA + (px - xlo) * PITCH + (py - ylo)] = val;
    }
    __syncthreads();
}

// Length of and positions in the parts of [c0, c1) and its images in [a, b).
__device__ __forceinline__ int image_count(int c0, int c1, int n, int a, int b) {
    int t = 0;
#pragma unroll
    for (int s = -1; s <= 1; ++s) t += max(0, min(c1 + s * n, b) - max(c0 + s * n, a));
    return t;
}
__device__ __forceinline__ int image_at(int c0, int c1, int n, int a, int b, int i) {
    int at = a;
#pragma unroll
    for (int s = -1; s <= 1; ++s) {
        const int l = max(c0 + s * n, a), len = max(0, min(c1 + s * n, b) - l);
        if (i >= 0 && i < len) at = l + i;
        i -= len;
    }
    return at;
}

// The K steps of one tile, given the regions.  Items: the tile has items or its
// region reaches the border; the other tiles run the bare pulls.  Two copies of
// the code, so that the items' registers do not weigh on the other tiles.
template <typename T, bool Rows, int BS, int PITCH, int NA, bool Items, bool Pbc>
__device__ __forceinline__ void ghost_tile(const T *__restrict__ src, T *__restrict__ dst, const GhostParams &p,
                                           int K, const Region &rg, const Region *ext, const GhostItems &it,
                                           bool items, const lbm_ghost_rule *rules, T *buf,
                                           T *__restrict__ rho_out, T *__restrict__ ux_out,
                                           T *__restrict__ uy_out) {
    const int t = int(threadIdx.x), nx = p.nx, ny = p.ny, xlo = rg.xa, ylo = rg.ya;
    const T om = T(p.omega);
    {
        const int w = rg.yb - rg.ya, N = (rg.xb - rg.xa) * w;
        const float inv = 1.0f / float(w);
        if constexpr (!Items) {
            // a thread with two nodes issues both nodes' loads before either
            // collides
            for (int n0 = t; n0 < N; n0 += 2 * BS) {
                T h[2][9];
                int m[2];
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const int n = min(n0 + v * BS, N - 1);
                    const int r = row_of(n, inv), c = n - r * w;
                    m[v] = r * PITCH + c;
                    if (n0 + v * BS < N) {
                        const T *s = src + index_of<Rows>(0, xlo + r, ylo + c, nx, ny);
#pragma unroll
                        for (int i = 0; i < 9; ++i)
                            h[v][i] = s[index_of<Rows>(i, -cx_of(i), -cy_of(i), nx, ny)];
                    }
                }
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    if (n0 + v * BS >= N) continue;
                    T rho, ux, uy;
                    sf_collide<T>(h[v], om, rho, ux, uy);
#pragma unroll
                    for (int i = 0; i < 9; ++i) buf[i * NA + m[v]] = h[v][i];
                }
            }
        } else {
            const Grid<T, Rows> g{src, nx, ny};
            for (int n = t; n < N; n += BS) {
                const int r = row_of(n, inv), c = n - r * w;
                T h[9];
#pragma unroll
                for (int i = 0; i < 9; ++i) h[i] = g.at(i, xlo + r - cx_of(i), ylo + c - cy_of(i));
#pragma unroll
                for (int i = 0; i < 9; ++i) buf[i * NA + r * PITCH + c] = h[i];
            }
            if (items) {
                item_pass<T, PITCH, NA, true, Pbc>(g, buf, xlo, ylo, p, rules, it, rg);
            }
            for (int n = t; n < N; n += BS) {
                const int r = row_of(n, inv), m = r * PITCH + (n - r * w);
                T h[9], rho, ux, uy;
#pragma unroll
                for (int i = 0; i < 9; ++i) h[i] = buf[i * NA + m];
                sf_collide<T>(h, om, rho, ux, uy);
#pragma unroll
                for (int i = 0; i < 9; ++i) buf[i * NA + m] = h[i];
            }
        }
    }
    __syncthreads();

    const Tile<T, PITCH, NA> g{buf, xlo, ylo};
    // nodes of a thread in an LDS step, whose region is two narrower than the tile
    constexpr int VM = ((NA / PITCH - 2) * (PITCH - 2) + BS - 1) / BS;
    for (int d = K - 2; d > 0; --d) {       // d steps follow this one
        const Region w = ext[d];
        if (Items && items) {
            item_pass<T, PITCH, NA, false, Pbc>(g, buf, xlo, ylo, p, rules, it, w);
        }
        const int wy = w.yb - w.ya, N = (w.xb - w.xa) * wy;
        const float inv = 1.0f / float(wy);
        T h[VM][9];
        int m[VM];
#pragma unroll
        for (int v = 0; v < VM; ++v) {
            const int n = t + v * BS;
            const int r = row_of(n, inv), c = n - r * wy;
            m[v] = (w.xa + r - xlo) * PITCH + (w.ya + c - ylo);
            if (n >= N) continue;
#pragma unroll
            for (int i = 0; i < 9; ++i) h[v][i] = buf[i * NA + m[v] - cx_of(i) * PITCH - cy_of(i)];
        }
        __syncthreads();  // every read of the old values is done
#pragma unroll
        for (int v = 0; v < VM; ++v) {
            if (t + v * BS >= N) continue;
            T rho, ux, uy;
            sf_collide<T>(h[v], om, rho, ux, uy);
#pragma unroll
            for (int i = 0; i < 9; ++i) buf[i * NA + m[v]] = h[v][i];
        }
        __syncthreads();
    }

    const Region w = ext[0];
    if (Items && items) {
        item_pass<T, PITCH, NA, false, Pbc>(g, buf, xlo, ylo, p, rules, it, w);
    }
    const int wy = w.yb - w.ya, N = (w.xb - w.xa) * wy;
    const float inv = 1.0f / float(wy);
    for (int n = t; n < N; n += BS) {
        const int r = row_of(n, inv), X = w.xa + r, Y = w.ya + (n - r * wy);
        const int m = (X - xlo) * PITCH + (Y - ylo);
        T h[9], rho, ux, uy;
#pragma unroll
        for (int i = 0; i < 9; ++i) h[i] = buf[i * NA + m - cx_of(i) * PITCH - cy_of(i)];
        sf_collide<T>(h, om, rho, ux, uy);
        // the next launch reads this, no other tile of this one: leave the
        // caches to the state that neighbouring tiles still read
        T *o = dst + index_of<Rows>(0, X, Y, nx, ny);
#pragma unroll
        for (int i = 0; i < 9; ++i) st<true>(o + index_of<Rows>(i, 0, 0, nx, ny), h[i]);
        if (rho_out) {
            const int64_t node = int64_t(X) * ny + Y;
            rho_out[node] = rho;
            ux_out[node] = ux;
            uy_out[node] = uy;
        }
    }
}

// PITCH x (NA / PITCH) nodes: the widest region of step 1 that fits the tile.
// The host has checked that every tile's region does, that it is no wider than
// the grid, and that a tile has at most BS rule items.
template <typename T, bool Rows, bool Pbc, int TR, int TC, int BS, int PITCH, int NA, int WPE>
__global__ __launch_bounds__(BS, WPE) void k_ghost_multi(const T *__restrict__ src, T *__restrict__ dst,
                                                         const GhostParams p, const GhostPlan plan,
                                                         int K, int ntc, int ntiles,
                                                         T *__restrict__ rho_out,
                                                         T *__restrict__ ux_out,
                                                         T *__restrict__ uy_out) {
    __shared__ T buf[9 * NA];
    __shared__ lbm_ghost_rule rules[LBM_GHOST_MAX_RULES];
    __shared__ int first[LBM_GHOST_MAX_RULES + 1];  // first item of each rule
    __shared__ Region ext[kGhostMaxK];              // ext[d]: d steps follow
    const int tile = xcd_tile(ntiles);
    if (tile >= ntiles) return;  // whole block: before any barrier
    const int t = int(threadIdx.x), lane = t & 63;
    const int nx = p.nx, ny = p.ny;
    const int tx = (tile / ntc) * TR, ty = (tile % ntc) * TC;

    // plan entries and rules once, side by side: the arguments lie far away
    int at = 0, lo = 0, hi = 0;
    if (lane < 2 * kGhostMaxWide) at = plan.at[0][lane], lo = plan.lo[0][lane], hi = plan.hi[0][lane];
    constexpr int kRuleWords = int(sizeof(lbm_ghost_rule) / sizeof(int));
    int mine[kRuleWords];  // rule `lane`
    {
        const int *q = reinterpret_cast<const int *>(&p.rules[lane & (LBM_GHOST_MAX_RULES - 1)]);
#pragma unroll
        for (int i = 0; i < kRuleWords; ++i) mine[i] = q[i];
    }

    Region rg{tx, min(tx + TR, nx), ty, min(ty + TC, ny)};
    if (t == 0) ext[0] = rg;
#pragma unroll
    for (int d = 1; d < kGhostMaxK; ++d) {
        if (d >= K) break;
        Region w{rg.xa - 1, rg.xb + 1, rg.ya - 1, rg.yb + 1};
        for (int e = 0; e < plan.n[0]; ++e) {
            const int c = __builtin_amdgcn_readlane(at, e);
            if (c < rg.xa || c >= rg.xb) continue;
            w.xa = min(w.xa, c + __builtin_amdgcn_readlane(lo, e));
            w.xb = max(w.xb, c + __builtin_amdgcn_readlane(hi, e) + 1);
        }
        for (int e = 0; e < plan.n[1]; ++e) {
            const int c = __builtin_amdgcn_readlane(at, kGhostMaxWide + e);
            if (c < rg.ya || c >= rg.yb) continue;
            w.ya = min(w.ya, c + __builtin_amdgcn_readlane(lo, kGhostMaxWide + e));
            w.yb = max(w.yb, c + __builtin_amdgcn_readlane(hi, kGhostMaxWide + e) + 1);
        }
        rg = w;
        if (t == 0) ext[d] = rg;
    }

    // items of rule `lane` in the region
    const int nxi = image_count(mine[0], mine[1], nx, rg.xa, rg.xb);
    const int nyi = image_count(mine[2], mine[3], ny, rg.ya, rg.yb);
    const int cnt = lane < p.nrules ? nxi * nyi : 0;
    const bool any_rule = __ballot(cnt > 0) != 0;
    // the region's pulls reach the border columns or rows
    const bool border = rg.xa < 2 || rg.xb > nx - 2 || rg.ya < 1 || rg.yb > ny - 1;
    const bool items = any_rule || (Pbc && border);
    GhostItems it{-1, 0, 0, 0, 0, false};
    if (items) {
        int sum = cnt;  // inclusive sums over the lanes
#pragma unroll
        for (int o = 1; o < LBM_GHOST_MAX_RULES; o <<= 1) {
            const int v = __shfl_up(sum, o);
            if (lane >= o) sum += v;
        }
        if (t < LBM_GHOST_MAX_RULES) {
            int *q = reinterpret_cast<int *>(&rules[t]);
#pragma unroll
            for (int i = 0; i < kRuleWords; ++i) q[i] = mine[i];
            first[t + 1] = sum;
            if (t == 0) first[0] = 0;
        }
        __syncthreads();
        if (t < first[LBM_GHOST_MAX_RULES]) {
            int r = 0;  // the last rule whose first item is not past t
#pragma unroll
            for (int o = LBM_GHOST_MAX_RULES / 2; o > 0; o >>= 1)
                if (first[r + o] <= t) r += o;
            const lbm_ghost_rule &q = rules[r];
            const int n = image_count(q.y0, q.y1, ny, rg.ya, rg.yb);
            const int i = (t - first[r]) / n, j = (t - first[r]) - i * n;
            it.X = image_at(q.x0, q.x1, nx, rg.xa, rg.xb, i);
            it.Y = image_at(q.y0, q.y1, ny, rg.ya, rg.yb, j);
            it.rule = r;
            const int x = wrap1(it.X, nx), y = wrap1(it.Y, ny);
            for (uint32_t m = plan.over[r]; m; m &= m - 1) {
                const lbm_ghost_rule &b = rules[__builtin_ctz(m)];
                if (x >= b.x0 && x < b.x1 && y >= b.y0 && y < b.y1) it.rule = -1;
            }
        }
        if constexpr (Pbc) {  // from the last thread down
            const int h = rg.yb - rg.ya + 2, u = BS - 1 - t, c = u / h;
            it.PX = c == 0 ? -1 : (c == 1 ? 0 : (c == 2 ? nx - 1 : nx));
            it.PY = rg.ya - 1 + (u - c * h);
            it.pbc = c < 4 && rg.has(it.PX, it.PY, 1);
        }
    }
    __syncthreads();  // ext
    if (items || border)
        ghost_tile<T, Rows, BS, PITCH, NA, true, Pbc>(src, dst, p, K, rg, ext, it, items, rules, buf, rho_out,
                                                      ux_out, uy_out);
    else
        ghost_tile<T, Rows, BS, PITCH, NA, false, Pbc>(src, dst, p, K, rg, ext, it, items, rules, buf, rho_out,
                                                       ux_out, uy_out);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_ghost_equilibrium(const T *__restrict__ rho,
                                                              const T *__restrict__ ux,
                                                              const T *__restrict__ uy,
                                                              T *__restrict__ f, int64_t n) {
    const int64_t k = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (k >= n) return;
    T e[9];
    eq_of_node<T>(rho[k], ux[k], uy[k], e);
#pragma unroll
    for (int i = 0; i < 9; ++i) f[int64_t(i) * n + k] = e[i];
}

template <typename T>
int ghost_equilibrium(const T *rho, const T *ux, const T *uy, T *f, int64_t n, void *stream) {
    if (!rho || !ux || !uy || !f) return LBM_E_NULL;
    if (n <= 0 || n > (int64_t(1) << 40)) return LBM_E_SIZE;
    const int64_t fb = 9 * n * int64_t(sizeof(T)), mb = n * int64_t(sizeof(T));
    if (overlaps(rho, mb, f, fb) || overlaps(ux, mb, f, fb) || overlaps(uy, mb, f, fb))
        return LBM_E_ALIAS;
    const int64_t blocks = (n + kBlock - 1) / kBlock;
    if (blocks > INT32_MAX) return LBM_E_SIZE;
    hipLaunchKernelGGL(k_ghost_equilibrium<T>, dim3(unsigned(blocks)), dim3(kBlock), 0,
                       as_stream(stream), rho, ux, uy, f, n);
    return launch_status();
}

bool rect_hits(int ax0, int ax1, int ay0, int ay1, int bx0, int bx1, int by0, int by1) {
    return ax0 < bx1 && bx0 < ax1 && ay0 < by1 && by0 < ay1;
}

// Validates the rule table: ranges inside the grid, sources inside the grid,
// and no rule reading a population an earlier rule writes.
int check_rules(const lbm_ghost_rule *rules, int nrules, int nx, int ny) {
    for (int r = 0; r < nrules; ++r) {
        const lbm_ghost_rule &a = rules[r];
        if (a.kind < LBM_RULE_COPY || a.kind > LBM_RULE_ZERO) return LBM_E_ARG;
        if (a.ch < 0 || a.ch > 8) return LBM_E_ARG;
        if (a.x0 < 0 || a.x1 > nx || a.x0 >= a.x1 || a.y0 < 0 || a.y1 > ny || a.y0 >= a.y1)
            return LBM_E_ARG;
        if (a.kind == LBM_RULE_ZERO) continue;
        if (a.src_ch < 0 || a.src_ch > 8) return LBM_E_ARG;
        if (a.x0 + a.dx < 0 || a.x1 + a.dx > nx || a.y0 + a.dy < 0 || a.y1 + a.dy > ny)
            return LBM_E_ARG;
        if ((a.kind == LBM_RULE_LID || a.kind == LBM_RULE_LID_RHO) && !(a.coef == a.coef))
            return LBM_E_ARG;
        const int sx0 = a.x0 + a.dx, sx1 = a.x1 + a.dx, sy0 = a.y0 + a.dy, sy1 = a.y1 + a.dy;
        for (int q = 0; q < r; ++q) {
            const lbm_ghost_rule &b = rules[q];
            if (!rect_hits(sx0, sx1, sy0, sy1, b.x0, b.x1, b.y0, b.y1)) continue;
            if (b.ch == a.src_ch) return LBM_E_ARG;
            if (a.kind == LBM_RULE_LID_RHO &&
                (b.ch == 0 || b.ch == 1 || b.ch == 2 || b.ch == 3 || b.ch == 5 || b.ch == 6))
                return LBM_E_ARG;
        }
    }
    return LBM_OK;
}

// Checks the arguments of a step and fills its parameters.
template <typename T>
int ghost_params(const T *src, const T *dst, int64_t nx, int64_t ny, int layout, double omega,
                 const lbm_ghost_rule *rules, int nrules, const lbm_ghost_pbc *pbc, int flags,
                 const T *rho, const T *ux, const T *uy, GhostParams &p) {
    if (!src || !dst) return LBM_E_NULL;
    if (nx < 3 || ny < 3 || nx > 65535 || ny > (int64_t(1) << 30) || nx * ny > INT32_MAX)
        return LBM_E_SIZE;
    if (!valid_layout(layout)) return LBM_E_ARG;
    if (nrules < 0 || nrules > LBM_GHOST_MAX_RULES || (nrules > 0 && !rules)) return LBM_E_ARG;
    if ((flags & ~(LBM_GHOST_NO_COLLIDE | LBM_GHOST_COLLIDE_ONLY)) ||
        flags == (LBM_GHOST_NO_COLLIDE | LBM_GHOST_COLLIDE_ONLY))
        return LBM_E_ARG;
    if (!(omega == omega)) return LBM_E_ARG;
    const bool any = rho || ux || uy;
    if (any && !(rho && ux && uy)) return LBM_E_NULL;
    const int64_t bytes = 9 * nx * ny * int64_t(sizeof(T));
    if (overlaps(src, bytes, dst, bytes)) return LBM_E_ALIAS;
    if (any) {
        const int64_t mb = nx * ny * int64_t(sizeof(T));
        if (overlaps(rho, mb, dst, bytes) || overlaps(ux, mb, dst, bytes) ||
            overlaps(uy, mb, dst, bytes) || overlaps(rho, mb, src, bytes) ||
            overlaps(ux, mb, src, bytes) || overlaps(uy, mb, src, bytes))
            return LBM_E_ALIAS;
    }
    p = GhostParams{};
    p.nx = int(nx);
    p.ny = int(ny);
    p.flags = flags;
    p.omega = omega;
    p.pbc_mode = LBM_PBC_NONE;
    if (pbc) {
        if (pbc->mode < LBM_PBC_NONE || pbc->mode > LBM_PBC_AFTER_STREAM) return LBM_E_ARG;
        if (!(pbc->rho_in == pbc->rho_in) || !(pbc->rho_out == pbc->rho_out)) return LBM_E_ARG;
        p.pbc_mode = pbc->mode;
        p.rho_in = pbc->rho_in;
        p.rho_out = pbc->rho_out;
    }
    if (flags & LBM_GHOST_COLLIDE_ONLY) {
        p.nrules = 0;
        p.pbc_mode = LBM_PBC_NONE;
    } else {
        const int rc = check_rules(rules, nrules, p.nx, p.ny);
        if (rc) return rc;
        p.nrules = nrules;
        p.reach = 2;  // pulls from columns 0 and nx-1 reach 1 and nx-2
        for (int r = 0; r < nrules; ++r) {
            p.rules[r] = rules[r];
            const int d = rules[r].dx < 0 ? -rules[r].dx : rules[r].dx;
            if (d + 2 > p.reach) p.reach = d + 2;  // sources at x + dx, pulls from there
        }
        if (p.reach > p.nx) p.reach = p.nx;  // k_ghost_step counts its columns from -reach
    }
    return LBM_OK;
}

template <typename T>
int launch_ghost_step(const T *src, T *dst, int layout, const GhostParams &p, T *rho, T *ux, T *uy,
                      hipStream_t s) {
    const dim3 grid(unsigned((p.ny + kGhostBlock - 1) / kGhostBlock), unsigned(p.nx));
    // HBM-bound in FP64, three blocks a CU instead of four read fewer rows at a time
    // (the LDS they reserve is not used).  us a step of the sliding lid, four / three:
    // 1500 x 4000 162 / 154, 4098^2 467 / 448, 6000 x 3000 478 / 462, 6000^2 996 / 973;
    // but 2500 x 2001, half in the last-level cache, 143 / 145, 8192^2 1712 / 1752, short
    // rows (16000 x 1000) 433 / 450, FP32 3000 x 6000 246 / 244, 4000^2 210 / 247.
    // The kernel with inlet and outlet has registers for two blocks anyway.
    const int64_t nodes = int64_t(p.nx) * p.ny;
    const bool three = sizeof(T) == 8 && p.pbc_mode == LBM_PBC_NONE && p.ny >= 1500 &&
                       nodes >= 5500000 && nodes <= 40000000;
    const unsigned lds = three ? 52 * 1024 : 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kGhostBlock), lds, s, src, dst, p, rho, ux, uy);
    };
    const bool rows = layout == LBM_LAYOUT_ROWS;
    if (p.pbc_mode == LBM_PBC_NONE) {
        if (rows) launch(k_ghost_step<T, true, false>);
        else launch(k_ghost_step<T, false, false>);
    } else {
        if (rows) launch(k_ghost_step<T, true, true>);
        else launch(k_ghost_step<T, false, true>);
    }
    return launch_status();
}

template <typename T>
int ghost_step(const T *src, T *dst, int64_t nx, int64_t ny, int layout, double omega,
               const lbm_ghost_rule *rules, int nrules, const lbm_ghost_pbc *pbc, int flags, T *rho,
               T *ux, T *uy, void *stream) {
    GhostParams p;
    const int rc = ghost_params<T>(src, dst, nx, ny, layout, omega, rules, nrules, pbc, flags, rho,
                                   ux, uy, p);
    if (rc) return rc;
    return launch_ghost_step<T>(src, dst, layout, p, rho, ux, uy, as_stream(stream));
}

// Enters offsets lo .. hi of the nodes at coordinate c (and its images) along
// an axis of n nodes; false when the table is full.
bool plan_wide(GhostPlan &w, int axis, int c, int lo, int hi, int n) {
    if (lo >= -1 && hi <= 1) return true;
    for (int s = -1; s <= 1; ++s) {
        const int at = c + s * n;
        if (at < -16 || at >= n + 16) continue;  // no region reaches further
        int e = 0;
        while (e < w.n[axis] && w.at[axis][e] != at) ++e;
        if (e == kGhostMaxWide) return false;
        if (e == w.n[axis]) {
            w.at[axis][w.n[axis]++] = at;
            w.lo[axis][e] = w.hi[axis][e] = 0;
        }
        if (lo < w.lo[axis][e]) w.lo[axis][e] = lo;
        if (hi > w.hi[axis][e]) w.hi[axis][e] = hi;
    }
    return true;
}

// Collects the columns and rows that read beyond their neighbours; false when
// a rule does so over a range of several columns or rows, or too many do.
bool ghost_plan(const GhostParams &p, GhostPlan &w) {
    w = GhostPlan{};
    const int nx = p.nx, ny = p.ny;
    const bool before = p.pbc_mode == LBM_PBC_BEFORE_STREAM, after = p.pbc_mode == LBM_PBC_AFTER_STREAM;
    if (after)  // columns 0 and nx-1 pull column nx-2 = -2 and column 1 = (nx-1) + 2
        if (!plan_wide(w, 0, 0, -3, -1, nx) || !plan_wide(w, 0, nx - 1, 1, 3, nx)) return false;
    if (before)  // pulls from column 0 read column nx-2, from nx-1 column 1
        if (!plan_wide(w, 0, 0, -2, 1, nx) || !plan_wide(w, 0, 1, -3, 1, nx) ||
            !plan_wide(w, 0, nx - 1, -1, 2, nx) || !plan_wide(w, 0, nx - 2, -1, 3, nx))
            return false;
    for (int r = 0; r < p.nrules; ++r) {
        const lbm_ghost_rule &a = p.rules[r];
        if (a.kind == LBM_RULE_ZERO) continue;
        auto cxi = [](int i) { return int(i == 1 || i == 5 || i == 8) - int(i == 3 || i == 6 || i == 7); };
        auto cyi = [](int i) { return int(i == 2 || i == 5 || i == 6) - int(i == 4 || i == 7 || i == 8); };
        int lx = a.dx - cxi(a.src_ch), hx = lx, ly = a.dy - cyi(a.src_ch), hy = ly;
        if (a.kind == LBM_RULE_LID_RHO) {  // channels 0, 1, 2, 3, 5, 6 as well
            lx = a.dx - 1, hx = a.dx + 1;
            ly = ly < a.dy - 1 ? ly : a.dy - 1, hy = hy > a.dy ? hy : a.dy;
        }
        if ((lx < -1 || hx > 1) && a.x1 - a.x0 > 1) return false;
        if (!plan_wide(w, 0, a.x0, lx, hx, nx)) return false;
        // targets whose source is (AFTER) or is pulled from (BEFORE) an inlet
        // or outlet column read the opposite interior columns
        for (int side = 0; side < 2 && (after || before); ++side) {
            const int col = side ? nx - 1 : 0;
            const int first = after ? col - a.dx : col - hx, last = after ? col - a.dx : col - lx;
            for (int s = -1; s <= 1; ++s)
                for (int x = first + s * nx; x <= last + s * nx; ++x) {
                    if (x < a.x0 || x >= a.x1) continue;
                    const int o = col + s * nx - x;  // offset of that column
                    const int l = after ? o + (side ? 1 : -3) : o + (side ? 2 : -2);
                    const int h = after ? o + (side ? 3 : -1) : l;
                    if (!plan_wide(w, 0, x, l, h, nx)) return false;
                    if (after) {
                        ly = ly < a.dy - 1 ? ly : a.dy - 1;
                        hy = hy > a.dy + 1 ? hy : a.dy + 1;
                    }
                }
        }
        if (ly < -1 || hy > 1) {
            if (a.y1 - a.y0 > 1) return false;
            if (!plan_wide(w, 1, a.y0, ly, hy, ny)) return false;
        }
    }
    for (int r = 0; r < p.nrules; ++r)
        for (int q = r + 1; q < p.nrules; ++q) {
            const lbm_ghost_rule &a = p.rules[r], &b = p.rules[q];
            if (a.ch == b.ch && rect_hits(a.x0, a.x1, a.y0, a.y1, b.x0, b.x1, b.y0, b.y1))
                w.over[r] |= uint32_t(1) << q;
        }
    return true;
}

// What the d steps after it read of a step along one axis, given that they
// end on [a, b): widens a and b (b exclusive).
void ghost_extent(const GhostPlan &w, int axis, int d, int &a, int &b) {
    for (int j = 0; j < d; ++j) {
        int l = a - 1, h = b + 1;
        for (int e = 0; e < w.n[axis]; ++e) {
            const int c = w.at[axis][e];
            if (c < a || c >= b) continue;
            if (c + w.lo[axis][e] < l) l = c + w.lo[axis][e];
            if (c + w.hi[axis][e] >= h) h = c + w.hi[axis][e] + 1;
        }
        a = l;
        b = h;
    }
}

// Whether every tile's region along an axis of n nodes, in tiles of t, fits
// `room` nodes, and the grid is at least as wide.
bool plan_fits(const GhostPlan &w, int axis, int n, int t, int K, int room) {
    if (n < room) return false;
    for (int a0 = 0; a0 < n; a0 += t) {
        int a = a0, b = a0 + t < n ? a0 + t : n;
        ghost_extent(w, axis, K - 1, a, b);
        if (b - a > room || a < -12 || b > n + 12) return false;
        if (w.n[axis] == 0 && a0 == 0) break;  // the others are shifted copies
    }
    return true;
}

template <typename T, int TR, int TC, int BS, int PITCH, int ROWS, int WPE>
bool launch_ghost_multi(const T *src, T *dst, int layout, const GhostParams &p, const GhostPlan &w,
                        int K, T *rho, T *ux, T *uy, hipStream_t s, bool check) {
    // an inlet and outlet always need room beyond the K - 1 nodes of the pulls
    constexpr bool wide = ROWS > TR + 2 * (kGhostMaxK - 1);
    if (check) {
        if (p.pbc_mode != LBM_PBC_NONE && !wide) return false;
        int64_t items = 0;  // of the rules in one tile, at most
        for (int r = 0; r < p.nrules; ++r) {
            const int w0 = p.rules[r].x1 - p.rules[r].x0, h0 = p.rules[r].y1 - p.rules[r].y0;
            items += int64_t(w0 < ROWS ? w0 : ROWS) * (h0 < PITCH ? h0 : PITCH);
        }
        static_assert(4 * (PITCH + 2) <= BS, "an inlet / outlet node per thread");
        return items <= BS && plan_fits(w, 0, p.nx, TR, K, ROWS) && plan_fits(w, 1, p.ny, TC, K, PITCH);
    }
    constexpr int NA = ROWS * PITCH;
    const int ntc = (p.ny + TC - 1) / TC, nt = ntc * ((p.nx + TR - 1) / TR);
    const dim3 grid(unsigned((nt + 7) / 8 * 8));
    const bool rows = layout == LBM_LAYOUT_ROWS;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(BS), 0, s, src, dst, p, w, K, ntc, nt, rho, ux, uy);
    };
    if (p.pbc_mode == LBM_PBC_NONE) {
        if (rows) launch(k_ghost_multi<T, true, false, TR, TC, BS, PITCH, NA, WPE>);
        else launch(k_ghost_multi<T, false, false, TR, TC, BS, PITCH, NA, WPE>);
    } else if constexpr (wide) {
        if (rows) launch(k_ghost_multi<T, true, true, TR, TC, BS, PITCH, NA, WPE>);
        else launch(k_ghost_multi<T, false, true, TR, TC, BS, PITCH, NA, WPE>);
    }
    return true;
}

// Tile shapes, four steps per launch.  VALU-bound at large grids, like the
// cavity's tiles, so the widest tile that leaves two blocks per CU:
// 1: flows that read their neighbours only; 4098^2 FP64 sliding lid 173 us a
//    step (97 GLUPS), 452 us with one step per launch (HBM-bound, 5.4 TB/s);
// 0: room for the inlet and outlet columns, 512 threads because their
//    arithmetic spills at the 80 registers that 768 leave: 4098^2 FP64 canal
//    253 us a step against 425 with one step per launch, 1000 x 1501 24 us
//    against 33 with 768 threads;
// 2: grids of so few tiles of shape 0 that half of the CUs had none: more and
//    smaller blocks, all latency; 102 x 52 FP64 canal 4.1 us a step against 12.0,
//    where the inlet and outlet take 1.9 us of it and the rules 1.0.  Six or eight
//    steps per launch (4.4, 4.6 us), also with one loop body for all steps, gave nothing.
template <typename T>
bool ghost_multi(int shape, const T *src, T *dst, int layout, const GhostParams &p, const GhostPlan &w,
                 int K, T *rho, T *ux, T *uy, hipStream_t s, bool check) {
    switch (shape) {
    case 0: return launch_ghost_multi<T, 17, 32, 512, 39, 28, 4>(src, dst, layout, p, w, K, rho, ux, uy, s, check);
    case 1: return launch_ghost_multi<T, 22, 32, 768, 38, 28, 6>(src, dst, layout, p, w, K, rho, ux, uy, s, check);
    default: return launch_ghost_multi<T, 6, 16, 512, 24, 17, 4>(src, dst, layout, p, w, K, rho, ux, uy, s, check);
    }
}

template <typename T>
int ghost_run(T *a, T *b, int64_t nx, int64_t ny, int layout, double omega, const lbm_ghost_rule *rules,
              int nrules, const lbm_ghost_pbc *pbc, int64_t steps, T *rho, T *ux, T *uy, int *in_b,
              void *stream) {
    if (!in_b) return LBM_E_NULL;
    *in_b = 0;
    GhostParams p;
    int rc = ghost_params<T>(a, b, nx, ny, layout, omega, rules, nrules, pbc, 0, rho, ux, uy, p);
    if (rc) return rc;
    if (steps < 0) return LBM_E_SIZE;
    hipStream_t s = as_stream(stream);
    GhostPlan w;
    int shape = -1;
    if (steps > 1 && ghost_plan(p, w)) {
        // us a step, FP64 (FP32), shapes 0 / 1 / 2: canal 102 x 52, 12 tiles of shape 0,
        // 5.5 / - / 4.1 (4.4 / 3.9), 200^2, 84 tiles, 5.4 / - / 4.5 (4.4 / 4.3), 300^2,
        // 180 tiles, 5.4 / - / 6.4 (4.4 / 6.0), 600^2 8.2 / - / 16.5 (6.5 / 14.9); lid
        // 200^2 3.3 / 3.6 / 3.0 (2.9 / 3.1 / 2.6), 300^2 3.4 / 3.7 / 4.3 (3.0 / 3.2 /
        // 3.1), 500^2 4.9 / 5.3 / 7.6 (3.6 / 4.2 / 5.7).  Shape 1 where it saves a round
        // of two blocks a CU: 1000 x 300, 590 tiles against 460, 6.0 / 5.3 / 8.4 (4.1 /
        // 3.9 / 6.3), but 600^2, 684 against 532, 6.6 / 7.2 / 9.9 (4.1 / 5.2 / 6.9).
        const int64_t cus = device_cus();
        const int64_t tiles0 = ((nx + 16) / 17) * ((ny + 31) / 32), tiles1 = ((nx + 21) / 22) * ((ny + 31) / 32);
        auto rounds = [&](int64_t tiles) { return (tiles + 2 * cus - 1) / (2 * cus); };
        // wide-reading flows do not fit shape 1, and narrow or crowded grids may
        // fit shape 2 only
        const int order[3] = {2 * tiles0 <= cus ? 2 : (rounds(tiles1) < rounds(tiles0) ? 1 : 0), 0, 2};
        for (int k = 0; k < 3 && shape < 0; ++k)
            if (ghost_multi<T>(order[k], a, b, layout, p, w, kGhostMaxK, rho, ux, uy, s, true))
                shape = order[k];
    }
    // The state has to end where single-step launches would leave it (a graph that a
    // program captures of an even number of steps reads the buffer it ends in), so
    // their number is odd for an odd number of steps, even for an even one.  Large
    // tiles: four steps a launch as long as the others get one each, because a
    // single step is HBM-bound and cheap beside two or three on tiles (4098^2 FP64
    // sliding lid, us a launch of 1, 2, 3, 4 steps: 445, 664, 640, 692; canal 425,
    // 667, 814, 977).  Small tiles: as even as possible (102 x 52 canal, two steps
    // 10.3 us, three 13.6, four 16.6, a single step 12.1).
    int64_t launches = shape < 0 ? steps : (steps + kGhostMaxK - 1) / kGhostMaxK;
    if ((launches ^ steps) & 1) ++launches;
    for (; launches > 0; --launches) {
        const T *src = *in_b ? b : a;
        T *dst = *in_b ? a : b;
        const int64_t most = shape == 2 ? (steps + launches - 1) / launches : steps - launches + 1;
        const int K = int(most < kGhostMaxK ? most : kGhostMaxK);
        const bool last = steps == K;
        T *r = last ? rho : nullptr, *u = last ? ux : nullptr, *v = last ? uy : nullptr;
        if (K == 1) {
            rc = launch_ghost_step<T>(src, dst, layout, p, r, u, v, s);
        } else {
            (void)ghost_multi<T>(shape, src, dst, layout, p, w, K, r, u, v, s, false);
            rc = launch_status();
        }
        if (rc) return rc;
        *in_b = !*in_b;
        steps -= K;
    }
    return LBM_OK;
}

}  // namespace
}  // namespace lbm

extern "C" {

int lbm_ghost_equilibrium_f64(const double *rho, const double *ux, const double *uy, double *f,
                              int64_t n, void *stream) {
    return lbm::ghost_equilibrium<double>(rho, ux, uy, f, n, stream);
}

int lbm_ghost_equilibrium_f32(const float *rho, const float *ux, const float *uy, float *f,
                              int64_t n, void *stream) {
    return lbm::ghost_equilibrium<float>(rho, ux, uy, f, n, stream);
}

int lbm_ghost_step_f64(const double *src, double *dst, int64_t nx, int64_t ny, int layout,
                       double omega, const lbm_ghost_rule *rules, int nrules,
                       const lbm_ghost_pbc *pbc, int flags, double *rho, double *ux, double *uy,
                       void *stream) {
    return lbm::ghost_step<double>(src, dst, nx, ny, layout, omega, rules, nrules, pbc, flags,
                                   rho, ux, uy, stream);
}

int lbm_ghost_step_f32(const float *src, float *dst, int64_t nx, int64_t ny, int layout,
                       double omega, const lbm_ghost_rule *rules, int nrules,
                       const lbm_ghost_pbc *pbc, int flags, float *rho, float *ux, float *uy,
                       void *stream) {
    return lbm::ghost_step<float>(src, dst, nx, ny, layout, omega, rules, nrules, pbc, flags, rho,
                                  ux, uy, stream);
}

int lbm_ghost_run_f64(double *a, double *b, int64_t nx, int64_t ny, int layout, double omega,
                      const lbm_ghost_rule *rules, int nrules, const lbm_ghost_pbc *pbc,
                      int64_t steps, double *rho, double *ux, double *uy, int *in_b, void *stream) {
    return lbm::ghost_run<double>(a, b, nx, ny, layout, omega, rules, nrules, pbc, steps, rho, ux, uy,
                                  in_b, stream);
}

int lbm_ghost_run_f32(float *a, float *b, int64_t nx, int64_t ny, int layout, double omega,
                      const lbm_ghost_rule *rules, int nrules, const lbm_ghost_pbc *pbc,
                      int64_t steps, float *rho, float *ux, float *uy, int *in_b, void *stream) {
    return lbm::ghost_run<float>(a, b, nx, ny, layout, omega, rules, nrules, pbc, steps, rho, ux, uy,
                                 in_b, stream);
}

}  // extern "C"
