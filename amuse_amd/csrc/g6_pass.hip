// Full passes over slots holding distinct ids (g6x_calc_self over every
// slot), every unordered pair evaluated once for both of its particles.
//
// The scheme of g6_sym.h at the scale of a workgroup: a block is R = 256 IPL
// slots, 64 IPL rows for each of the workgroup's four waves, and the column
// tiles (64 slots) are staged once for all four.  Row block b takes its own
// tiles row by row (one side, the self pair left out) and once for both
// sides those of the nb / 2 blocks that follow it round the circle of nb
// blocks.  At step k of a tile lane l of each wave pairs its rows with column
// (l + k) mod 64, whose sums and smallest r^2 come to it from the next lane; a
// tile's column sums are added over the four waves in wave order and written
// as one record per (row block, column), the rows' sums as one per workgroup
// and row.  Blocks are taken some distances round the circle at a time
// (launches whose column records fit the workspace), and after each a second
// kernel adds every particle's records, in a fixed order, to its running sums.
//
// Nearest neighbour: the smallest r^2 with, for a row, the tile, and for a
// column, the row block it was met in; of equal r^2 the range with the lower
// slots is kept (ranges are disjoint), and the slot, the first in the range
// with that r^2, is found once at the end.  r^2 of a pair has the same bits
// from both sides.
#include "g6_kernels.h"
#include "g6_predict.h"
#include "g6_reduce.h"
#include "g6_sym.h"

#include <algorithm>

namespace g6k {

namespace {

constexpr int kCol = g6s::kCol;
constexpr int kColFields = 8;
// One launch: rows of every block against the blocks d0 <= d < d1 places on.
struct PassArgs {
    const double *jx, *jy, *jz, *jm, *jvx, *jvy, *jvz;                     // FP64
    const float *hx, *hy, *hz, *lx, *ly, *lz, *fm, *fvx, *fvy, *fvz;       // mixed
    double eps2;
    int n, nb, d0, d1;
    int per, parts;     // tiles per workgroup, workgroups per row block
    double *rowrec;     // [workgroup][Op::kRow][R]: the sums (FP64: hi and lo), r^2, its tile
    double *colrec;     // [d - max(d0, 1)][kColFields][n]: the sums, r^2
};

__device__ __forceinline__ bool pass_takes(const PassArgs &p, int b, int d)
{
    return d == 0 || 2 * d < p.nb || b < p.nb / 2;
}

__device__ __forceinline__ double rsqrt64(double s)
{
    const double y = __builtin_amdgcn_rsq(s);
    const double h = s * y;
    const double e = __builtin_fma(-h, y, 1.0);
    const double t = __builtin_fma(e, 0.375, 0.5);
    return __builtin_fma(y * e, t, y);
}

// The smaller value, without the canonicalising maxima the compiler puts
// before fmin (both come out of arithmetic or are +inf): the other one where
// one is NaN.
__device__ __forceinline__ double vmin(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float vmin(float a, float b)
{
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// What every form's pair does with its separation d, r^2 q and r^-1 y: row
// mass and velocity (m, v), column's (cm, cv); adds to the row's sums s and,
// for BOTH, to the column's z (FIRST: sets them).
template <class T, bool BOTH, bool FIRST>
__device__ __forceinline__ void pass_terms(T dx, T dy, T dz, T y, T m, const T *v, T cm,
                                           const T *cv, T *s, T *z)
{
    const T y2 = y * y, y3 = y * y2;
    const T wx = cv[0] - v[0], wy = cv[1] - v[1], wz = cv[2] - v[2];
    const T rv = fma_t(dz, wz, fma_t(dy, wy, dx * wx));
    const T a = (T(-3) * rv) * y2;
    const T ex = fma_t(a, dx, wx), ey = fma_t(a, dy, wy), ez = fma_t(a, dz, wz);
    const T m3 = cm * y3;
    s[0] = fma_t(m3, dx, s[0]);
    s[1] = fma_t(m3, dy, s[1]);
    s[2] = fma_t(m3, dz, s[2]);
    s[3] = fma_t(m3, ex, s[3]);
    s[4] = fma_t(m3, ey, s[4]);
    s[5] = fma_t(m3, ez, s[5]);
    s[6] = fma_t(-cm, y, s[6]);
    if (BOTH) {
        const T n3 = -m * y3;
        if (FIRST) {
            z[0] = n3 * dx; z[1] = n3 * dy; z[2] = n3 * dz;
            z[3] = n3 * ex; z[4] = n3 * ey; z[5] = n3 * ez;
            z[6] = -m * y;
        } else {
            z[0] = fma_t(n3, dx, z[0]);
            z[1] = fma_t(n3, dy, z[1]);
            z[2] = fma_t(n3, dz, z[2]);
            z[3] = fma_t(n3, ex, z[3]);
            z[4] = fma_t(n3, ey, z[4]);
            z[5] = fma_t(n3, ez, z[5]);
            z[6] = fma_t(-m, y, z[6]);
        }
    }
}

// The plain path (as g6k::pair_f64): r^2 rounded as the reference does,
// everything else in FP64.
struct PassF64 {
    using T = double;
    using V = double2;
    static constexpr int W = 4;  // LDS words of a column: (x y), (z m), (vx vy), (vz -)
    // tiles a lane's plain sums run over before they are folded: 128 pairs below
    // 50000 particles, 256 above, as the pair by pair kernels.  Root mean square
    // error over theirs, acc / jerk / pot: 0.91 / 0.90 / 0.90 at N = 20000 (256 pairs
    // and columns' sums of a whole tile: 1.11 / 1.07 / 1.21), 0.90 / 0.83 / 0.87 at
    // 65536.  Folds at 64 pairs: 0.87 / 0.82 / 0.76, and N = 45000 2010 -> 2150 us.
    template <int IPL>
    static constexpr int kFold = IPL == 2 ? 2 : 4;
    static constexpr int kSum = 2, kRow = 16;  // values of a row's sum, of its record
    // the columns' sums continue on from lane to lane (plain sums of kSeg IPL
    // terms): a rotation moves 64-bit values and does not fuse with an add
    static constexpr bool kChain = true;

    struct Row {
        T x[3], m, v[3];
    };
    static __device__ __forceinline__ void load(const PassArgs &p, int j, Row &r)
    {
        const bool in = j < p.n;
        const int k = in ? j : 0;
        r.x[0] = in ? p.jx[k] : kFar; r.x[1] = in ? p.jy[k] : kFar; r.x[2] = in ? p.jz[k] : kFar;
        r.m = in ? p.jm[k] : 0.0;
        r.v[0] = p.jvx[k]; r.v[1] = p.jvy[k]; r.v[2] = p.jvz[k];
    }
    static __device__ __forceinline__ V word(const PassArgs &p, int w, int j)
    {
        const bool in = j < p.n;
        const int k = in ? j : 0;
        switch (w) {
        case 0: return make_double2(in ? p.jx[k] : kFar, in ? p.jy[k] : kFar);
        case 1: return make_double2(in ? p.jz[k] : kFar, in ? p.jm[k] : 0.0);
        case 2: return make_double2(p.jvx[k], p.jvy[k]);
        default: return make_double2(p.jvz[k], 0.0);
        }
    }
    static __device__ __forceinline__ T r2_of(T dx, T dy, T dz)
    {
#pragma clang fp contract(off)
        T r2 = dx * dx;
        r2 = r2 + dy * dy;
        r2 = r2 + dz * dz;
        return r2;
    }
    // r^2 of particles i and j
    static __device__ __forceinline__ T r2(const PassArgs &p, int i, int j)
    {
        Row r, c;
        load(p, i, r);
        load(p, j, c);
        return r2_of(c.x[0] - r.x[0], c.x[1] - r.x[1], c.x[2] - r.x[2]);
    }
    template <bool BOTH, bool FIRST, class R>
    static __device__ __forceinline__ void pair(const R &r, const V (&c)[W], T eps2, bool self,
                                                T *s, T &rm, T *z, T &zm)
    {
        const T dx = c[0].x - r.x[0], dy = c[0].y - r.x[1], dz = c[1].x - r.x[2];
        const T q = r2_of(dx, dy, dz);
        T y = rsqrt64(q + eps2);
        if (BOTH) {
            rm = vmin(rm, q);
            zm = FIRST ? q : vmin(zm, q);
        } else {
            y = self ? 0.0 : y;
            rm = vmin(rm, self ? __builtin_inf() : q);
        }
        const T cv[3] = {c[2].x, c[2].y, c[3].x};
        pass_terms<T, BOTH, FIRST>(dx, dy, dz, y, r.m, r.v, c[1].y, cv, s, z);
    }
};

// The mixed path (as g6k::pair_mx): dx from double-single positions, FP32 sums
// over 64 pairs.
struct PassMx {
    using T = float;
    using V = float4;
    static constexpr int W = 3;  // (hx hy hz m), (lx ly lz vx), (vy vz - -)
    template <int IPL>
    static constexpr int kFold = 1;
    static constexpr int kSum = 1, kRow = 9;
    static constexpr bool kChain = false;

    struct Row {
        T h[3], l[3], m, v[3];
    };
    static __device__ __forceinline__ void load(const PassArgs &p, int j, Row &r)
    {
        const bool in = j < p.n;
        const int k = in ? j : 0;
        r.h[0] = in ? p.hx[k] : kFarF; r.h[1] = in ? p.hy[k] : kFarF; r.h[2] = in ? p.hz[k] : kFarF;
        r.l[0] = p.lx[k]; r.l[1] = p.ly[k]; r.l[2] = p.lz[k];
        r.m = in ? p.fm[k] : 0.0f;
        r.v[0] = p.fvx[k]; r.v[1] = p.fvy[k]; r.v[2] = p.fvz[k];
    }
    static __device__ __forceinline__ V word(const PassArgs &p, int w, int j)
    {
        const bool in = j < p.n;
        const int k = in ? j : 0;
        switch (w) {
        case 0:
            return make_float4(in ? p.hx[k] : kFarF, in ? p.hy[k] : kFarF, in ? p.hz[k] : kFarF,
                               in ? p.fm[k] : 0.0f);
        case 1: return make_float4(p.lx[k], p.ly[k], p.lz[k], p.fvx[k]);
        default: return make_float4(p.fvy[k], p.fvz[k], 0.0f, 0.0f);
        }
    }
    static __device__ __forceinline__ T r2_of(T dx, T dy, T dz)
    {
        return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
    }
    template <class R>
    static __device__ __forceinline__ T r2_near(const R &r, const R &c)
    {
        return r2_of((c.h[0] - r.h[0]) + (c.l[0] - r.l[0]), (c.h[1] - r.h[1]) + (c.l[1] - r.l[1]),
                     (c.h[2] - r.h[2]) + (c.l[2] - r.l[2]));
    }
    static __device__ __forceinline__ T r2(const PassArgs &p, int i, int j)
    {
        Row r, c;
        load(p, i, r);
        load(p, j, c);
        return r2_near(r, c);
    }
    // The rest of a pair from its separation.
    template <bool BOTH, bool FIRST>
    static __device__ __forceinline__ void terms(T dx, T dy, T dz, T m, const T *v, T cm,
                                                 const T *cv, T eps2, bool self, T *s, T &rm, T *z,
                                                 T &zm)
    {
        const T q = r2_of(dx, dy, dz);
        T y = __builtin_amdgcn_rsqf(q + eps2);
        if (BOTH) {
            rm = vmin(rm, q);
            zm = FIRST ? q : vmin(zm, q);
        } else {
            y = self ? 0.0f : y;
            rm = vmin(rm, self ? __builtin_inff() : q);
        }
        pass_terms<T, BOTH, FIRST>(dx, dy, dz, y, m, v, cm, cv, s, z);
    }
    template <bool BOTH, bool FIRST, class R>
    static __device__ __forceinline__ void pair(const R &r, const V (&c)[W], T eps2, bool self,
                                                T *s, T &rm, T *z, T &zm)
    {
        const T dx = (c[0].x - r.h[0]) + (c[1].x - r.l[0]);
        const T dy = (c[0].y - r.h[1]) + (c[1].y - r.l[1]);
        const T dz = (c[0].z - r.h[2]) + (c[1].z - r.l[2]);
        const T cv[3] = {c[1].w, c[2].x, c[2].y};
        terms<BOTH, FIRST>(dx, dy, dz, r.m, r.v, c[0].w, cv, eps2, self, s, rm, z, zm);
    }
};

// The 64 steps of a tile; acc: its columns' sums (g6s::settle) and smallest r^2.
template <class Op, int IPL, bool BOTH, class Row, int TW>
__device__ __forceinline__ void pass_steps(const typename Op::V (&tile)[TW][2 * kCol],
                                           typename Op::T (&acc)[8][kCol], typename Op::T eps2,
                                           int col0, int row0, const Row (&r)[IPL],
                                           typename Op::T (&s)[IPL][7], typename Op::T (&rm)[IPL])
{
    using T = typename Op::T;
    constexpr int kStep = BOTH ? g6s::kSeg : kCol;
    const int lane = threadIdx.x & 63;
    T u[8];
    u[7] = T(__builtin_inf());
    if (BOTH) g6s::put_zero<7>(acc);
#pragma unroll 1
    for (int k0 = 0; k0 < kCol; k0 += kStep) {
#pragma unroll
        for (int q = 0; q < 7; q++) u[q] = T(0);
#pragma unroll 1
        for (int k = k0; k < k0 + kStep; k++) {
            typename Op::V c[Op::W];
#pragma unroll
            for (int w = 0; w < Op::W; w++) c[w] = tile[w][lane + k];
            const int j = col0 + ((lane + k) & 63);
            T z[8];
            if (BOTH && Op::kChain) {
#pragma unroll
                for (int q = 0; q < 8; q++) z[q] = g6s::from_next_lane(u[q]);
            }
            Op::template pair<BOTH, !Op::kChain>(r[0], c, eps2, j == row0 + lane, s[0], rm[0], z, z[7]);
#pragma unroll
            for (int q = 1; q < IPL; q++)
                Op::template pair<BOTH, false>(r[q], c, eps2, j == row0 + lane + kCol * q, s[q],
                                               rm[q], z, z[7]);
            if (BOTH) {
#pragma unroll
                for (int q = 0; q < 7; q++)
                    u[q] = Op::kChain ? z[q] : z[q] + g6s::from_next_lane(u[q]);
                u[7] = Op::kChain ? z[7] : vmin(z[7], g6s::from_next_lane(u[7]));
            }
        }
        if (BOTH) g6s::settle<7>(acc, k0 + kStep - 1, u);
    }
    if (BOTH) acc[7][lane] = g6s::from_next_lane(u[7]);
}

template <class Op, int IPL>
__global__ void __launch_bounds__(kWG, (sizeof(typename Op::T) == 8 ? 2 : IPL == 2 ? 4 : 3)) k_pass(PassArgs p)
{
    using T = typename Op::T;
    using V = typename Op::V;
    constexpr int W = Op::W, R = kWG * IPL, Q = R / kCol;
    static_assert(W <= 4, "each wave stages one word of a column");
    __shared__ V tile[2][W][2 * kCol];
    __shared__ T sum[2][4][8][kCol];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int b = blockIdx.x / p.parts, u0 = (blockIdx.x - b * p.parts) * p.per;
    const int u1 = min((p.d1 - p.d0) * Q, u0 + p.per);
    const int row0 = b * R + wave * kCol * IPL;
    const T eps2 = T(p.eps2);
    auto dist = [&](int u) { return p.d0 + u / Q; };
    auto column = [&](int u) {  // first column of unit u's tile, or n where there is none
        const int d = dist(u), cb = b + d < p.nb ? b + d : b + d - p.nb;
        return u < u1 && pass_takes(p, b, d) ? min(cb * R + (u % Q) * kCol, p.n) : p.n;
    };
    auto next = [&](int u) {  // the first unit from u on that has a tile
        while (u < u1 && column(u) >= p.n) u++;
        return u;
    };
    typename Op::Row r[IPL];
    T s[IPL][7], best[IPL];
    g6s::Long<T> tot[IPL][7];  // FP32 sums: folded every tile (in FP64), kept in registers
    int btile[IPL];
#pragma unroll
    for (int i = 0; i < IPL; i++) {
        Op::load(p, row0 + lane + kCol * i, r[i]);
#pragma unroll
        for (int k = 0; k < 7; k++) s[i][k] = T(0);
        best[i] = T(__builtin_inf());
        btile[i] = 0x7fffffff;
    }
    // the rows' record; FP64: hi and lo of the sums so far (in cache between
    // folds: in registers they would cost the kernel a row per lane)
    double *const rec = p.rowrec + size_t(blockIdx.x) * Op::kRow * R;  // wave-uniform
    const unsigned at = wave * kCol * IPL + lane;
    bool any = false;
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < IPL; i++) {
#pragma unroll
            for (int k = 0; k < 7; k++) {
                if constexpr (sizeof(T) == 4) {
                    tot[i][k].add(s[i][k]);
                } else {
                    double *const qh = rec + 2 * k * R, *const ql = qh + R;
                    double h = 0.0, l = 0.0;
                    if (any) {
                        h = qh[at + kCol * i];
                        l = ql[at + kCol * i];
                    }
                    two_sum_add_d(h, l, double(s[i][k]));
                    qh[at + kCol * i] = h;
                    ql[at + kCol * i] = l;
                }
                s[i][k] = T(0);
            }
        }
        any = true;
    };
    auto stage = [&](int buf, V e) {
        if (wave < W) {
            tile[buf][wave][lane] = e;
            tile[buf][wave][lane + kCol] = e;
        }
    };
    int u = next(u0), buf = 0, tiles = 0;
    V pre{};
    if (u < u1) stage(0, Op::word(p, wave, column(u) + lane));
    __syncthreads();
    while (u < u1) {
        const int un = next(u + 1), col0 = column(u), d = dist(u);
        if (un < u1) pre = Op::word(p, wave, column(un) + lane);
        T rm[IPL];
#pragma unroll
        for (int i = 0; i < IPL; i++) rm[i] = T(__builtin_inf());
        if (d > 0)
            pass_steps<Op, IPL, true>(tile[buf], sum[buf][wave], eps2, col0, row0, r, s, rm);
        else
            pass_steps<Op, IPL, false>(tile[buf], sum[buf][wave], eps2, col0, row0, r, s, rm);
#pragma unroll
        for (int i = 0; i < IPL; i++) {
            const bool less = rm[i] < best[i] || (rm[i] == best[i] && col0 < btile[i]);
            best[i] = less ? rm[i] : best[i];
            btile[i] = less ? col0 : btile[i];
        }
        if (un < u1) stage(buf ^ 1, pre);
        __syncthreads();
        if (d > 0) {
            // this tile's column records: the other buffers are in use meanwhile
            double *cr = p.colrec + size_t(d - max(p.d0, 1)) * kColFields * p.n;
            for (int k = t; k < kColFields * kCol; k += kWG) {
                const int f = k >> 6, e = k & 63;
                double v;
                if (f < 7) {
                    g6s::Long<T> z;
#pragma unroll
                    for (int w = 0; w < 4; w++) z.add(sum[buf][w][f][e]);
                    v = z.value();
                } else {
                    T q = sum[buf][0][7][e];
#pragma unroll
                    for (int w = 1; w < 4; w++) q = vmin(q, sum[buf][w][7][e]);
                    v = double(q);
                }
                if (col0 + e < p.n) cr[size_t(f) * p.n + col0 + e] = v;
            }
        }
        if (++tiles == Op::template kFold<IPL>) {
            tiles = 0;
            fold();
        }
        u = un;
        buf ^= 1;
    }
    if (tiles > 0 || !any) fold();
#pragma unroll
    for (int i = 0; i < IPL; i++) {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int k = 0; k < 7; k++) (rec + k * R)[at + kCol * i] = tot[i][k].value();
        }
        (rec + (Op::kRow - 2) * R)[at + kCol * i] = double(best[i]);
        (rec + (Op::kRow - 1) * R)[at + kCol * i] = double(btile[i]);
    }
}

// Adds the records of one launch to the running sums: blockIdx.y < 7 one sum
// of 256 particles each (run[2 f], run[2 f + 1]: hi and lo), 7 the smallest
// r^2 (run[14]) and its range (run[15]: twice its first slot, plus 1 for a
// row block's).  first: nothing is running yet.  HBM-bound.
template <class Op>
__global__ void __launch_bounds__(256) k_pass_sum(PassArgs p, int R, double *__restrict__ run,
                                                  int first)
{
    const int i = blockIdx.x * 256 + threadIdx.x, f = blockIdx.y;
    if (i >= p.n) return;
    const size_t n = size_t(p.n);
    const int b = i / R, e0 = max(p.d0, 1);
    const double *col = p.colrec + size_t(f) * n + i;
    const size_t cs = kColFields * n, rs = size_t(Op::kRow) * R;
    const double *row = p.rowrec + size_t(b) * p.parts * rs + size_t(Op::kSum * f) * R + (i - b * R);
    // the block opposite (nb even) has no record from the second half's side
    int e1 = p.d1;
    if (e1 > e0 && 2 * (e1 - 1) == p.nb && b < p.nb / 2) e1--;
    if (f < 7) {
        double h = first ? 0.0 : run[size_t(2 * f) * n + i];
        double l = first ? 0.0 : run[size_t(2 * f + 1) * n + i];
#pragma unroll 8
        for (int d = e0; d < e1; d++) two_sum_add_d(h, l, col[size_t(d - e0) * cs]);
#pragma unroll 4
        for (int k = 0; k < p.parts; k++) {
            two_sum_add_d(h, l, row[k * rs]);
            if (Op::kSum == 2) l += row[k * rs + R];
        }
        run[size_t(2 * f) * n + i] = h;
        run[size_t(2 * f + 1) * n + i] = l;
        return;
    }
    double best = first ? __builtin_inf() : run[14 * n + i];
    double at = first ? -1.0 : run[15 * n + i];
    auto take = [&](double r2, double where) {
        if (r2 < best || (r2 == best && r2 < __builtin_inf() && where < at)) {
            best = r2;
            at = where;
        }
    };
#pragma unroll 8
    for (int d = e0; d < e1; d++) {
        const int rb = b - d >= 0 ? b - d : b - d + p.nb;
        take(col[size_t(d - e0) * cs], 2.0 * (double(rb) * R) + 1.0);
    }
#pragma unroll 4
    for (int k = 0; k < p.parts; k++)
        take(row[k * rs], 2.0 * row[k * rs + R]);
    run[14 * n + i] = best;
    run[15 * n + i] = at;
}

// The result rows from the running sums, and the nearest neighbours' ids: a
// wave takes kEnd particles and searches each one's range, lane by lane, for
// the first slot with its r^2.
constexpr int kEnd = 4;
template <class Op>
__global__ void __launch_bounds__(256) k_pass_end(PassArgs p, int R, const double *__restrict__ run,
                                                  const int *__restrict__ pid,
                                                  double *__restrict__ out, int *__restrict__ nn,
                                                  int S, int want_nn)
{
    using T = typename Op::T;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const size_t n = size_t(p.n);
    const int base = blockIdx.x * 4 * kEnd;  // the workgroup's particles
    for (int k = t; k < 7 * 4 * kEnd; k += 256) {
        const int f = k / (4 * kEnd), i = base + k % (4 * kEnd);
        if (i < p.n)
            out[size_t(f) * S + i] = run[size_t(2 * f) * n + i] + run[size_t(2 * f + 1) * n + i];
    }
    if (!want_nn) return;
#pragma unroll 1
    for (int q = 0; q < kEnd; q++) {
        const int i = base + wave * kEnd + q;  // wave-uniform
        if (i >= p.n) return;
        const T best = T(run[14 * n + i]);
        const double at = run[15 * n + i];
        int slot = -1;
        if (best < T(__builtin_inf()) && at >= 0.0) {
            const int code = int(at * 0.5);
            const bool row = at - 2.0 * code < 0.5;  // met as a row, its range a tile
            const int len = row ? kCol : R;
#pragma unroll 4
            for (int k = 0; k < len; k += kCol) {
                const int j = code + k + lane;
                const unsigned long long mask = __ballot(
                    j < p.n && j != i && Op::r2(p, i, min(j, p.n - 1)) == best);
                if (slot < 0 && mask) slot = code + k + __ffsll((long long)mask) - 1;
            }
        }
        if (lane == 0) nn[i] = slot >= 0 ? pid[slot] : -1;
    }
}

// A pass's launches: how many distances round the circle each takes and the
// workgroups of one.
struct PassPlan {
    int R, nb, q, last;  // distances 0 .. last
    int step;            // distances per launch
    long long rec, run;  // values of the records of one launch, of the running sums

    int slots;           // workgroups the chip holds at a time

    PassPlan(int n, int ipl, int slots_, int fields) : slots(slots_)
    {
        R = kWG * ipl;
        nb = (n + R - 1) / R;
        q = R / kCol;
        last = nb / 2;
        // column records of one launch: at most kPassRecs bytes of them
        const long long per = 8ll * kColFields * n;
        step = int(std::max(1ll, std::min((long long)last + 1, kPassRecs / per)));
        run = 16ll * n;
        // (a launch over fewer distances may have more workgroups than one of
        // `step`, but not more than these)
        const long long parts = std::min(step * q, std::max(1, kPassWgs / nb));
        rec = (long long)kColFields * step * n + (long long)fields * R * nb * parts;
    }
    static constexpr long long kPassRecs = 1ll << 29;
    // Workgroups per row block of a launch over `nd` distances: the split
    // that needs the fewest tiles one after another, with half a tile's time for a workgroup's start and end.
    int parts_of(int nd) const
    {
        const int u = nd * q, most = std::min(u, std::max(1, kPassWgs / nb));
        int best = 1;
        double cost = 1e30;
        for (int parts = 1; parts <= most; parts++) {
            const double t = double((nb * parts + slots - 1) / slots) *
                             ((u + parts - 1) / parts + 0.5);
            if (t < cost) {
                cost = t;
                best = parts;
            }
        }
        return best;
    }
    static constexpr int kPassWgs = 8192;
};

// rows per lane
int pass_ipl(int n, int prec)
{
    return n < (prec == kF64 ? 50000 : 20000) ? 2 : 3;
}

// Workgroups the chip's 256 CUs hold at a time (by registers)
int pass_slots(int ipl, int prec) { return 256 * (prec == kF64 ? 2 : ipl == 2 ? 4 : 3); }

template <class Op, int IPL>
hipError_t pass_run(PassArgs a, const JStore &s, const IBlock &b, bool want_nn, double *ws,
                    hipStream_t st)
{
    const PassPlan pl(a.n, IPL, pass_slots(IPL, sizeof(typename Op::T) == 8 ? kF64 : kMixed),
                      Op::kRow);
    double *run = ws;
    a.colrec = ws + pl.run;
    a.rowrec = a.colrec + (long long)kColFields * pl.step * a.n;
    a.nb = pl.nb;
    for (int d = 0; d <= pl.last; d += pl.step) {
        a.d0 = d;
        a.d1 = std::min(pl.last + 1, d + pl.step);
        const int u = (a.d1 - a.d0) * pl.q;
        a.parts = pl.parts_of(a.d1 - a.d0);
        a.per = (u + a.parts - 1) / a.parts;
        hipLaunchKernelGGL((k_pass<Op, IPL>), dim3(pl.nb * a.parts), dim3(kWG), 0, st, a);
        hipLaunchKernelGGL(k_pass_sum<Op>, dim3((a.n + 255) / 256, want_nn ? 8 : 7), dim3(256), 0, st,
                           a, pl.R, run, int(d == 0));
    }
    hipLaunchKernelGGL(k_pass_end<Op>, dim3((a.n + 4 * kEnd - 1) / (4 * kEnd)), dim3(256), 0, st, a, pl.R, run,
                       s.pid, b.out, b.nn, b.cap, int(want_nn));
    return hipGetLastError();
}

}  // namespace

size_t pass_bytes(int n, int prec)
{
    const int ipl = pass_ipl(n, prec);
    const PassPlan pl(n, ipl, pass_slots(ipl, prec),
                      prec == kF64 ? PassF64::kRow : PassMx::kRow);
    return sizeof(double) * size_t(pl.run + pl.rec);
}

hipError_t launch_pass(const JStore &s, const IBlock &b, int n, double eps2, int prec,
                       bool want_nn, double *ws, hipStream_t st)
{
    PassArgs a{};
    a.jx = s.px[0]; a.jy = s.px[1]; a.jz = s.px[2]; a.jm = s.pm;
    a.jvx = s.pv[0]; a.jvy = s.pv[1]; a.jvz = s.pv[2];
    a.hx = s.hx[0]; a.hy = s.hx[1]; a.hz = s.hx[2];
    a.lx = s.lx[0]; a.ly = s.lx[1]; a.lz = s.lx[2];
    a.fm = s.fm; a.fvx = s.fv[0]; a.fvy = s.fv[1]; a.fvz = s.fv[2];
    a.eps2 = eps2;
    a.n = n;
    const int ipl = pass_ipl(n, prec);
    if (prec == kF64)
        return ipl == 2 ? pass_run<PassF64, 2>(a, s, b, want_nn, ws, st)
                        : pass_run<PassF64, 3>(a, s, b, want_nn, ws, st);
    return ipl == 2 ? pass_run<PassMx, 2>(a, s, b, want_nn, ws, st)
                    : pass_run<PassMx, 3>(a, s, b, want_nn, ws, st);
}

}  // namespace g6k
