// Forces inside a cluster with every unordered pair evaluated once (the
// scheme of g6_sym.h, a wave at a time): device code of the ensemble kernels
// (g6_clusters.hip).
//
// A cluster's particles are cut into nb blocks of kRows = 128 (two rows per
// lane).  Unit 0 of a row block is the pairs inside it, units 2 d - 1 and
// 2 d the two halves (64 columns) of the block d places on round the circle
// of blocks, 1 <= d <= nb / 2 (with nb even, only the first nb / 2 row blocks
// take the opposite one).  Each unit costs about the same: 64 steps of two
// pairs per lane.  A wave takes `per` consecutive units of one row block and
// writes one record of its rows' sums and one per tile of columns; the
// records of a particle are added in a fixed order, columns' first, by
// whoever needs its force, so results do not depend on scheduling.
#pragma once
#include "g6_sym.h"

namespace g6cp {

constexpr int kRows = 128, kCol = g6s::kCol, kIPL = 2;
constexpr int kNC = 7;  // sums per record: acc, jerk, pot

// A cluster's cut into waves, and where its records lie.
struct Plan {
    int n, per, nb, parts;  // parts: waves per row block (those without units write nothing)

    __host__ __device__ Plan(int n_, int per_) : n(n_), per(per_)
    {
        nb = (n + kRows - 1) / kRows;
        parts = (1 + kIPL * (nb / 2) + per - 1) / per;
    }
    // distances row block b takes, and blocks that take block b
    __host__ __device__ int distances(int b) const
    {
        return nb / 2 - (nb % 2 == 0 && b >= nb / 2 ? 1 : 0);
    }
    __host__ __device__ int takers(int b) const
    {
        return nb / 2 - (nb % 2 == 0 && b < nb / 2 ? 1 : 0);
    }
    __host__ __device__ int units(int b) const { return 1 + kIPL * distances(b); }
    __host__ __device__ int waves() const { return nb * parts; }
    // all units of the cluster
    __host__ __device__ long long work() const
    {
        return (long long)nb * (1 + kIPL * (nb / 2)) - (nb % 2 == 0 ? kIPL * (nb / 2) : 0);
    }
    // values (FP64) of the records
    __host__ __device__ long long col_values() const { return (long long)(nb / 2) * kNC * n; }
    __host__ __device__ long long values() const
    {
        return col_values() + (long long)waves() * kNC * kRows;
    }
};

// One wave's LDS: the columns' values twice over, so that column
// (l + k) mod 64 is entry l + k, and the columns' sums put down on the way.
template <class T, int W>
struct WaveLds {
    typename g6s::Word<T>::type tile[W][2 * kCol];
    T put[kNC][kCol];
};

// Steps k0 <= k < k1 of a tile: lane l pairs its rows with column
// (l + k) mod 64.  BOTH: the columns' sums u travel with their columns and
// come out with lane l holding those of column (l + k1 - 1) mod 64 (for
// g6s::settle).
template <class Op, int IPL, int NC, bool BOTH, int W>
__device__ __forceinline__ void steps(const typename g6s::Word<typename Op::T>::type (&tile)[W][2 * kCol],
                                      int k0, int k1, const Op &op,
                                      const typename Op::T (*r)[Op::NV], typename Op::T (*s)[kNC],
                                      typename Op::T (&u)[kNC], typename Op::Near &near)
{
    using T = typename Op::T;
    constexpr int N = g6s::Word<T>::n;
    const int lane = threadIdx.x & 63;
    if (BOTH) {
#pragma unroll
        for (int q = 0; q < NC; q++) u[q] = T(0);
    }
#pragma unroll 1
    for (int k = k0; k < k1; k++) {
        T c[W * N], z[kNC];
#pragma unroll
        for (int w = 0; w < W; w++) {
            const auto e = tile[w][lane + k];
            const T *f = reinterpret_cast<const T *>(&e);
#pragma unroll
            for (int q = 0; q < N; q++) c[w * N + q] = f[q];
        }
        op.template pair<NC, BOTH, true>(r[0], c, s[0], z, near);
#pragma unroll
        for (int q = 1; q < IPL; q++) op.template pair<NC, BOTH, false>(r[q], c, s[q], z, near);
        if (BOTH) {
#pragma unroll
            for (int q = 0; q < NC; q++) u[q] = z[q] + g6s::from_next_lane(u[q]);
        }
    }
}

// The pair sums of both kinds: separation d, r^-1 y; row mass and velocity
// (m, v), column's (cm, cv).  Adds to the row's sums s, and for BOTH to the
// column's z (FIRST: sets them).  Returns w = relative velocity.
template <class T, int NC, bool BOTH, bool FIRST>
__device__ __forceinline__ void add_terms(T dx, T dy, T dz, T wx, T wy, T wz, T y, T y2, T m, T cm,
                                          T *s, T *z)
{
    auto fma = [](T a, T b, T c) { return sizeof(T) == 4 ? T(__builtin_fmaf(a, b, c)) : T(__builtin_fma(a, b, c)); };
    const T y3 = y * y2;
    const T rv = fma(dz, wz, fma(dy, wy, dx * wx));
    const T a = (T(-3) * rv) * y2;
    const T ex = fma(a, dx, wx), ey = fma(a, dy, wy), ez = fma(a, dz, wz);
    const T m3 = cm * y3;
    s[0] = fma(m3, dx, s[0]);
    s[1] = fma(m3, dy, s[1]);
    s[2] = fma(m3, dz, s[2]);
    s[3] = fma(m3, ex, s[3]);
    s[4] = fma(m3, ey, s[4]);
    s[5] = fma(m3, ez, s[5]);
    if (NC == 7) s[6] = fma(-cm, y, s[6]);
    if (BOTH) {
        const T n3 = -m * y3;
        if (FIRST) {
            z[0] = n3 * dx; z[1] = n3 * dy; z[2] = n3 * dz;
            z[3] = n3 * ex; z[4] = n3 * ey; z[5] = n3 * ez;
            if (NC == 7) z[6] = -m * y;
        } else {
            z[0] = fma(n3, dx, z[0]);
            z[1] = fma(n3, dy, z[1]);
            z[2] = fma(n3, dz, z[2]);
            z[3] = fma(n3, ex, z[3]);
            z[4] = fma(n3, ey, z[4]);
            z[5] = fma(n3, ez, z[5]);
            if (NC == 7) z[6] = fma(-m, y, z[6]);
        }
    }
}

// The larger of two values, without the canonicalising maxima before fmax
// (the other one where one is NaN, as fmax).
__device__ __forceinline__ double vmax(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ float bits_max(float a, float b)
{
    return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
}

// Mixed: dx from double-single positions, everything else FP32.  Values:
// hx hy hz m lx ly lz vx vy vz.  Near: the largest v^2/s and m_ij^2 r^2/s^4
// (the inverse quartic collision time is the larger of the first squared and
// the second).
struct Mixed {
    using T = float;
    static constexpr int NV = 10, W = 3;
    static constexpr int kRowSteps = kCol;  // steps of a row's plain sum
    struct Near {
        float a = 0.0f, b = 0.0f;
        __device__ __forceinline__ float value() const { return bits_max(a * a, b); }
    };
    const float *hx, *hy, *hz, *lx, *ly, *lz, *m, *vx, *vy, *vz;
    float eps2;

    __device__ __forceinline__ void load(int p, bool in, float far, float (&f)[NV]) const
    {
        f[0] = in ? hx[p] : far; f[1] = in ? hy[p] : far; f[2] = in ? hz[p] : far;
        f[3] = in ? m[p] : 0.0f;
        f[4] = in ? lx[p] : 0.0f; f[5] = in ? ly[p] : 0.0f; f[6] = in ? lz[p] : 0.0f;
        f[7] = in ? vx[p] : 0.0f; f[8] = in ? vy[p] : 0.0f; f[9] = in ? vz[p] : 0.0f;
    }
    static __device__ __forceinline__ float far() { return 1e17f; }
    template <int NC, bool BOTH, bool FIRST>
    __device__ __forceinline__ void pair(const float (&r)[NV], const float *c, float *s, float *z,
                                         Near &near) const
    {
        const float dx = (c[0] - r[0]) + (c[4] - r[4]);
        const float dy = (c[1] - r[1]) + (c[5] - r[5]);
        const float dz = (c[2] - r[2]) + (c[6] - r[6]);
        const float q = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, eps2)));
        const float y = __builtin_amdgcn_rsqf(q);
        const float y2 = y * y;
        const float wx = c[7] - r[7], wy = c[8] - r[8], wz = c[9] - r[9];
        const float v2 = wx * wx + wy * wy + wz * wz;
        near.a = bits_max(near.a, v2 * y2);
        const float u = (r[3] + c[3]) * y2 * y2;
        near.b = bits_max(near.b, u * u * (q - eps2));
        add_terms<float, NC, BOTH, FIRST>(dx, dy, dz, wx, wy, wz, y, y2, r[3], c[3], s, z);
    }
};

// FP64.  Values: x y z m vx vy vz.
struct Plain {
    using T = double;
    static constexpr int NV = 7, W = 4;
    // (of 32 terms; 32 steps would leave the rows' records, rounded once each,
    // above the pair by pair kernels' error by 3-8 % below 1000 particles)
    static constexpr int kRowSteps = kCol / 4;
    struct Near {
        float b = 0.0f;
        __device__ __forceinline__ float value() const { return b; }
    };
    const double *x, *y, *z, *m, *vx, *vy, *vz;
    double eps2;

    __device__ __forceinline__ void load(int p, bool in, double far, double (&f)[NV]) const
    {
        f[0] = in ? x[p] : far; f[1] = in ? y[p] : far; f[2] = in ? z[p] : far;
        f[3] = in ? m[p] : 0.0;
        f[4] = in ? vx[p] : 0.0; f[5] = in ? vy[p] : 0.0; f[6] = in ? vz[p] : 0.0;
    }
    static __device__ __forceinline__ double far() { return 1e100; }
    template <int NC, bool BOTH, bool FIRST>
    __device__ __forceinline__ void pair(const double (&r)[NV], const double *c, double *s,
                                         double *zz, Near &near) const
    {
        const double dx = c[0] - r[0], dy = c[1] - r[1], dz = c[2] - r[2];
        const double q = __builtin_fma(dz, dz, __builtin_fma(dy, dy, __builtin_fma(dx, dx, eps2)));
        double y = __builtin_amdgcn_rsq(q);
        const double e = __builtin_fma(-(q * y), y, 1.0);
        y = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
        const double y2 = y * y;
        const double wx = c[4] - r[4], wy = c[5] - r[5], wz = c[6] - r[6];
        const double v2 = wx * wx + wy * wy + wz * wz;
        const double q1 = v2 * y2;
        const double u = (r[3] + c[3]) * y2 * y2;
        near.b = bits_max(near.b, float(vmax(q1 * q1, u * u * (q - eps2))));
        add_terms<double, NC, BOTH, FIRST>(dx, dy, dz, wx, wy, wz, y, y2, r[3], c[3], s, zz);
    }
};

// Stages columns p0 .. p0 + 63 (those below p1; the others far away and
// massless) in the wave's own LDS.  Its LDS operations are in order: the
// fences only keep the compiler from moving them across each other.
template <class Op>
__device__ __forceinline__ void stage(const Op &op, WaveLds<typename Op::T, Op::W> &lds, int p0, int p1)
{
    using T = typename Op::T;
    using V = typename g6s::Word<T>::type;
    constexpr int N = g6s::Word<T>::n;
    const int lane = threadIdx.x & 63;
    T f[Op::NV];
    op.load(p0 + lane, p0 + lane < p1, Op::far(), f);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int w = 0; w < Op::W; w++) {
        V e;
        T *g = reinterpret_cast<T *>(&e);
#pragma unroll
        for (int k = 0; k < N; k++) g[k] = w * N + k < Op::NV ? f[w * N + k < Op::NV ? w * N + k : 0] : T(0);
        lds.tile[w][lane] = e;
        lds.tile[w][lane + kCol] = e;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

template <class T, int NC, int IPL>
__device__ __forceinline__ void fold(g6s::Long<T> (*tot)[kNC], T (*s)[kNC])
{
#pragma unroll
    for (int i = 0; i < IPL; i++)
#pragma unroll
        for (int k = 0; k < NC; k++) {
            tot[i][k].add(s[i][k]);
            s[i][k] = T(0);
        }
}

// The pairs among 64 rows and themselves: the circle again, lane l with the
// next 31 columns for both sides and the opposite one for its own (each such
// pair is met from both ends).
template <class Op, int NC>
__device__ __forceinline__ void diagonal(const Op &op, WaveLds<typename Op::T, Op::W> &lds,
                                         const typename Op::T (*r)[Op::NV],
                                         g6s::Long<typename Op::T> (*tot)[kNC],
                                         typename Op::T (*s)[kNC], typename Op::Near &near)
{
    using T = typename Op::T;
    T u[kNC];
    g6s::put_zero<NC>(lds.put);
    steps<Op, 1, NC, true>(lds.tile, 1, kCol / 2, op, r, s, u, near);
    g6s::settle<NC>(lds.put, kCol / 2 - 1, u);
    fold<T, NC, 1>(tot, s);
#pragma unroll
    for (int q = 0; q < NC; q++) tot[0][q].add(lds.put[q][threadIdx.x & 63]);
    steps<Op, 1, NC, false>(lds.tile, kCol / 2, kCol / 2 + 1, op, r, s, u, near);
    fold<T, NC, 1>(tot, s);
}

// All 64 steps of a staged tile for IPL rows per lane; sink(q, sum) takes the
// columns' sums, in their own lanes.
template <class Op, int NC, int IPL, class Sink>
__device__ __forceinline__ void whole(const Op &op, WaveLds<typename Op::T, Op::W> &lds,
                                      const typename Op::T (*r)[Op::NV],
                                      g6s::Long<typename Op::T> (*tot)[kNC],
                                      typename Op::T (*s)[kNC], typename Op::Near &near,
                                      Sink &&sink)
{
    using T = typename Op::T;
    constexpr int kSeg = g6s::kSeg;
    T u[kNC];
    g6s::put_zero<NC>(lds.put);
#pragma unroll 1
    for (int h = 0; h < kCol; h += Op::kRowSteps) {
#pragma unroll 1
        for (int k = h; k < h + Op::kRowSteps; k += kSeg) {
            steps<Op, IPL, NC, true>(lds.tile, k, k + kSeg, op, r, s, u, near);
            g6s::settle<NC>(lds.put, k + kSeg - 1, u);
        }
        fold<T, NC, IPL>(tot, s);
    }
#pragma unroll
    for (int q = 0; q < NC; q++) sink(q, lds.put[q][threadIdx.x & 63]);
}

// Wave `wi` of a cluster whose particles are off .. off + n - 1: its rows'
// and columns' records to `col` (values of T) and `row`; returns the lane's
// largest inverse quartic collision time.
template <class Op, int NC>
__device__ __forceinline__ float wave_item(const Op &op, const Plan &p, int off, int wi,
                                           WaveLds<typename Op::T, Op::W> &lds,
                                           typename Op::T *__restrict__ colrec,
                                           double *__restrict__ rowrec)
{
    using T = typename Op::T;
    const int lane = threadIdx.x & 63;
    const int b = wi / p.parts, u0 = (wi - b * p.parts) * p.per;
    const int u1 = min(p.units(b), u0 + p.per);
    typename Op::Near near;
    if (u0 >= u1) return 0.0f;
    const int end = off + p.n, row0 = off + b * kRows;
    T r[kIPL][Op::NV], s[kIPL][kNC];
    g6s::Long<T> tot[kIPL][kNC];
#pragma unroll
    for (int i = 0; i < kIPL; i++) {
        const int q = row0 + lane + kCol * i;
        op.load(q, q < end, -Op::far(), r[i]);
#pragma unroll
        for (int k = 0; k < kNC; k++) s[i][k] = T(0);
    }
#pragma unroll 1
    for (int u = u0; u < u1; u++) {
        if (u == 0) {
            stage(op, lds, row0, end);
            diagonal<Op, NC>(op, lds, &r[0], &tot[0], &s[0], near);
            if (row0 + kCol < end) {
                stage(op, lds, row0 + kCol, end);
                // (the columns are the second rows)
                whole<Op, NC, 1>(op, lds, &r[0], &tot[0], &s[0], near,
                                  [&](int q, T x) { tot[1][q].add(x); });
                diagonal<Op, NC>(op, lds, &r[1], &tot[1], &s[1], near);
            }
            continue;
        }
        const int d = (u + 1) / kIPL, cb = b + d < p.nb ? b + d : b + d - p.nb;
        const int c0 = cb * kRows + ((u + 1) & 1) * kCol;  // in the cluster
        if (c0 >= p.n) continue;
        stage(op, lds, off + c0, end);
        T *w = colrec + (size_t(d - 1) * kNC) * p.n + c0;
        whole<Op, NC, kIPL>(op, lds, &r[0], &tot[0], &s[0], near, [&](int q, T x) {
            if (c0 + lane < p.n) w[size_t(q) * p.n + lane] = x;
        });
    }
    double *w = rowrec + size_t(wi) * kNC * kRows + lane;
#pragma unroll
    for (int i = 0; i < kIPL; i++)
#pragma unroll
        for (int k = 0; k < NC; k++) w[k * kRows + kCol * i] = tot[i][k].value();
    return near.value();
}

// Sum k of the cluster's particle i from its records.
template <class T>
__device__ __forceinline__ double record_sum(const Plan &p, const T *__restrict__ colrec,
                                             const double *__restrict__ rowrec, int i, int k)
{
    const int b = i / kRows, nd = p.takers(b);
    const int np = (p.units(b) + p.per - 1) / p.per;
    const T *c = colrec + size_t(k) * p.n + i;
    const double *r = rowrec + (size_t(b) * p.parts * kNC + k) * kRows + (i - b * kRows);
    g6s::Long<double> z;
#pragma unroll 4
    for (int d = 0; d < nd; d++) z.add(double(c[size_t(d) * kNC * p.n]));
#pragma unroll 4
    for (int q = 0; q < np; q++) z.add(r[size_t(q) * kNC * kRows]);
    return z.value();
}

}  // namespace g6cp
