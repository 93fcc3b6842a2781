// Pair sums over one particle set with every unordered pair evaluated once
// (Newton's third law): the index arithmetic shared by the kernels that do it.
//
// The n x n pair matrix is cut into blocks of R particles (the registers of a
// wave, R / 64 rows a lane), each taken as R / 64 column tiles of 64 columns
// (its lanes).  Row block b takes its own tiles pair by ordered pair, rows
// only, and once for both sides those of the nb / 2 blocks that follow it
// round the circle of nb blocks (with nb even, the first nb / 2 row blocks
// take the block opposite), so every row block has the same work and every
// column the same number of records.  At step k of a tile's 64 lane l pairs
// its rows with column (l + k) mod 64, whose values it reads from LDS and
// whose sums come to it from the lane that held the column before (a
// wavefront rotation), so every sum is taken in an order the program fixes.
// A workgroup takes `per` consecutive tiles of one row block, its waves every
// fourth of them, and writes one partial record for its rows and one per tile
// for the columns; a second kernel adds each particle's records in a fixed
// order, so results do not depend on scheduling.
#pragma once
#include <hip/hip_runtime.h>

namespace g6s {

constexpr int kWG = 256;  // a workgroup's lanes
constexpr int kWaves = kWG / 64;
constexpr int kCol = 64;  // columns of a tile
struct Plan {
    int n = 0, rows = 0;  // particles, rows of a block (multiple of 64)
    int nb = 0;           // blocks
    int per = 0;          // tiles per workgroup
    int parts = 0;        // workgroups per row block

    Plan() = default;
    // The most tiles per workgroup (the same number for each of its waves)
    // that leave `wgs` workgroups.
    Plan(int n_, int rows_, int wgs) : n(n_), rows(rows_)
    {
        nb = (n + rows - 1) / rows;
        const int u = units(), want = (wgs + nb - 1) / nb;
        per = u / want / kWaves * kWaves;
        if (per < kWaves) per = kWaves;
        parts = (u + per - 1) / per;
    }
    __host__ __device__ int units() const { return rows / kCol * (1 + nb / 2); }
    __host__ __device__ int items() const { return nb * parts; }
    // Whether row block b takes the block d places on (1 <= d <= nb / 2).
    __host__ __device__ bool takes(int b, int d) const { return 2 * d < nb || b < nb / 2; }
    // values of the partial records, `nc` sums per particle (the rows' in FP64,
    // the columns', one per tile, in the pass's own type)
    long long row_values(int nc) const { return (long long)items() * nc * rows; }
    long long col_values(int nc) const { return (long long)(nb / 2) * nc * n; }
    // row record of workgroup `it`, sum c, row i of the block
    __host__ __device__ long long row_at(int it, int nc, int c, int i) const
    {
        return ((long long)it * nc + c) * rows + i;
    }
    // column record of particle j's block as the d-th from its row block, sum c
    __host__ __device__ long long col_at(int d, int nc, int c, int j) const
    {
        return ((long long)(d - 1) * nc + c) * n + j;
    }
};

// One 16-byte LDS word.
template <class T>
struct Word;
template <>
struct Word<float> {
    using type = float4;
    static constexpr int n = 4;
};
template <>
struct Word<double> {
    using type = double2;
    static constexpr int n = 2;
};

// Lane l's value of lane l + 1 (lane 63: of lane 0): a DPP wavefront rotation.
__device__ __forceinline__ float from_next_lane(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x134, 0xf, 0xf, true));
}
__device__ __forceinline__ double from_next_lane(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, int(b), 0x134, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, int(b >> 32), 0x134, 0xf, 0xf, true);
    return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}

// A sum kept over many short plain sums: FP32 ones in FP64, FP64 ones as
// hi + lo by TwoSum.
template <class T>
struct Long;
template <>
struct Long<float> {
    double h = 0.0;
    __device__ __forceinline__ void add(float x) { h += double(x); }
    __device__ __forceinline__ double value() const { return h; }
};
template <>
struct Long<double> {
    double h = 0.0, l = 0.0;
    __device__ __forceinline__ void add(double x)
    {
        const double s = h + x;
        const double bp = s - h;
        l += (h - (s - bp)) + (x - bp);
        h = s;
    }
    __device__ __forceinline__ double value() const { return h + l; }
};

// The operation of a pass (Op): NV values read per particle (position first)
// and NC sums; load(j, f) reads particle j's values; pair<BOTH, FIRST>(r, c,
// self, s, z) adds the pair of row r and column c to the row's sums s and, for
// BOTH, to the column's z (FIRST: sets them); self: r and c are one particle
// (only met without BOTH).

// Particle j's values, or for j >= n those of one that contributes nothing:
// zero mass and adjoints, away from every particle (so that y is finite with
// eps2 = 0) but no further than its products with real particles' values stay
// finite, as 0 times an infinity would reach their sums: in FP32 velocities and
// adjoints up to 1e28 (at 1e18, adjoints of 1e21 made every gradient NaN).
template <class T, class Op>
__device__ __forceinline__ void load_values(const Op &op, int j, int n, T (&f)[Op::NV])
{
    if (j < n) {
        op.load(j, f);
    } else {
#pragma unroll
        for (int k = 0; k < Op::NV; k++)
            f[k] = k < 3 ? T(sizeof(T) == 4 ? 1.03e10 - 0.07e10 * k : 1e150) : T(0);
    }
}

// LDS words of a column's values.
template <class T, class Op>
constexpr int kWords = (Op::NV + Word<T>::n - 1) / Word<T>::n;

// Steps between two settlements of the columns' travelling sums, each of IPL
// terms: plain sums of 16 to 64 terms and three additions more per tile, where
// the pair by pair kernels fold plain sums of 64 (FP32 and the FP64
// differentiable sums) or 32 (FP64 clusters) terms.  Settled once a tile, their
// error was up to 1.2 times that of those kernels (pot of clusters and full
// passes); now it is no larger (tests/test_gpu_rounding.py).  1-3 % of a pass:
// FP32 forward n = 16384 125.7 -> 127.7 us, FP64 adjoint 542 -> 553 us.
constexpr int kSeg = 16;

// Settles the columns' sums u after step k of a tile, lane l holding those of
// column (l + k) mod 64: added to put[sum][column] (put_zero before a tile's
// first; all read before the first is written, so one LDS round trip).  put is
// the wave's own LDS and its LDS operations are in order: the fences only keep
// the compiler from moving them across each other.
template <int NC, class T>
__device__ __forceinline__ void put_zero(T (*put)[kCol])
{
#pragma unroll
    for (int q = 0; q < NC; q++) put[q][threadIdx.x & 63] = T(0);
}
template <int NC, class T>
__device__ __forceinline__ void settle(T (*put)[kCol], int k, const T *u)
{
    const int e = ((threadIdx.x & 63) + k) & 63;
    T had[NC];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int q = 0; q < NC; q++) had[q] = put[q][e];
#pragma unroll
    for (int q = 0; q < NC; q++) put[q][e] = had[q] + u[q];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The 64 steps of a tile whose column c is stored at entries c and c + 64, so
// that column (l + k) mod 64 is entry l + k.  The columns' sums travel from
// lane to lane and are settled in `put`.
template <class T, class Op, int IPL, bool BOTH, int W>
__device__ __forceinline__ void sym_steps(const Op &op, const typename Word<T>::type (&tile)[W][2 * kCol],
                                          T (*put)[kCol], int col0, int row0,
                                          const T (&r)[IPL][Op::NV], T (&s)[IPL][Op::NC])
{
    constexpr int N = Word<T>::n, kStep = BOTH ? kSeg : kCol;
    const int lane = threadIdx.x & 63;
    T u[Op::NC];
#pragma unroll 1
    for (int k0 = 0; k0 < kCol; k0 += kStep) {
#pragma unroll
        for (int q = 0; q < Op::NC; q++) u[q] = T(0);
#pragma unroll 1
        for (int k = k0; k < k0 + kStep; k++) {
            T c[W * N], z[Op::NC];
#pragma unroll
            for (int w = 0; w < W; w++) {
                const auto e = tile[w][lane + k];
                const T *f = reinterpret_cast<const T *>(&e);
#pragma unroll
                for (int q = 0; q < N; q++) c[w * N + q] = f[q];
            }
            const int j = col0 + ((lane + k) & 63);
            op.template pair<BOTH, true>(r[0], c, j == row0 + lane, s[0], z);
#pragma unroll
            for (int q = 1; q < IPL; q++)
                op.template pair<BOTH, false>(r[q], c, j == row0 + lane + 64 * q, s[q], z);
            if (BOTH) {
#pragma unroll
                for (int q = 0; q < Op::NC; q++) u[q] = z[q] + from_next_lane(u[q]);
            }
        }
        if (BOTH) settle<Op::NC>(put, k0 + kStep - 1, u);
    }
}

// VALU-bound.  Each wave stages its own tiles (64 lanes load 64 columns once
// per 64 IPL steps' work) and the next tile's loads are under way during the
// steps, so the waves meet only to add up their row sums at the end.  The
// columns' sums rotate in registers: LDS float additions (ds_add_f32) in
// their place took 190 cycles each here (n = 16384 FP32 forward 1036 us
// against 154), ds_add_f64 cost the same as the rotation.
template <class T, class Op, int IPL>
__global__ void __launch_bounds__(kWG) k_sym(Plan p, Op op, double *__restrict__ rowpart,
                                             T *__restrict__ colpart)
{
    using V = typename Word<T>::type;
    constexpr int W = kWords<T, Op>, NC = Op::NC, R = kCol * IPL, N = Word<T>::n;
    __shared__ union {
        // each wave's own tile and its columns' sums, on 2 KB boundaries (with
        // an address register more the compiler takes the FP32 forward's two
        // rows one after the other: n = 8192 56.3 us, not 49.7)
        struct alignas(2048) {
            V tile[W][2 * kCol];
            T put[NC][kCol];
        } wave[kWaves];
        double sum[kWaves][NC][R];  // then the waves' row sums
    } sh;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int b = blockIdx.x / p.parts, u0 = (blockIdx.x - b * p.parts) * p.per;
    const int u1 = min(p.units(), u0 + p.per);
    const int row0 = b * R;
    // the first column of unit u's tile, or n where there is none
    auto column = [&](int u) {
        const int d = u / IPL, cb = b + d < p.nb ? b + d : b + d - p.nb;
        return u < u1 && (d == 0 || p.takes(b, d)) ? min(cb * R + (u % IPL) * kCol, p.n) : p.n;
    };
    T r[IPL][Op::NV], s[IPL][NC], pre[Op::NV];
    Long<T> tot[IPL][NC];
#pragma unroll
    for (int i = 0; i < IPL; i++) load_values<T, Op>(op, row0 + lane + kCol * i, p.n, r[i]);
    auto &tile = sh.wave[wave].tile;
    auto &put = sh.wave[wave].put;
    load_values<T, Op>(op, column(u0 + wave) + lane, p.n, pre);
    for (int u = u0 + wave; u < u1; u += kWaves) {
        const int col0 = column(u);
        if (col0 >= p.n) {  // beyond the last block's particles, or not this block's
            load_values<T, Op>(op, column(u + kWaves) + lane, p.n, pre);
            continue;
        }
        // the tile is the wave's own and its LDS operations are in order: the
        // fences only keep the compiler from moving them across each other
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int w = 0; w < W; w++) {
            V e;
            T *f = reinterpret_cast<T *>(&e);
#pragma unroll
            for (int k = 0; k < N; k++) f[k] = w * N + k < Op::NV ? pre[w * N + k] : T(0);
            tile[w][lane] = e;
            tile[w][lane + kCol] = e;
        }
        put_zero<NC>(put);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        load_values<T, Op>(op, column(u + kWaves) + lane, p.n, pre);
#pragma unroll
        for (int i = 0; i < IPL; i++)
#pragma unroll
            for (int k = 0; k < NC; k++) s[i][k] = T(0);
        if (u >= IPL)
            sym_steps<T, Op, IPL, true>(op, tile, put, col0, row0, r, s);
        else
            sym_steps<T, Op, IPL, false>(op, tile, put, col0, row0, r, s);
#pragma unroll
        for (int i = 0; i < IPL; i++)
#pragma unroll
            for (int k = 0; k < NC; k++) tot[i][k].add(s[i][k]);
        if (u >= IPL && col0 + lane < p.n) {
#pragma unroll
            for (int k = 0; k < NC; k++)
                colpart[p.col_at(u / IPL, NC, k, col0 + lane)] = put[k][lane];
        }
    }
    // the waves' row sums, added in wave order
    __syncthreads();
#pragma unroll
    for (int i = 0; i < IPL; i++)
#pragma unroll
        for (int k = 0; k < NC; k++) sh.sum[wave][k][lane + kCol * i] = tot[i][k].value();
    __syncthreads();
    for (int k = t; k < NC * R; k += kWG) {
        Long<double> z;
#pragma unroll
        for (int w = 0; w < kWaves; w++) z.add((&sh.sum[w][0][0])[k]);
        rowpart[p.row_at(blockIdx.x, NC, 0, 0) + k] = z.value();
    }
}

// Adds the records of (particle i, sum c): the columns' by distance of their
// row block, then those of its own block's workgroups.  HBM-bound.
template <class T, int NC>
__global__ void __launch_bounds__(256) k_sym_sum(Plan p, const double *__restrict__ rowpart,
                                                 const T *__restrict__ colpart,
                                                 T *__restrict__ o0, T *__restrict__ o1,
                                                 T *__restrict__ o2)
{
    const int i = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
    if (i >= p.n) return;
    const int b = i / p.rows;
    // with nb even, only the second half of the blocks is taken by the opposite one
    const int nd = p.nb / 2 - (p.nb % 2 == 0 && b < p.nb / 2 ? 1 : 0);
    Long<double> z;
#pragma unroll 8
    for (int d = 1; d <= nd; d++) z.add(double(colpart[p.col_at(d, NC, c, i)]));
#pragma unroll 8
    for (int k = 0; k < p.parts; k++)
        z.add(rowpart[p.row_at(b * p.parts + k, NC, c, i - b * p.rows)]);
    T *o = c < 3 ? o0 + 3 * size_t(i) + c : c < 6 ? o1 + 3 * size_t(i) + c - 3 : o2 + i;
    *o = T(z.value());
}

}  // namespace g6s
