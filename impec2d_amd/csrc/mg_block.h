// mg_block.h -- multigrid legs and the bottom of the V-cycle on 2 x 2 blocks of
// cells in LDS.
//
// One thread owns one 2 x 2 block: cell (r, c) of block (bi, bj) is the level's
// cell (2 bi + r, 2 bj + c).  A block holds one cell of each of the four
// colours of the 9-point operator (and two of each colour of the 5-point one),
// so a colour sweep leaves no lane idle, and the block is one cell of the next
// coarser level, so the restriction and the prolongation are block-local too.
// A thread keeps its cells, right-hand sides and coefficients in registers; LDS
// holds the cells as four planes, one per parity (r, c), so that the lanes of a
// wave read and write consecutive words, with a ring of one block around them
// that stays finite (its coefficients are zero).  A sweep of one colour reads
// only other colours, so one barrier per colour suffices.
//
// Names: W / E is the neighbour in row i - 1 / i + 1, S / N in column j - 1 / j + 1.
#pragma once
#include "impec_device.h"

namespace impec {

// cells of a P x P block array in LDS: plane (r, c), pitch P + 2, ring 1
template <int P>
struct BlkGeo {
    static constexpr int LD = P + 2, PLANE = LD * LD, CELLS = 4 * PLANE;
};

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the neighbour of cell (R, C) of the thread's block in direction (DI, DJ):
// from the block's registers x, or from LDS (o: the block's place in a plane)
template <int P, int R, int C, int DI, int DJ, typename T>
__device__ __forceinline__ T blk_nb(const T (&x)[4], const T *sm, int o) {
    constexpr int r = R + DI, c = C + DJ;
    constexpr int bi = r < 0 ? -1 : (r > 1 ? 1 : 0), bj = c < 0 ? -1 : (c > 1 ? 1 : 0);
    constexpr int cell = (r & 1) * 2 + (c & 1);
    if constexpr (bi == 0 && bj == 0) return x[cell];
    else return sm[cell * BlkGeo<P>::PLANE + o + bi * BlkGeo<P>::LD + bj];
}

// 9-point coefficients of a block's cells: the folded rows (zero outside the
// level), W SW S SE E NE N NW, and the reciprocal diagonals
template <typename T>
struct Co9 {
    T a[4][8], rc[4];
};

template <int P, int CELL, typename T>
__device__ __forceinline__ T off_sum(const Co9<T> &k, T s, const T (&x)[4], const T *sm, int o) {
#pragma clang fp contract(fast)
    constexpr int R = CELL >> 1, C = CELL & 1;
    const T (&a)[8] = k.a[CELL];
    s -= a[0] * blk_nb<P, R, C, -1, 0>(x, sm, o);
    s -= a[1] * blk_nb<P, R, C, -1, -1>(x, sm, o);
    s -= a[2] * blk_nb<P, R, C, 0, -1>(x, sm, o);
    s -= a[3] * blk_nb<P, R, C, 1, -1>(x, sm, o);
    s -= a[4] * blk_nb<P, R, C, 1, 0>(x, sm, o);
    s -= a[5] * blk_nb<P, R, C, 1, 1>(x, sm, o);
    s -= a[6] * blk_nb<P, R, C, 0, 1>(x, sm, o);
    s -= a[7] * blk_nb<P, R, C, -1, 1>(x, sm, o);
    return s;
}

// 5-point coefficients of a block's cells: the face of each cell towards each
// neighbour (zero on the boundary of the level)
template <typename T>
struct Co5 {
    T W[2], E[2], S[2], N[2];   // outward faces: of cells (0, c), (1, c), (r, 0), (r, 1)
    T iE[2], iN[2];             // inner faces: between (0, c) and (1, c), between (r, 0) and (r, 1)
    T rc[4];
    template <int CELL> __device__ __forceinline__ T w() const { return CELL < 2 ? W[CELL & 1] : iE[CELL & 1]; }
    template <int CELL> __device__ __forceinline__ T e() const { return CELL < 2 ? iE[CELL & 1] : E[CELL & 1]; }
    template <int CELL> __device__ __forceinline__ T s() const { return (CELL & 1) ? iN[CELL >> 1] : S[CELL >> 1]; }
    template <int CELL> __device__ __forceinline__ T n() const { return (CELL & 1) ? N[CELL >> 1] : iN[CELL >> 1]; }
    template <int CELL> __device__ __forceinline__ T diag() const {
        return -((w<CELL>() + e<CELL>()) + (s<CELL>() + n<CELL>()));
    }
};

template <int P, int CELL, typename T>
__device__ __forceinline__ T off_sum(const Co5<T> &k, T s, const T (&x)[4], const T *sm, int o) {
#pragma clang fp contract(fast)
    constexpr int R = CELL >> 1, C = CELL & 1;
    s -= k.template w<CELL>() * blk_nb<P, R, C, -1, 0>(x, sm, o);
    s -= k.template s<CELL>() * blk_nb<P, R, C, 0, -1>(x, sm, o);
    s -= k.template e<CELL>() * blk_nb<P, R, C, 1, 0>(x, sm, o);
    s -= k.template n<CELL>() * blk_nb<P, R, C, 0, 1>(x, sm, o);
    return s;
}

// one Gauss-Seidel update of cell CELL, into the registers and LDS
template <int P, int CELL, typename Co, typename T>
__device__ __forceinline__ void blk_gs(const Co &k, const T (&b)[4], T (&x)[4], T *sm, int o) {
    x[CELL] = off_sum<P, CELL>(k, b[CELL], x, sm, o) * k.rc[CELL];
    sm[CELL * BlkGeo<P>::PLANE + o] = x[CELL];
}

// a colour of the operator's ordering: one cell per colour for the 9-point
// operator, the red pair (0, 0), (1, 1) and the black pair for the 5-point one
template <int P, int COL, typename T>
__device__ __forceinline__ void blk_colour(const Co9<T> &k, const T (&b)[4], T (&x)[4], T *sm, int o) {
    blk_gs<P, COL>(k, b, x, sm, o);
}
template <int P, int COL, typename T>
__device__ __forceinline__ void blk_colour(const Co5<T> &k, const T (&b)[4], T (&x)[4], T *sm, int o) {
    blk_gs<P, (COL == 0 ? 0 : 1)>(k, b, x, sm, o);
    blk_gs<P, (COL == 0 ? 3 : 2)>(k, b, x, sm, o);
}
template <typename Co> struct Colours;
template <typename T> struct Colours<Co9<T>> { static constexpr int N = 4; };
template <typename T> struct Colours<Co5<T>> { static constexpr int N = 2; };

// the workgroup's barrier, or the wave's where one wave holds the level
template <bool WAVE_ONLY>
__device__ __forceinline__ void blk_sync() {
    if constexpr (WAVE_ONLY) wave_sync();
    else __syncthreads();
}

// `ns` sweeps over the colours, ascending (down leg) or descending (up leg);
// a barrier after every colour
template <int P, bool UP, bool W1, typename Co, typename T>
__device__ __forceinline__ void blk_sweeps(const Co &k, const T (&b)[4], T (&x)[4], T *sm, int o, bool act, int ns) {
    for (int q = 0; q < ns; q++) {
        if constexpr (Colours<Co>::N == 4) {
            if (act) blk_colour<P, UP ? 3 : 0>(k, b, x, sm, o);
            blk_sync<W1>();
            if (act) blk_colour<P, UP ? 2 : 1>(k, b, x, sm, o);
            blk_sync<W1>();
            if (act) blk_colour<P, UP ? 1 : 2>(k, b, x, sm, o);
            blk_sync<W1>();
            if (act) blk_colour<P, UP ? 0 : 3>(k, b, x, sm, o);
            blk_sync<W1>();
        } else {
            if (act) blk_colour<P, UP ? 1 : 0>(k, b, x, sm, o);
            blk_sync<W1>();
            if (act) blk_colour<P, UP ? 0 : 1>(k, b, x, sm, o);
            blk_sync<W1>();
        }
    }
}

// residuals of the block's cells; c: the diagonals
template <int P, typename Co, typename T>
__device__ __forceinline__ void blk_residual(const Co &k, const T (&c)[4], const T (&b)[4], const T (&x)[4],
                                             const T *sm, int o, T (&r)[4]) {
#pragma clang fp contract(fast)
    r[0] = off_sum<P, 0>(k, b[0], x, sm, o) - c[0] * x[0];
    r[1] = off_sum<P, 1>(k, b[1], x, sm, o) - c[1] * x[1];
    r[2] = off_sum<P, 2>(k, b[2], x, sm, o) - c[2] * x[2];
    r[3] = off_sum<P, 3>(k, b[3], x, sm, o) - c[3] * x[3];
}

// weights of the fine cells 2 I - 1 .. 2 I + 2 in coarse cell I (the transpose
// of the cell-centred bilinear prolongation with constant extrapolation at the
// ends), zero outside the fine level of n cells
template <typename T>
__device__ __forceinline__ void rest_weights(int I, int n, int m, T (&w)[4]) {
    w[0] = I > 0 ? T(0.25) : T(0);
    w[1] = I == 0 ? T(1) : T(0.75);
    w[2] = 2 * I + 1 < n ? (I == m - 1 ? T(1) : T(0.75)) : T(0);
    w[3] = 2 * I + 2 < n ? T(0.25) : T(0);
}

// full weighting of the residual planes sm into the block's coarse cell
template <int P, typename T>
__device__ __forceinline__ T blk_restrict(const T (&r)[4], const T *sm, int o, const T (&wi)[4], const T (&wj)[4]) {
#pragma clang fp contract(fast)
    T acc = T(0);
    auto row = [&](auto rr, int q) {   // fine row 2 I + rr: its four columns
        constexpr int RR = decltype(rr)::value;
        const T rL = blk_nb<P, 0, 0, RR, -1>(r, sm, o), r0 = blk_nb<P, 0, 0, RR, 0>(r, sm, o);
        const T r1 = blk_nb<P, 0, 0, RR, 1>(r, sm, o), rR = blk_nb<P, 0, 0, RR, 2>(r, sm, o);
        acc += wi[q] * (((wj[0] * rL + wj[1] * r0) + wj[2] * r1) + wj[3] * rR);
    };
    row(std::integral_constant<int, -1>{}, 0);
    row(std::integral_constant<int, 0>{}, 1);
    row(std::integral_constant<int, 1>{}, 2);
    row(std::integral_constant<int, 2>{}, 3);
    return T(0.25) * acc;
}

// x += P e: e[a][b] the coarse cells (bi - 1 + a, bj - 1 + b), clamped
template <typename T>
__device__ __forceinline__ void blk_prolong(const T (&e)[3][3], T (&x)[4]) {
#pragma clang fp contract(fast)
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int a = r ? 2 : 0, b = c ? 2 : 0;
            x[r * 2 + c] += T(0.5625) * e[1][1] + T(0.1875) * e[1][b] + T(0.1875) * e[a][1] + T(0.0625) * e[a][b];
        }
}

// ---------------------------------------------------------------------------
// legs of the 9-point V-cycle: one launch per leg and level
//
// A tile is P x P blocks (P = 32: 64 x 64 cells, one workgroup of 1024 threads),
// of which the middle 26 x 22 are written on the way down and 28 x 24 on the way
// up; a sweep of one kernel per colour took eleven launches per leg and level,
// each a latency of about 4.5 us whatever its size.  The legs are bound by that
// latency, the first loads and the eight barriers of the sweeps: 7.6-9 us at 71^2
// and 283^2, 9.5 / 11.6 us at 141^2 and 14.6 / 14.9 us at 566^2 (two sweeps)
// against 50-60 us for the separate kernels; 4.5 ms per time step against 28 at
// 141^2 (39 iterations), 6.0 against 17.7 ms at 566^2.  Coefficients are read
// (80 B per cell from the caches) rather than formed from the mobilities: eight
// divisions per cell and leg would cost more.
// ---------------------------------------------------------------------------
// the assembled operator of a level: plane k of stencil order {C, W, SW, S, SE,
// E, NE, N, NW} (k < 9) and the reciprocal diagonal (k = 9), cell (i, j) of a
// plane at i * ld + j; ld even, planes zero outside the level
template <typename T>
struct OpPlanes {
    const T *a;
    long plane;
    int ld;
};

template <typename T>
struct Pair {
    T a, b;
};

template <typename T>
__device__ __forceinline__ void load_co9(const OpPlanes<T> &A, int bi, int bj, Co9<T> &k) {
    const T *p = A.a + (long)(2 * bi) * A.ld + 2 * bj;
#pragma unroll
    for (int q = 0; q < 9; q++)
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const Pair<T> v = *reinterpret_cast<const Pair<T> *>(__builtin_assume_aligned(p + (q + 1) * A.plane + (long)r * A.ld, 2 * sizeof(T)));
            if (q < 8) {
                k.a[2 * r][q] = v.a;
                k.a[2 * r + 1][q] = v.b;
            } else {
                k.rc[2 * r] = v.a;
                k.rc[2 * r + 1] = v.b;
            }
        }
}
template <typename T>
__device__ __forceinline__ void load_diag9(const OpPlanes<T> &A, int bi, int bj, T (&c)[4]) {
    const T *p = A.a + (long)(2 * bi) * A.ld + 2 * bj;
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const Pair<T> v = *reinterpret_cast<const Pair<T> *>(__builtin_assume_aligned(p + (long)r * A.ld, 2 * sizeof(T)));
        c[2 * r] = v.a;
        c[2 * r + 1] = v.b;
    }
}

// blocks by which a tile's cells lose validity from its edges, down leg
// (sweeps from a zero guess, residual, full weighting) and up leg (sweeps): a
// sweep of the 9-point ordering reaches 2 rows and 4 columns
template <int NS> struct Halo9;
template <> struct Halo9<1> { static constexpr int DI = 2, DJ = 3, UI = 1, UJ = 2; };
template <> struct Halo9<2> { static constexpr int DI = 3, DJ = 5, UI = 2, UJ = 4; };

// tiles of P blocks over nb blocks with a halo of H: tile k covers the blocks
// from tile_origin and writes those of [tile_lo, tile_hi)
__host__ __device__ __forceinline__ int tile_count(int nb, int P, int H) {
    return nb <= P ? 1 : (nb - 2 * H + (P - 2 * H) - 1) / (P - 2 * H);
}
__device__ __forceinline__ int tile_origin(int k, int nb, int P, int H) {
    const int o = k * (P - 2 * H);
    return o + P <= nb ? o : (nb > P ? nb - P : 0);
}
__device__ __forceinline__ int tile_lo(int k, int P, int H) { return k == 0 ? 0 : k * (P - 2 * H) + H; }
__device__ __forceinline__ int tile_hi(int k, int n, int nb, int P, int H) {
    return k == n - 1 ? nb : (k + 1) * (P - 2 * H) + H;
}

// one leg over one level; level arrays at cell (0, 0) with pitch ld
struct Leg9Args {
    OpPlanes<double> A;
    int n1, n2, ld;
    const double *b;      // right-hand side (level 0: the CG residual)
    const double *S;      // level 0: b - S[S_RSUM] inv_n
    double inv_n;
    double *x;            // down: written; up: read
    double *xo;           // up: written
    double *bc;           // down: the coarser level's right-hand side
    const double *xc;     // up: its solution
    int m1, m2, ldc;
    int ti, tj;           // tiles per direction
    double *part;         // up at level 0: partials of sum x and r x per workgroup
};

template <int P, int NS, bool FINE0>
__global__ void __launch_bounds__(P *P) k_mg9_down(Leg9Args A) {
    using G = BlkGeo<P>;
    using H = Halo9<NS>;
    __shared__ double sm[G::CELLS];
    const int t = threadIdx.x;
    const int ki = blockIdx.x / A.tj, kj = blockIdx.x - ki * A.tj;
    const int nb1 = (A.n1 + 1) >> 1, nb2 = (A.n2 + 1) >> 1;
    const int li = t / P, lj = t % P;
    const int bi = tile_origin(ki, nb1, P, H::DI) + li, bj = tile_origin(kj, nb2, P, H::DJ) + lj;
    const bool act = bi < nb1 && bj < nb2;
    const int o = (li + 1) * G::LD + lj + 1;
    Co9<double> k;
    double b[4], x[4] = {0., 0., 0., 0.};
    if (act) {
        load_co9(A.A, bi, bj, k);
        const double mean = FINE0 ? A.S[S_RSUM] * A.inv_n : 0.;
        const double *bp = A.b + (long)(2 * bi) * A.ld + 2 * bj;
        const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
        b[0] = bp[0] - mean;
        b[1] = v1 ? bp[1] - mean : 0.;
        b[2] = w1 ? bp[A.ld] - mean : 0.;
        b[3] = v1 && w1 ? bp[A.ld + 1] - mean : 0.;
    }
    for (int q = t; q < G::CELLS; q += P * P) sm[q] = 0.;
    __syncthreads();
    blk_sweeps<P, false, false>(k, b, x, sm, o, act, NS);
    double r[4] = {0., 0., 0., 0.};
    if (act) {
        double c[4];
        load_diag9(A.A, bi, bj, c);
        blk_residual<P>(k, c, b, x, sm, o, r);
    }
    __syncthreads();   // the planes now take the residual
    if (act)
#pragma unroll
        for (int q = 0; q < 4; q++) sm[q * G::PLANE + o] = r[q];
    __syncthreads();
    const bool out = act && bi >= tile_lo(ki, P, H::DI) && bi < tile_hi(ki, A.ti, nb1, P, H::DI) &&
                     bj >= tile_lo(kj, P, H::DJ) && bj < tile_hi(kj, A.tj, nb2, P, H::DJ);
    if (out) {
        double wi[4], wj[4];
        rest_weights(bi, A.n1, A.m1, wi);
        rest_weights(bj, A.n2, A.m2, wj);
        A.bc[(long)bi * A.ldc + bj] = blk_restrict<P>(r, sm, o, wi, wj);
        double *xp = A.x + (long)(2 * bi) * A.ld + 2 * bj;
        const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
        xp[0] = x[0];
        if (v1) xp[1] = x[1];
        if (w1) xp[A.ld] = x[2];
        if (v1 && w1) xp[A.ld + 1] = x[3];
    }
}

template <int P, int NS, bool FINE0>
__global__ void __launch_bounds__(P *P) k_mg9_up(Leg9Args A) {
    using G = BlkGeo<P>;
    using H = Halo9<NS>;
    __shared__ double sm[G::CELLS];
    const int t = threadIdx.x;
    const int ki = blockIdx.x / A.tj, kj = blockIdx.x - ki * A.tj;
    const int nb1 = (A.n1 + 1) >> 1, nb2 = (A.n2 + 1) >> 1;
    const int li = t / P, lj = t % P;
    const int bi = tile_origin(ki, nb1, P, H::UI) + li, bj = tile_origin(kj, nb2, P, H::UJ) + lj;
    const bool act = bi < nb1 && bj < nb2;
    const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
    const int o = (li + 1) * G::LD + lj + 1;
    Co9<double> k;
    const double mean = FINE0 ? A.S[S_RSUM] * A.inv_n : 0.;
    double b[4], x[4] = {0., 0., 0., 0.};
    for (int q = t; q < G::CELLS; q += P * P) sm[q] = 0.;
    if (act) {
        load_co9(A.A, bi, bj, k);
        const long c0 = (long)(2 * bi) * A.ld + 2 * bj;
        const double *bp = A.b + c0, *xp = A.x + c0;
        b[0] = bp[0] - mean;
        b[1] = v1 ? bp[1] - mean : 0.;
        b[2] = w1 ? bp[A.ld] - mean : 0.;
        b[3] = v1 && w1 ? bp[A.ld + 1] - mean : 0.;
        x[0] = xp[0];
        if (v1) x[1] = xp[1];
        if (w1) x[2] = xp[A.ld];
        if (v1 && w1) x[3] = xp[A.ld + 1];
        double e[3][3];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const int I = bi + q - 1 < 0 ? 0 : (bi + q - 1 > A.m1 - 1 ? A.m1 - 1 : bi + q - 1);
                const int J = bj + p - 1 < 0 ? 0 : (bj + p - 1 > A.m2 - 1 ? A.m2 - 1 : bj + p - 1);
                e[q][p] = A.xc[(long)I * A.ldc + J];
            }
        blk_prolong(e, x);
    }
    __syncthreads();
    if (act)
#pragma unroll
        for (int q = 0; q < 4; q++) sm[q * G::PLANE + o] = x[q];
    __syncthreads();
    blk_sweeps<P, true, false>(k, b, x, sm, o, act, NS);
    const bool out = act && bi >= tile_lo(ki, P, H::UI) && bi < tile_hi(ki, A.ti, nb1, P, H::UI) &&
                     bj >= tile_lo(kj, P, H::UJ) && bj < tile_hi(kj, A.tj, nb2, P, H::UJ);
    double s[2] = {0., 0.};
    if (out) {
        double *xp = A.xo + (long)(2 * bi) * A.ld + 2 * bj;
        const double *rp = A.b + (long)(2 * bi) * A.ld + 2 * bj;
        auto put = [&](int q, long at) {
            xp[at] = x[q];
            if (FINE0) {
                s[0] += x[q];
                s[1] += rp[at] * x[q];
            }
        };
        put(0, 0);
        if (v1) put(1, 1);
        if (w1) put(2, A.ld);
        if (v1 && w1) put(3, A.ld + 1);
    }
    if (FINE0) {
        block_reduce<RED_SUM, 2>(s);
        if (t == 0) {
            A.part[blockIdx.x] = s[0];
            A.part[RED_BLOCKS + blockIdx.x] = s[1];
        }
    }
}

// ---------------------------------------------------------------------------
// the bottom of the 9-point V-cycle: from the first level of at most 64 x 64
// cells down to the coarsest and back up in one workgroup.  Depth D holds a
// level of at most 64 >> D cells a side on (32 >> D)^2 threads; from depth 2 on
// one wave does the work and needs no workgroup barrier.  24-26 us per cycle, in
// place of 20 launches per level on six levels (about 500 us).
// ---------------------------------------------------------------------------
constexpr int BOT9_DEPTHS = 6;   // 64, 32, 16, 8, 4, 2 cells a side
struct Bot9Args {
    int d0, nl;                  // depth of the first level; levels
    struct {
        OpPlanes<double> A;
        int n1, n2;
    } lev[BOT9_DEPTHS];
    const double *inv;           // the coarsest level's solution operator, n x n (k_op9_coarsest)
    const double *b;             // right-hand side of the first level at (0, 0)
    double *out;                 // its solution
    int ldb, ldo;
};

template <int D>
struct Bot9Sm {   // offsets of depth D in the LDS arrays
    static constexpr int P = 32 >> D;
    static constexpr int X = D == 0 ? 0 : Bot9Sm<(D > 0 ? D - 1 : 0)>::X + BlkGeo<(64 >> D)>::CELLS;
    static constexpr int B = D <= 1 ? 0 : Bot9Sm<(D > 0 ? D - 1 : 0)>::B + 4 * (64 >> D) * (64 >> D);
};
constexpr int BOT9_X = Bot9Sm<5>::X + BlkGeo<1>::CELLS, BOT9_B = Bot9Sm<5>::B + 4;

template <int D, int NS>
__device__ __forceinline__ void bot9_down(const Bot9Args &A, double *sx, double *sr, double *sb) {
    constexpr int P = 32 >> D;
    constexpr bool W1 = P * P <= 64;
    using G = BlkGeo<P>;
    if (D < A.d0 || D - A.d0 + 1 >= A.nl) return;
    const auto &L = A.lev[D - A.d0], &Lc = A.lev[D - A.d0 + 1];
    const int t = threadIdx.x, bi = t / P, bj = t % P;
    const bool act = t < P * P && 2 * bi < L.n1 && 2 * bj < L.n2;
    const int o = (bi + 1) * G::LD + bj + 1;
    double *sm = sx + Bot9Sm<D>::X;
    Co9<double> k;
    double b[4], x[4] = {0., 0., 0., 0.}, r[4] = {0., 0., 0., 0.};
    if (act) {
        load_co9(L.A, bi, bj, k);
        if (D == A.d0) {
            const double *bp = A.b + (long)(2 * bi) * A.ldb + 2 * bj;
            const bool v1 = 2 * bj + 1 < L.n2, w1 = 2 * bi + 1 < L.n1;
            b[0] = bp[0];
            b[1] = v1 ? bp[1] : 0.;
            b[2] = w1 ? bp[A.ldb] : 0.;
            b[3] = v1 && w1 ? bp[A.ldb + 1] : 0.;
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) b[q] = sb[Bot9Sm<D>::B + q * P * P + t];
        }
    }
    blk_sweeps<P, false, W1>(k, b, x, sm, o, act, NS);
    if (act) {
        double c[4];
        load_diag9(L.A, bi, bj, c);
        blk_residual<P>(k, c, b, x, sm, o, r);
#pragma unroll
        for (int q = 0; q < 4; q++) sr[q * G::PLANE + o] = r[q];
    }
    blk_sync<W1>();
    // the coarse cell (bi, bj) is cell (bi & 1, bj & 1) of block (bi / 2, bj / 2)
    if (act) {
        double wi[4], wj[4];
        rest_weights(bi, L.n1, Lc.n1, wi);
        rest_weights(bj, L.n2, Lc.n2, wj);
        constexpr int PC = P / 2 > 0 ? P / 2 : 1;
        sb[Bot9Sm<D + 1>::B + ((bi & 1) * 2 + (bj & 1)) * PC * PC + (bi >> 1) * PC + (bj >> 1)] =
            blk_restrict<P>(r, sr, o, wi, wj);
    }
}

template <int D, int NS>
__device__ __forceinline__ void bot9_up(const Bot9Args &A, double *sx, double *sr, double *sb) {
    constexpr int P = 32 >> D;
    constexpr bool W1 = P * P <= 64;
    using G = BlkGeo<P>;
    if (D < A.d0 || D - A.d0 + 1 >= A.nl) return;
    const auto &L = A.lev[D - A.d0], &Lc = A.lev[D - A.d0 + 1];
    const int t = threadIdx.x, bi = t / P, bj = t % P;
    const bool act = t < P * P && 2 * bi < L.n1 && 2 * bj < L.n2;
    const int o = (bi + 1) * G::LD + bj + 1;
    double *sm = sx + Bot9Sm<D>::X;
    Co9<double> k;
    double b[4], x[4] = {0., 0., 0., 0.};
    if (act) {
        load_co9(L.A, bi, bj, k);
        if (D == A.d0) {
            const double *bp = A.b + (long)(2 * bi) * A.ldb + 2 * bj;
            const bool v1 = 2 * bj + 1 < L.n2, w1 = 2 * bi + 1 < L.n1;
            b[0] = bp[0];
            b[1] = v1 ? bp[1] : 0.;
            b[2] = w1 ? bp[A.ldb] : 0.;
            b[3] = v1 && w1 ? bp[A.ldb + 1] : 0.;
        } else {
#pragma unroll
            for (int q = 0; q < 4; q++) b[q] = sb[Bot9Sm<D>::B + q * P * P + t];
        }
        constexpr int PC = P / 2 > 0 ? P / 2 : 1;
        using GC = BlkGeo<PC>;
        const double *sc = sx + Bot9Sm<D + 1>::X;
        double e[3][3];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const int I = bi + q - 1 < 0 ? 0 : (bi + q - 1 > Lc.n1 - 1 ? Lc.n1 - 1 : bi + q - 1);
                const int J = bj + p - 1 < 0 ? 0 : (bj + p - 1 > Lc.n2 - 1 ? Lc.n2 - 1 : bj + p - 1);
                e[q][p] = sc[((I & 1) * 2 + (J & 1)) * GC::PLANE + ((I >> 1) + 1) * GC::LD + (J >> 1) + 1];
            }
#pragma unroll
        for (int q = 0; q < 4; q++) x[q] = sm[q * G::PLANE + o];
        blk_prolong(e, x);
#pragma unroll
        for (int q = 0; q < 4; q++) sm[q * G::PLANE + o] = x[q];
    }
    blk_sync<W1>();
    blk_sweeps<P, true, W1>(k, b, x, sm, o, act, NS);
    if (D == A.d0 && act) {
        double *xp = A.out + (long)(2 * bi) * A.ldo + 2 * bj;
        const bool v1 = 2 * bj + 1 < L.n2, w1 = 2 * bi + 1 < L.n1;
        xp[0] = x[0];
        if (v1) xp[1] = x[1];
        if (w1) xp[A.ldo] = x[2];
        if (v1 && w1) xp[A.ldo + 1] = x[3];
    }
}

template <int NS>
__global__ void __launch_bounds__(1024) k_mg9_bottom(Bot9Args A) {
    __shared__ double sx[BOT9_X], sb[BOT9_B], sr[BlkGeo<32>::CELLS];
    const int t = threadIdx.x;
    for (int q = t; q < BOT9_X; q += blockDim.x) sx[q] = 0.;
    for (int q = t; q < BlkGeo<32>::CELLS; q += blockDim.x) sr[q] = 0.;
    for (int q = t; q < BOT9_B; q += blockDim.x) sb[q] = 0.;
    __syncthreads();
    bot9_down<0, NS>(A, sx, sr, sb);
    __syncthreads();
    bot9_down<1, NS>(A, sx, sr, sb);
    __syncthreads();
    if (t < 64) {
        bot9_down<2, NS>(A, sx, sr, sb);
        wave_sync();
        bot9_down<3, NS>(A, sx, sr, sb);
        wave_sync();
        bot9_down<4, NS>(A, sx, sr, sb);
        wave_sync();
        {   // the coarsest level, at most 2 x 2 cells: x = inv b, cell (r, c) on lane 2 r + c
            const auto &L = A.lev[A.nl - 1];
            const int r = t >> 1, c = t & 1;
            if (t < 4 && r < L.n1 && c < L.n2) {
                const int n = L.n1 * L.n2, row = r * L.n2 + c;
                double s = 0.;
                for (int q = 0; q < n; q++)
                    s += A.inv[row * n + q] * sb[Bot9Sm<5>::B + (q / L.n2) * 2 + q % L.n2];
                sx[Bot9Sm<5>::X + t * BlkGeo<1>::PLANE + BlkGeo<1>::LD + 1] = s;
            }
        }
        wave_sync();
        bot9_up<4, NS>(A, sx, sr, sb);
        wave_sync();
        bot9_up<3, NS>(A, sx, sr, sb);
        wave_sync();
        bot9_up<2, NS>(A, sx, sr, sb);
    }
    __syncthreads();
    bot9_up<1, NS>(A, sx, sr, sb);
    __syncthreads();
    bot9_up<0, NS>(A, sx, sr, sb);
}

}  // namespace impec
