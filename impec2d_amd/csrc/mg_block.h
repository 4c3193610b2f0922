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
#include <type_traits>

namespace impec {

// Gaussian elimination with partial pivoting, then back substitution, of a
// bordered system of n = N cells: M holds the (N+1) x (N+1) matrix and, in
// column N+1, the right-hand side; sol receives the N+1 unknowns.  The sizes
// are compile-time constants and every loop is unrolled, so M stays in
// registers (with a run-time size it lives in scratch memory and each of the
// elimination's dependent accesses is a memory round trip).  The pivot row is
// exchanged by selects over the candidate rows, which keeps every index
// static.  FUSED: the updates rounded once, as fused multiply-adds; otherwise
// as a rounded product and a rounded difference.
template <int N, bool FUSED>
__device__ __forceinline__ void bordered_solve(double (&M)[N + 1][N + 2], double (&sol)[N + 1]) {
    constexpr int m = N + 1;
#pragma unroll
    for (int col = 0; col < m; col++) {
        int piv = col;
        double best = fabs(M[col][col]);
#pragma unroll
        for (int r = col + 1; r < m; r++) {
            const double a = fabs(M[r][col]);
            if (a > best) { piv = r; best = a; }
        }
#pragma unroll
        for (int r = col + 1; r < m; r++) {
            const bool sw = piv == r;
#pragma unroll
            for (int q = 0; q <= m; q++) {
                const double a = M[col][q], b = M[r][q];
                M[col][q] = sw ? b : a;
                M[r][q] = sw ? a : b;
            }
        }
        const double d = M[col][col];
        if (d == 0.) continue;
#pragma unroll
        for (int r = col + 1; r < m; r++) {
            const double f = M[r][col] / d;
#pragma unroll
            for (int q = col; q <= m; q++) M[r][q] = FUSED ? fma(-f, M[col][q], M[r][q]) : M[r][q] - f * M[col][q];
        }
    }
#pragma unroll
    for (int r = m - 1; r >= 0; r--) {
        double t = M[r][m];
#pragma unroll
        for (int q = r + 1; q < m; q++) t = FUSED ? fma(-M[r][q], sol[q], t) : t - M[r][q] * sol[q];
        sol[r] = M[r][r] != 0. ? t / M[r][r] : 0.;
    }
}

// a P x P block array in LDS: pitch of the blocks of a plane (ring 1) and size
// of a plane
template <int P>
struct BlkGeo {
    static constexpr int LD = P + 2, PLANE = LD * LD, CELLS = 4 * PLANE;
};

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the neighbour of cell (R, C) of the thread's block in direction (DI, DJ):
// from the block's registers x, or from LDS (G: the geometry of the planes, o:
// the block's place in a plane)
template <typename G, int R, int C, int DI, int DJ, typename T>
__device__ __forceinline__ T blk_nb(const T (&x)[4], const T *sm, int o) {
    constexpr int r = R + DI, c = C + DJ;
    constexpr int bi = r < 0 ? -1 : (r > 1 ? 1 : 0), bj = c < 0 ? -1 : (c > 1 ? 1 : 0);
    constexpr int cell = (r & 1) * 2 + (c & 1);
    if constexpr (bi == 0 && bj == 0) return x[cell];
    else return sm[cell * G::PLANE + o + bi * G::LD + bj];
}

// 9-point coefficients of a block's cells: the folded rows (zero outside the
// level), W SW S SE E NE N NW, and the reciprocal diagonals
template <typename T>
struct Co9 {
    T a[4][8], rc[4];
};

template <typename G, int CELL, typename T>
__device__ __forceinline__ T off_sum(const Co9<T> &k, T s, const T (&x)[4], const T *sm, int o) {
#pragma clang fp contract(fast)
    constexpr int R = CELL >> 1, C = CELL & 1;
    const T (&a)[8] = k.a[CELL];
    s -= a[0] * blk_nb<G, R, C, -1, 0>(x, sm, o);
    s -= a[1] * blk_nb<G, R, C, -1, -1>(x, sm, o);
    s -= a[2] * blk_nb<G, R, C, 0, -1>(x, sm, o);
    s -= a[3] * blk_nb<G, R, C, 1, -1>(x, sm, o);
    s -= a[4] * blk_nb<G, R, C, 1, 0>(x, sm, o);
    s -= a[5] * blk_nb<G, R, C, 1, 1>(x, sm, o);
    s -= a[6] * blk_nb<G, R, C, 0, 1>(x, sm, o);
    s -= a[7] * blk_nb<G, R, C, -1, 1>(x, sm, o);
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

template <typename G, int CELL, typename T>
__device__ __forceinline__ T off_sum(const Co5<T> &k, T s, const T (&x)[4], const T *sm, int o) {
#pragma clang fp contract(fast)
    constexpr int R = CELL >> 1, C = CELL & 1;
    s -= k.template w<CELL>() * blk_nb<G, R, C, -1, 0>(x, sm, o);
    s -= k.template s<CELL>() * blk_nb<G, R, C, 0, -1>(x, sm, o);
    s -= k.template e<CELL>() * blk_nb<G, R, C, 1, 0>(x, sm, o);
    s -= k.template n<CELL>() * blk_nb<G, R, C, 0, 1>(x, sm, o);
    return s;
}

// one Gauss-Seidel update of cell CELL, into the registers and LDS
template <typename G, int CELL, typename Co, typename T>
__device__ __forceinline__ void blk_gs(const Co &k, const T (&b)[4], T (&x)[4], T *sm, int o) {
    x[CELL] = off_sum<G, CELL>(k, b[CELL], x, sm, o) * k.rc[CELL];
    sm[CELL * G::PLANE + o] = x[CELL];
}

// a colour of the operator's ordering: one cell per colour for the 9-point
// operator, the red pair (0, 0), (1, 1) and the black pair for the 5-point one
template <typename G, int COL, typename T>
__device__ __forceinline__ void blk_colour(const Co9<T> &k, const T (&b)[4], T (&x)[4], T *sm, int o) {
    blk_gs<G, COL>(k, b, x, sm, o);
}
template <typename G, int COL, typename T>
__device__ __forceinline__ void blk_colour(const Co5<T> &k, const T (&b)[4], T (&x)[4], T *sm, int o) {
    blk_gs<G, (COL == 0 ? 0 : 1)>(k, b, x, sm, o);
    blk_gs<G, (COL == 0 ? 3 : 2)>(k, b, x, sm, o);
}
template <typename Co> struct Colours;
template <typename T> struct Colours<Co9<T>> { static constexpr int N = 4; };
template <typename T> struct Colours<Co5<T>> { static constexpr int N = 2; };

// the workgroup's barrier, or the wave's where one wave holds the level
__device__ __forceinline__ void blk_sync(bool workgroup) {
    if (workgroup) __syncthreads();
    else wave_sync();
}

// `ns` sweeps over the colours, ascending (down leg) or descending (up leg);
// a barrier after every colour
template <typename G, bool UP, typename Co, typename T>
__device__ __forceinline__ void blk_sweeps(const Co &k, const T (&b)[4], T (&x)[4], T *sm, int o, bool act, int ns,
                                           bool workgroup) {
    for (int q = 0; q < ns; q++) {
        if constexpr (Colours<Co>::N == 4) {
            if (act) blk_colour<G, UP ? 3 : 0>(k, b, x, sm, o);
            blk_sync(workgroup);
            if (act) blk_colour<G, UP ? 2 : 1>(k, b, x, sm, o);
            blk_sync(workgroup);
            if (act) blk_colour<G, UP ? 1 : 2>(k, b, x, sm, o);
            blk_sync(workgroup);
            if (act) blk_colour<G, UP ? 0 : 3>(k, b, x, sm, o);
            blk_sync(workgroup);
        } else {
            if (act) blk_colour<G, UP ? 1 : 0>(k, b, x, sm, o);
            blk_sync(workgroup);
            if (act) blk_colour<G, UP ? 0 : 1>(k, b, x, sm, o);
            blk_sync(workgroup);
        }
    }
}

// residual of cell CELL; c: the diagonal
template <typename G, int CELL, typename T>
__device__ __forceinline__ T cell_residual(const Co9<T> &k, T c, T b, const T (&x)[4], const T *sm, int o) {
#pragma clang fp contract(fast)
    return off_sum<G, CELL>(k, b, x, sm, o) - c * x[CELL];
}
template <typename G, int CELL, typename T>
__device__ __forceinline__ T cell_residual(const Co5<T> &k, T c, T b, const T (&x)[4], const T *sm, int o) {
#pragma clang fp contract(fast)
    constexpr int R = CELL >> 1, C = CELL & 1;
    T s = c * x[CELL];
    s += k.template w<CELL>() * blk_nb<G, R, C, -1, 0>(x, sm, o);
    s += k.template s<CELL>() * blk_nb<G, R, C, 0, -1>(x, sm, o);
    s += k.template e<CELL>() * blk_nb<G, R, C, 1, 0>(x, sm, o);
    s += k.template n<CELL>() * blk_nb<G, R, C, 0, 1>(x, sm, o);
    return b - s;
}
template <typename G, typename Co, typename T>
__device__ __forceinline__ void blk_residual(const Co &k, const T (&c)[4], const T (&b)[4], const T (&x)[4],
                                             const T *sm, int o, T (&r)[4]) {
    r[0] = cell_residual<G, 0>(k, c[0], b[0], x, sm, o);
    r[1] = cell_residual<G, 1>(k, c[1], b[1], x, sm, o);
    r[2] = cell_residual<G, 2>(k, c[2], b[2], x, sm, o);
    r[3] = cell_residual<G, 3>(k, c[3], b[3], x, sm, o);
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
template <typename G, typename T>
__device__ __forceinline__ T blk_restrict(const T (&r)[4], const T *sm, int o, const T (&wi)[4], const T (&wj)[4]) {
#pragma clang fp contract(fast)
    T acc = T(0);
    auto row = [&](auto rr, int q) {   // fine row 2 I + rr: its four columns
        constexpr int RR = decltype(rr)::value;
        const T rL = blk_nb<G, 0, 0, RR, -1>(r, sm, o), r0 = blk_nb<G, 0, 0, RR, 0>(r, sm, o);
        const T r1 = blk_nb<G, 0, 0, RR, 1>(r, sm, o), rR = blk_nb<G, 0, 0, RR, 2>(r, sm, o);
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
    blk_sweeps<G, false>(k, b, x, sm, o, act, NS, true);
    double r[4] = {0., 0., 0., 0.};
    if (act) {
        double c[4];
        load_diag9(A.A, bi, bj, c);
        blk_residual<G>(k, c, b, x, sm, o, r);
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
        A.bc[(long)bi * A.ldc + bj] = blk_restrict<G>(r, sm, o, wi, wj);
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
    blk_sweeps<G, true>(k, b, x, sm, o, act, NS, true);
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
// the 5-point operator: faces formed from the mobility quantity w
// ---------------------------------------------------------------------------
// 1/d from the hardware reciprocal estimate refined by one Newton-Raphson
// step, r' = r + r (1 - d r).  Only the multigrid preconditioner uses it: its
// rounding differs from IEEE division but is the same every time for the same
// d, so the preconditioner stays a fixed linear operator.
__device__ __forceinline__ double recip(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, r, 1.);
    return fma(r, e, r);
}
__device__ __forceinline__ float recip(float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    const float e = fmaf(-d, r, 1.f);
    return fmaf(r, e, r);
}

// face mobility as face_mob, with recip in place of the division
template <typename T>
__device__ __forceinline__ T face_mob_pc(T wl, T wr, int harmonic) {
    return harmonic ? T(2) * recip(wl + wr) : T(0.5) * (wl + wr);
}

// the faces of block (bi, bj) of an n1 x n2 level from its cells' w and the
// eight cells around it: wu / wd the cells beyond the block in rows 2 bi - 1
// and 2 bi + 2, wl / wr those in columns 2 bj - 1 and 2 bj + 2.  Faces outside the
// level are dropped by a zero factor, not by a branch around them (twelve short
// branches cost four times the twelve reciprocals run together): their cells' w
// must be finite and, for the harmonic average, not zero.  The averaging
// procedure is chosen the same way, ch / s + cm s with one of the two zero; for
// the mean concentration the reciprocal is taken of 1, since the sum s of two
// cells without permeability is zero there, and the face is too.
template <typename T>
__device__ __forceinline__ void make_co5(const T (&w)[4], const T (&wu)[2], const T (&wd)[2], const T (&wl)[2],
                                         const T (&wr)[2], int bi, int bj, int n1, int n2, T cx, T cy, int hm,
                                         Co5<T> &k) {
#pragma clang fp contract(fast)
    const bool r1 = 2 * bi + 1 < n1, r2 = 2 * bi + 2 < n1, c1 = 2 * bj + 1 < n2, c2 = 2 * bj + 2 < n2;
    const bool u = bi > 0, l = bj > 0;
    auto face = [&](T a, T b, T c, bool in) {
        const T f = in ? c : T(0), s = a + b;
        const T fh = hm ? T(2) * f : T(0), fm = hm ? T(0) : T(0.5) * f;
        return fh * recip(hm ? s : T(1)) + fm * s;
    };
    k.W[0] = face(wu[0], w[0], cx, u);
    k.W[1] = face(wu[1], w[1], cx, u && c1);
    k.iE[0] = face(w[0], w[2], cx, r1);
    k.iE[1] = face(w[1], w[3], cx, r1 && c1);
    k.E[0] = face(w[2], wd[0], cx, r2);
    k.E[1] = face(w[3], wd[1], cx, r2 && c1);
    k.S[0] = face(wl[0], w[0], cy, l);
    k.S[1] = face(wl[1], w[2], cy, l && r1);
    k.iN[0] = face(w[0], w[1], cy, c1);
    k.iN[1] = face(w[2], w[3], cy, c1 && r1);
    k.N[0] = face(w[1], wr[0], cy, c2);
    k.N[1] = face(w[3], wr[1], cy, c2 && r1);
    const T d[4] = {k.template diag<0>(), k.template diag<1>(), k.template diag<2>(), k.template diag<3>()};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const T in = d[q] != T(0) ? T(1) : T(0);
        k.rc[q] = in * recip(d[q] != T(0) ? d[q] : T(1));
    }
}

// ---------------------------------------------------------------------------
// the bottom of the V-cycle: from the first level of at most 64 x 64 cells down
// to the coarsest and back up in one workgroup.  Depth D holds a level of at
// most 64 >> D cells a side on (32 >> D)^2 threads; from depth 2 on one wave
// does the work and needs no workgroup barrier.  The coarsest level (at most
// 2 x 2 cells) has depth 5; its solution operator is formed once per solve.
//
// One workgroup is bound by latency: LDS round trips, dependent FP64 chains and
// the fetch of its own code, which every launch starts without.  So the depths
// share one loop body (the planes of all depths have one pitch) instead of an
// unrolled copy each, all loads of the level data are issued together, and what
// is needed again on the way up is kept in LDS.  The 5-point coefficients are
// formed once per solve (k_bot5_setup, 6 us): forming them from w on both ways of
// every V-cycle took a third of the bottom.  FP64, 5-point, kernel trace: 20.3 us
// from 64^2 (28.9 with the coefficients formed in the cycle), 14.5 us from 32^2
// (19.7); with one cell per thread and a barrier per phase on every level 21.5 us
// from 32^2, plus 19 us for the two legs of the 64^2 level.  A step of the 1024^2
// quarter five-spot: 2.46 -> 2.36 ms, of the 64^2 one 0.79 -> 0.74.
// 9-point: 24 us from 36^2, in place of about 100 launches of 4.5 us.  The
// 9-point coefficients of the deeper levels kept in LDS measured slower (27.6 us:
// the copy costs more than the cached reads).
// ---------------------------------------------------------------------------
constexpr int BOT_DEPTHS = 6;   // 64, 32, 16, 8, 4, 2 cells a side
// the planes of all depths: depth 0 in rows 0..33, the others side by side
// below it
struct BotGeo {
    static constexpr int LD = 34, PLANE = 52 * 34, CELLS = 4 * PLANE;
    static __device__ __forceinline__ int origin(int d) {   // rows 34 and 44, columns 0, 18, 28, 18, 22
        constexpr unsigned long long tab = 0ull | 18ull << 9 | 28ull << 18 | (10ull * LD + 18) << 27 | (10ull * LD + 22) << 36;
        return d == 0 ? 0 : 34 * LD + (int)(tab >> (9 * (d - 1)) & 511);
    }
};
struct BotResGeo {   // the residual planes, one depth at a time
    static constexpr int LD = 34, PLANE = 34 * 34, CELLS = 4 * PLANE;
};
// right-hand sides of depths 1..5, cell q of block t at rhs_at(d) + q P^2 + t
constexpr int BOT_RHS = 4 * (256 + 64 + 16 + 4 + 1);
__device__ __forceinline__ int bot_rhs_at(int d) {   // d >= 1
    constexpr unsigned long long tab = 0ull | 1024ull << 11 | 1280ull << 22 | 1344ull << 33 | 1360ull << 44;
    return (int)(tab >> (11 * (d - 1)) & 2047);
}

template <typename T>
struct BotLev {
    const T *w;          // mobility quantity at cell (0, 0), pitch ldw (5-point: k_bot5_setup)
    OpPlanes<T> A;       // assembled operator (9-point)
    int ldw;
};
// The 5-point coefficients of the bottom's levels, formed once per solve
// (k_bot5_setup): coefficient q of a block at q * blocks + block, for depth 0 and
// then, as they go into LDS, for depths 1..4 (block t of depth d at
// bot_rhs_at(d) / 4 + t).
constexpr int BOT_CO = 16, BOT_SMALL = 256 + 64 + 16 + 4 + 1;
constexpr int BOT_IMG = BOT_CO * (1024 + BOT_SMALL);
template <typename T>
constexpr size_t bot_img_bytes() { return 16 * sizeof(double) + BOT_IMG * sizeof(T); }
// The sizes and spacings of the deeper levels follow from the first one's
// (halved, rounded up; spacings doubled): reading them per level would be a
// cold scalar load in every depth's chain.
template <typename T>
struct BottomArgs {
    int d0, nl, ns, harmonic;      // depth of the first level, levels, sweeps per leg
    int n1, n2;                    // first level
    double cx, cy;                 // its 1 / dx^2, 1 / dy^2
    BotLev<T> lev[BOT_DEPTHS];
    const double *inv;             // coarsest level's solution operator
    const T *img;                  // 5-point coefficients (BOT_IMG values)
    const T *b;                    // right-hand side of the first level at (0, 0)
    T *out;                        // its solution
    int ldb, ldo;
    const double *S;               // loop state (ensembles)
};
template <typename T>
struct BotSize {   // of the level at depth d
    int n1, n2;
    T cx, cy;
    __device__ __forceinline__ BotSize(const BottomArgs<T> &A, int d) {
        const int l = d - A.d0, up = (1 << l) - 1;
        n1 = (A.n1 + up) >> l;
        n2 = (A.n2 + up) >> l;
        const double q = __hiloint2double((1023 - 2 * l) << 20, 0);   // 4^-l
        cx = T(A.cx * q);
        cy = T(A.cy * q);
    }
};

// LDS: the 5-point bottom keeps the coefficients of depths 1..4, the 9-point one
// reads its operator from the caches
template <typename T, bool NINE>
struct alignas(16) BotShared {
    T x[BotGeo::CELLS], r[BotResGeo::CELLS], b[BOT_RHS];   // cleared at the start
    T co[NINE ? 4 : BOT_CO * BOT_SMALL];
    double inv[16];
    static constexpr int CLEAR16 = (BotGeo::CELLS + BotResGeo::CELLS + BOT_RHS) * (int)sizeof(T) / 16;
};

// the coarsest level of N1 x N2 <= 2 x 2 cells: column k of the solution operator
// of the singular Neumann system bordered by the zero-mean condition,
// [A 1; 1^T 0][x; l] = [b; 0], A with the legs' faces; FP64 in both precisions
template <int N1, int N2, typename T>
__device__ __forceinline__ void bot5_inverse(const T *w, int ld, T cx, T cy, int hm, int k, double *inv) {
    constexpr int n = N1 * N2, m = n + 1;
    double M[m][m + 1];
#pragma unroll
    for (int r = 0; r < m; r++)
#pragma unroll
        for (int q = 0; q <= m; q++) M[r][q] = 0.;
    auto link = [&](int a, int b, T f) {
        M[a][a] -= (double)f;
        M[b][b] -= (double)f;
        M[a][b] += (double)f;
        M[b][a] += (double)f;
    };
    constexpr int C01 = N2 > 1 ? 1 : 0, C10 = N1 > 1 ? N2 : 0, C11 = N1 > 1 && N2 > 1 ? 3 : 0;
    if constexpr (N1 > 1) link(0, C10, cx * face_mob_pc(w[0], w[ld], hm));
    if constexpr (N2 > 1) link(0, C01, cy * face_mob_pc(w[0], w[1], hm));
    if constexpr (N1 > 1 && N2 > 1) {
        link(C01, C11, cx * face_mob_pc(w[1], w[ld + 1], hm));
        link(C10, C11, cy * face_mob_pc(w[ld], w[ld + 1], hm));
    }
#pragma unroll
    for (int r = 0; r < n; r++) {
        M[r][n] = 1.;
        M[n][r] = 1.;
        M[r][m] = r == k ? 1. : 0.;
    }
    double sol[m];
    bordered_solve<n, true>(M, sol);
#pragma unroll
    for (int r = 0; r < n; r++) inv[r * n + k] = sol[r];
}

// w of block (bi, bj) and around it, indices clamped into the level (a clamped
// value only enters a face that is dropped), and its faces
template <typename T>
__device__ __forceinline__ void co5_from_w(const T *w, int ldw, int n1, int n2, int bi, int bj, T cx, T cy, int hm,
                                           Co5<T> &k) {
    const int i0 = 2 * bi, j0 = 2 * bj;
    auto at = [&](int i, int j) -> T {
        i = i < 0 ? 0 : (i > n1 - 1 ? n1 - 1 : i);
        j = j < 0 ? 0 : (j > n2 - 1 ? n2 - 1 : j);
        return w[(long)i * ldw + j];
    };
    const T c[4] = {at(i0, j0), at(i0, j0 + 1), at(i0 + 1, j0), at(i0 + 1, j0 + 1)};
    const T wu[2] = {at(i0 - 1, j0), at(i0 - 1, j0 + 1)}, wd[2] = {at(i0 + 2, j0), at(i0 + 2, j0 + 1)};
    const T wl[2] = {at(i0, j0 - 1), at(i0 + 1, j0 - 1)}, wr[2] = {at(i0, j0 + 2), at(i0 + 1, j0 + 2)};
    make_co5(c, wu, wd, wl, wr, bi, bj, n1, n2, cx, cy, hm, k);
}

// Co5 as an array of BOT_CO values, and back
template <typename T, class F>
__device__ __forceinline__ void co5_each(Co5<T> &k, F &&f) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
        f(q, k.W[q]);
        f(2 + q, k.E[q]);
        f(4 + q, k.S[q]);
        f(6 + q, k.N[q]);
        f(8 + q, k.iE[q]);
        f(10 + q, k.iN[q]);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) f(12 + q, k.rc[q]);
}

// the coefficients of one depth (workgroup `d` of 6, 1024 threads), and the
// coarsest level's solution operator (workgroup 5)
template <typename T>
__device__ __forceinline__ void bot5_setup_body(const BottomArgs<T> &A, int d, T *img, double *inv) {
    const int t = threadIdx.x, dl = A.d0 + A.nl - 1;
    if (d < BOT_DEPTHS - 1) {
        const int p = 5 - d;
        if (d < A.d0 || d >= dl || t >= 1 << (2 * p)) return;
        const BotSize<T> L(A, d);
        const int bi = t >> p, bj = t & ((1 << p) - 1);
        const bool act = 2 * bi < L.n1 && 2 * bj < L.n2;
        Co5<T> k;
        if (act) {
            const BotLev<T> &v = A.lev[d - A.d0];
            co5_from_w(v.w, v.ldw, L.n1, L.n2, bi, bj, L.cx, L.cy, A.harmonic, k);
        } else {
            co5_each(k, [](int, T &v) { v = T(0); });
        }
        T *out = d == 0 ? img + t : img + BOT_CO * 1024 + bot_rhs_at(d) / 4 + t;
        const int blocks = d == 0 ? 1024 : BOT_SMALL;
        co5_each(k, [&](int q, T &v) { out[q * blocks] = v; });
    } else {
        const BotSize<T> L(A, dl);
        const BotLev<T> &v = A.lev[A.nl - 1];
        if (t >= L.n1 * L.n2) return;
        // the hierarchy is coarsened until both sides are at most 2
        if (L.n1 == 2 && L.n2 == 2) bot5_inverse<2, 2>(v.w, v.ldw, L.cx, L.cy, A.harmonic, t, inv);
        else if (L.n1 == 2 && L.n2 == 1) bot5_inverse<2, 1>(v.w, v.ldw, L.cx, L.cy, A.harmonic, t, inv);
        else if (L.n1 == 1 && L.n2 == 2) bot5_inverse<1, 2>(v.w, v.ldw, L.cx, L.cy, A.harmonic, t, inv);
        else bot5_inverse<1, 1>(v.w, v.ldw, L.cx, L.cy, A.harmonic, t, inv);
    }
}

// what is read before the first barrier: the coefficients and the right-hand side
// of the first level (k0: at depth 0, the others are in LDS), and what goes to LDS
template <typename T>
__device__ __forceinline__ void bot_preload(const BottomArgs<T> &A, BotShared<T, false> &s, int bi, int bj, bool act,
                                            Co5<T> &k0) {
    const int t = threadIdx.x, nt = blockDim.x;
    if (act && A.d0 == 0) co5_each(k0, [&](int q, T &v) { v = A.img[q * 1024 + t]; });
    constexpr int N = BOT_CO * BOT_SMALL * (int)sizeof(T) / 16;
    static_assert(N * 16 == BOT_CO * BOT_SMALL * (int)sizeof(T), "copied 16 bytes at a time");
    const double2 *src = reinterpret_cast<const double2 *>(A.img + BOT_CO * 1024);
    double2 *dst = reinterpret_cast<double2 *>(s.co);
    for (int base = t; base < N; base += 4 * nt) {
        double2 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = src[min(base + u * nt, N - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (base + u * nt < N) dst[base + u * nt] = v[u];
    }
    if (t < 16) s.inv[t] = A.inv[t];
}
__device__ __forceinline__ void bot_preload(const BottomArgs<double> &A, BotShared<double, true> &s, int bi, int bj,
                                            bool act, Co9<double> &k0) {
    if (threadIdx.x < 16) s.inv[threadIdx.x] = A.inv[threadIdx.x];
}

// the coefficients of block (bi, bj) of depth d
template <typename T>
__device__ __forceinline__ void bot_coeffs(const BottomArgs<T> &A, const BotShared<T, false> &s, int d, int bi, int bj,
                                           const Co5<T> &k0, Co5<T> &k) {
    if (d == 0) {
        k = k0;
        return;
    }
    const int at = bot_rhs_at(d) / 4 + (int)threadIdx.x;
    co5_each(k, [&](int q, T &v) { v = s.co[q * BOT_SMALL + at]; });
}
__device__ __forceinline__ void bot_coeffs(const BottomArgs<double> &A, const BotShared<double, true> &s, int d, int bi,
                                           int bj, const Co9<double> &k0, Co9<double> &k) {
    load_co9(A.lev[d - A.d0].A, bi, bj, k);
}
template <typename T>
__device__ __forceinline__ void bot_diag(const BottomArgs<T> &A, const BotShared<T, false> &s, int d, int bi, int bj,
                                         const Co5<T> &k, T (&c)[4]) {
    c[0] = k.template diag<0>();
    c[1] = k.template diag<1>();
    c[2] = k.template diag<2>();
    c[3] = k.template diag<3>();
}
__device__ __forceinline__ void bot_diag(const BottomArgs<double> &A, const BotShared<double, true> &s, int d, int bi,
                                         int bj, const Co9<double> &k, double (&c)[4]) {
    load_diag9(A.lev[d - A.d0].A, bi, bj, c);
}

// the right-hand side of the bottom's first level
template <typename T>
__device__ __forceinline__ void bot_rhs0(const BottomArgs<T> &A, int bi, int bj, T (&b)[4]) {
    const T *bp = A.b + (long)(2 * bi) * A.ldb + 2 * bj;
    const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
    b[0] = bp[0];
    b[1] = v1 ? bp[1] : T(0);
    b[2] = w1 ? bp[A.ldb] : T(0);
    b[3] = v1 && w1 ? bp[A.ldb + 1] : T(0);
}
// that of depth d: of the first level b0 (9-point: read again, its registers are
// needed for the operator), of the others from LDS
template <typename T, bool NINE>
__device__ __forceinline__ void bot_rhs(const BottomArgs<T> &A, const BotShared<T, NINE> &s, int d, int bi, int bj,
                                        const T (&b0)[4], T (&b)[4]) {
    if (NINE && d == A.d0) {
        bot_rhs0(A, bi, bj, b);
    } else if (d == A.d0) {
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = b0[q];
    } else {
        const int pp = 1 << (2 * (5 - d)), at = bot_rhs_at(d) + (int)threadIdx.x;
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = s.b[at + q * pp];
    }
}

template <typename T, bool NINE>
__device__ __forceinline__ void mg_bottom_body(const BottomArgs<T> &A, BotShared<T, NINE> &s) {
    using Co = typename std::conditional<NINE, Co9<T>, Co5<T>>::type;
    using G = BotGeo;
    using GR = BotResGeo;
    const int t = threadIdx.x, dl = A.d0 + A.nl - 1;   // the coarsest level's depth
    Co k0;
    T b0[4] = {T(0), T(0), T(0), T(0)};
    {
        const int p = 5 - A.d0, bi = t >> p, bj = t & ((1 << p) - 1);
        const bool act = t < 1 << (2 * p) && 2 * bi < A.n1 && 2 * bj < A.n2;
        if (!NINE && act) bot_rhs0(A, bi, bj, b0);
        bot_preload(A, s, bi, bj, act, k0);
    }
    for (int q = t; q < BotShared<T, NINE>::CLEAR16; q += blockDim.x)
        reinterpret_cast<double2 *>(s.x)[q] = double2{0., 0.};
    __syncthreads();
    // down: sweeps from a zero guess, residual, full weighting
    for (int d = A.d0; d < dl; d++) {
        if (d >= 2 && t >= 64) break;
        const int p = 5 - d, bi = t >> p, bj = t & ((1 << p) - 1);
        const bool wg = d < 2;
        const BotSize<T> L(A, d), Lc(A, d + 1);
        const bool act = t < 1 << (2 * p) && 2 * bi < L.n1 && 2 * bj < L.n2;
        const int o = G::origin(d) + (bi + 1) * G::LD + bj + 1, orr = (bi + 1) * GR::LD + bj + 1;
        Co k;
        T b[4], x[4] = {T(0), T(0), T(0), T(0)}, r[4];
        if (act) {
            bot_rhs<T, NINE>(A, s, d, bi, bj, b0, b);
            bot_coeffs(A, s, d, bi, bj, k0, k);
        }
        blk_sweeps<G, false>(k, b, x, s.x, o, act, A.ns, wg);
        if (act) {
            T c[4];
            bot_diag(A, s, d, bi, bj, k, c);
            blk_residual<G>(k, c, b, x, s.x, o, r);
#pragma unroll
            for (int q = 0; q < 4; q++) s.r[q * GR::PLANE + orr] = r[q];
        }
        blk_sync(wg);
        // the coarse cell (bi, bj) is cell (bi & 1, bj & 1) of block (bi / 2, bj / 2)
        if (act) {
            T wi[4], wj[4];
            rest_weights(bi, L.n1, Lc.n1, wi);
            rest_weights(bj, L.n2, Lc.n2, wj);
            const int pc = p > 0 ? p - 1 : 0;
            s.b[bot_rhs_at(d + 1) + (((bi & 1) * 2 + (bj & 1)) << (2 * pc)) + ((bi >> 1) << pc) + (bj >> 1)] =
                blk_restrict<GR>(r, s.r, orr, wi, wj);
        }
        blk_sync(wg);
    }
    const BotSize<T> Lb(A, dl);
    __syncthreads();
    if (t < 64) {
        const int r = t >> 1, c = t & 1;   // cell (r, c) on lane 2 r + c
        if (t < 4 && r < Lb.n1 && c < Lb.n2) {
            const int n = Lb.n1 * Lb.n2, row = r * Lb.n2 + c;
            double v = 0.;
            for (int q = 0; q < n; q++)
                v += s.inv[row * n + q] * (double)s.b[bot_rhs_at(5) + (q / Lb.n2) * 2 + q % Lb.n2];
            s.x[t * G::PLANE + G::origin(5) + G::LD + 1] = T(v);
        }
        wave_sync();
    }
    // up: x + P e, sweeps
    for (int d = dl - 1; d >= A.d0; d--) {
        const bool wg = d < 2;
        if (!wg && t >= 64) continue;
        if (wg) __syncthreads();
        const int p = 5 - d, bi = t >> p, bj = t & ((1 << p) - 1);
        const BotSize<T> L(A, d), Lc(A, d + 1);
        const bool act = t < 1 << (2 * p) && 2 * bi < L.n1 && 2 * bj < L.n2;
        const int o = G::origin(d) + (bi + 1) * G::LD + bj + 1;
        Co k;
        T b[4], x[4] = {T(0), T(0), T(0), T(0)};
        if (act) {
            const T *sc = s.x + G::origin(d + 1);
            T e[3][3];
#pragma unroll
            for (int q = 0; q < 3; q++)
#pragma unroll
                for (int u = 0; u < 3; u++) {
                    const int I = bi + q - 1 < 0 ? 0 : (bi + q - 1 > Lc.n1 - 1 ? Lc.n1 - 1 : bi + q - 1);
                    const int J = bj + u - 1 < 0 ? 0 : (bj + u - 1 > Lc.n2 - 1 ? Lc.n2 - 1 : bj + u - 1);
                    e[q][u] = sc[((I & 1) * 2 + (J & 1)) * G::PLANE + ((I >> 1) + 1) * G::LD + (J >> 1) + 1];
                }
#pragma unroll
            for (int q = 0; q < 4; q++) x[q] = s.x[q * G::PLANE + o];
            blk_prolong(e, x);
#pragma unroll
            for (int q = 0; q < 4; q++) s.x[q * G::PLANE + o] = x[q];
            bot_rhs<T, NINE>(A, s, d, bi, bj, b0, b);
            bot_coeffs(A, s, d, bi, bj, k0, k);
        }
        blk_sync(wg);
        blk_sweeps<G, true>(k, b, x, s.x, o, act, A.ns, wg);
        if (d == A.d0 && act) {
            T *xp = A.out + (long)(2 * bi) * A.ldo + 2 * bj;
            const bool v1 = 2 * bj + 1 < L.n2, w1 = 2 * bi + 1 < L.n1;
            xp[0] = x[0];
            if (v1) xp[1] = x[1];
            if (w1) xp[A.ldo] = x[2];
            if (v1 && w1) xp[A.ldo + 1] = x[3];
        }
    }
}

// ---------------------------------------------------------------------------
// legs of the 5-point V-cycle over one coarse level (level 1 and below), on
// tiles of 64 x 64 cells of which the middle 52 x 52 (down) and 56 x 56 (up) are
// written.  A streaming leg marches down at least a chunk and its halo rows, a
// chain of memory and FP64 latencies per row; a tile has all its cells in flight
// at once.  Levels of 128^2 to 512^2: 7.4 (down) and 8.1 us (up) against 12.7 and
// 9.2 us.
// ---------------------------------------------------------------------------
template <int NS> struct Halo5;
template <> struct Halo5<1> { static constexpr int D = 2, U = 1; };
template <> struct Halo5<2> { static constexpr int D = 3, U = 2; };

template <typename T>
struct Leg5Args {
    const T *w;           // mobility quantity at (0, 0), pitch ldw
    int ldw, harmonic;
    double cx, cy;
    int n1, n2, ld;       // level arrays at cell (0, 0), pitch ld
    const T *b;
    T *x;                 // down: written; up: read
    T *xo;                // up: written
    T *bc;                // down: the coarser level's right-hand side
    const T *xc;          // up: its solution
    int m1, m2, ldc;
    int ti, tj;           // tiles per direction
    const double *S;      // loop state (ensembles)
};

template <typename T>
__device__ __forceinline__ void leg5_inputs(const Leg5Args<T> &A, int bi, int bj, T (&b)[4], Co5<T> &k) {
    const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
    const T *bp = A.b + (long)(2 * bi) * A.ld + 2 * bj;
    b[0] = bp[0];
    b[1] = v1 ? bp[1] : T(0);
    b[2] = w1 ? bp[A.ld] : T(0);
    b[3] = v1 && w1 ? bp[A.ld + 1] : T(0);
    co5_from_w(A.w, A.ldw, A.n1, A.n2, bi, bj, T(A.cx), T(A.cy), A.harmonic, k);
}

// tile `wg` of a down leg: sweeps from a zero guess, residual, full weighting
template <int P, int NS, typename T>
__device__ __forceinline__ void leg5_down_body(const Leg5Args<T> &A, int wg, T *sm) {
    using G = BlkGeo<P>;
    constexpr int H = Halo5<NS>::D;
    const int t = threadIdx.x;
    const int ki = wg / A.tj, kj = wg - ki * A.tj;
    const int nb1 = (A.n1 + 1) >> 1, nb2 = (A.n2 + 1) >> 1;
    const int li = t / P, lj = t % P;
    const int bi = tile_origin(ki, nb1, P, H) + li, bj = tile_origin(kj, nb2, P, H) + lj;
    const bool act = bi < nb1 && bj < nb2;
    const int o = (li + 1) * G::LD + lj + 1;
    Co5<T> k;
    T b[4], x[4] = {T(0), T(0), T(0), T(0)}, r[4] = {T(0), T(0), T(0), T(0)};
    for (int q = t; q < G::CELLS; q += P * P) sm[q] = T(0);
    if (act) leg5_inputs(A, bi, bj, b, k);
    __syncthreads();
    blk_sweeps<G, false>(k, b, x, sm, o, act, NS, true);
    if (act) {
        const T c[4] = {k.template diag<0>(), k.template diag<1>(), k.template diag<2>(), k.template diag<3>()};
        blk_residual<G>(k, c, b, x, sm, o, r);
    }
    __syncthreads();   // the planes now take the residual
    if (act)
#pragma unroll
        for (int q = 0; q < 4; q++) sm[q * G::PLANE + o] = r[q];
    __syncthreads();
    const bool out = act && bi >= tile_lo(ki, P, H) && bi < tile_hi(ki, A.ti, nb1, P, H) && bj >= tile_lo(kj, P, H) &&
                     bj < tile_hi(kj, A.tj, nb2, P, H);
    if (out) {
        T wi[4], wj[4];
        rest_weights(bi, A.n1, A.m1, wi);
        rest_weights(bj, A.n2, A.m2, wj);
        A.bc[(long)bi * A.ldc + bj] = blk_restrict<G>(r, sm, o, wi, wj);
        T *xp = A.x + (long)(2 * bi) * A.ld + 2 * bj;
        const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
        xp[0] = x[0];
        if (v1) xp[1] = x[1];
        if (w1) xp[A.ld] = x[2];
        if (v1 && w1) xp[A.ld + 1] = x[3];
    }
}

template <int P, int NS, typename T>
__device__ __forceinline__ void leg5_up_body(const Leg5Args<T> &A, int wg, T *sm) {
    using G = BlkGeo<P>;
    constexpr int H = Halo5<NS>::U;
    const int t = threadIdx.x;
    const int ki = wg / A.tj, kj = wg - ki * A.tj;
    const int nb1 = (A.n1 + 1) >> 1, nb2 = (A.n2 + 1) >> 1;
    const int li = t / P, lj = t % P;
    const int bi = tile_origin(ki, nb1, P, H) + li, bj = tile_origin(kj, nb2, P, H) + lj;
    const bool act = bi < nb1 && bj < nb2;
    const bool v1 = 2 * bj + 1 < A.n2, w1 = 2 * bi + 1 < A.n1;
    const int o = (li + 1) * G::LD + lj + 1;
    Co5<T> k;
    T b[4], x[4] = {T(0), T(0), T(0), T(0)};
    for (int q = t; q < G::CELLS; q += P * P) sm[q] = T(0);
    if (act) {
        const T *xp = A.x + (long)(2 * bi) * A.ld + 2 * bj;
        x[0] = xp[0];
        if (v1) x[1] = xp[1];
        if (w1) x[2] = xp[A.ld];
        if (v1 && w1) x[3] = xp[A.ld + 1];
        T e[3][3];
#pragma unroll
        for (int q = 0; q < 3; q++)
#pragma unroll
            for (int p = 0; p < 3; p++) {
                const int I = bi + q - 1 < 0 ? 0 : (bi + q - 1 > A.m1 - 1 ? A.m1 - 1 : bi + q - 1);
                const int J = bj + p - 1 < 0 ? 0 : (bj + p - 1 > A.m2 - 1 ? A.m2 - 1 : bj + p - 1);
                e[q][p] = A.xc[(long)I * A.ldc + J];
            }
        leg5_inputs(A, bi, bj, b, k);
        blk_prolong(e, x);
    }
    __syncthreads();
    if (act)
#pragma unroll
        for (int q = 0; q < 4; q++) sm[q * G::PLANE + o] = x[q];
    __syncthreads();
    blk_sweeps<G, true>(k, b, x, sm, o, act, NS, true);
    const bool out = act && bi >= tile_lo(ki, P, H) && bi < tile_hi(ki, A.ti, nb1, P, H) && bj >= tile_lo(kj, P, H) &&
                     bj < tile_hi(kj, A.tj, nb2, P, H);
    if (out) {
        T *xp = A.xo + (long)(2 * bi) * A.ld + 2 * bj;
        xp[0] = x[0];
        if (v1) xp[1] = x[1];
        if (w1) xp[A.ld] = x[2];
        if (v1 && w1) xp[A.ld + 1] = x[3];
    }
}

template <int P, int NS, typename T>
__global__ void __launch_bounds__(P *P) k_mg5_down(Leg5Args<T> A) {
    __shared__ T sm[BlkGeo<P>::CELLS];
    leg5_down_body<P, NS, T>(A, blockIdx.x, sm);
}
template <int P, int NS, typename T>
__global__ void __launch_bounds__(P *P) k_mg5_up(Leg5Args<T> A) {
    __shared__ T sm[BlkGeo<P>::CELLS];
    leg5_up_body<P, NS, T>(A, blockIdx.x, sm);
}

}  // namespace impec
