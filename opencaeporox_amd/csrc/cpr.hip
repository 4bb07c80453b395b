// cpr.hip — pressure AMG, multicolour block Gauss-Seidel and FGMRES pieces
// of the device linear solve, for gfx950 (declarations and the method in
// cpr.hpp).
//
// Every kernel here is a plain gather: a thread (or a group of B lanes for a
// block row) owns its output entries and reductions sum in a fixed order, so
// the same bits on every run.  The AMG level matrices are formed as scalar CSR
// with the diagonal first in each row and walked by the V-cycle in sliced
// columns (amg::Sell).
#include <algorithm>
#include <cstring>

#include "amg_layout.hpp"
#include "cpr.hpp"
#include "ocpx_dev.hpp"
#include "ocpx_kernels.hpp"

namespace ocpx {

namespace {

constexpr double OMEGA = PressureAmg::OMEGA;
constexpr int MAX_LEVELS = 25;

// ------------------------------------------------------------------ kernels
// Column 0 of every decoupled block, d0[s] = Dinv_i A_s(:, 0), by B lanes per
// block row (lane r = row r; the block's column is passed round the lanes),
// and from its row 0 the pressure block a[s], made an M-matrix for the
// hierarchy: positive off-diagonal entries go to the diagonal, and the
// diagonal is at least the sum of the remaining off-diagonal magnitudes (the
// decoupled pressure block of a state far from equilibrium is indefinite, and a
// Jacobi-smoothed aggregation cycle on it diverges).  The correction of the
// pressure stage is non-zero in the pressures only, so its residual needs
// these columns and not the blocks: 1 / B of the matrix.
template <int B>
__global__ void __launch_bounds__(64) cpr_columns(int64_t n, const int64_t* __restrict__ rp,
                                                  const double* __restrict__ val, const double* __restrict__ dinv,
                                                  double* __restrict__ d0, double* __restrict__ a)
{
    constexpr int G = 64 / B;
    const int lane = threadIdx.x, g = lane / B, r = lane % B;
    const int64_t i = (int64_t)blockIdx.x * G + g;
    const bool valid = g < G && i < n;
    const int base = (g < G ? g : 0) * B;
    double d[B];
    UNROLL for (int m = 0; m < B; m++) d[m] = valid ? dinv[((size_t)i * B + r) * B + m] : 0.0;
    const int64_t s0 = valid ? rp[i] : 0, s1 = valid ? rp[i + 1] : 0;
    int cnt = (int)(s1 - s0);                       // the wavefront runs its longest row, so every
    for (int o = 32; o > 0; o >>= 1) cnt = max(cnt, __shfl_xor(cnt, o));   // lane takes part in the exchanges
    double diag = 0, pos = 0, neg = 0;
    for (int k = 0; k < cnt; k++) {
        const int64_t s = s0 + k;
        const bool in = s < s1;
        const double c = in ? val[((size_t)s * B + r) * B] : 0.0;
        double acc = 0;
        UNROLL for (int m = 0; m < B; m++) acc += d[m] * __shfl(c, base + m);
        if (!in) continue;
        d0[(size_t)s * B + r] = acc;
        if (r == 0) {
            if (k == 0) {
                diag = acc;
            } else {
                if (acc > 0) {
                    pos += acc;
                    acc = 0;
                } else {
                    neg -= acc;
                }
                a[s] = acc;
            }
        }
    }
    if (valid && r == 0) a[s0] = fmax(diag + pos, neg);
}

__global__ void __launch_bounds__(256) amg_gather(int64_t nnz, const int64_t* __restrict__ gp,
                                                  const int64_t* __restrict__ gs, const double* __restrict__ af,
                                                  double* __restrict__ ac)
{
    const int64_t s = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (s >= nnz) return;
    double acc = 0;
    for (int64_t t = gp[s]; t < gp[s + 1]; t++) acc += af[gs[t]];
    ac[s] = acc;
}

__global__ void __launch_bounds__(256) amg_dinv(int64_t n, const int64_t* __restrict__ rp,
                                                const double* __restrict__ a, double* __restrict__ dinv)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double d = a[rp[i]];
    dinv[i] = d != 0 ? 1 / d : 0.0;
}

// a level's pattern in V-cycle order, one thread per position
__global__ void __launch_bounds__(256) amg_sell_fill(int64_t nq, const int64_t* __restrict__ off,
                                                     const int32_t* __restrict__ row, const int64_t* __restrict__ rp,
                                                     const int32_t* __restrict__ gci,
                                                     const int32_t* __restrict__ agg, int32_t* __restrict__ ci,
                                                     int32_t* __restrict__ cagg, int32_t* __restrict__ src)
{
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q < nq) amg::sell_position(q, off, row, rp, gci, agg, ci, cagg, src);
}

// a level's values in V-cycle order
__global__ void __launch_bounds__(256) amg_sell(int64_t ne, const int32_t* __restrict__ src,
                                                const double* __restrict__ a, double* __restrict__ sa)
{
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= ne) return;
    const int32_t s = src[e];
    sa[e] = s >= 0 ? a[s] : 0.0;
}

// xo = x + OMEGA Dinv (b - A x)
__global__ void __launch_bounds__(256) amg_smooth(int64_t n, const int64_t* __restrict__ rp,
                                                  const int32_t* __restrict__ ci, const double* __restrict__ a,
                                                  const double* __restrict__ dinv, const double* __restrict__ b,
                                                  const double* __restrict__ x, double* __restrict__ xo)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    double r = b[i];
    for (int64_t s = rp[i]; s < rp[i + 1]; s++) r -= a[s] * x[ci[s]];
    xo[i] = x[i] + OMEGA * dinv[i] * r;
}

// Down a level: the residual of each position's row, summed over the
// aggregate's four positions, is the coarse right-hand side; the coarse level's
// first sweep from zero, OMEGA Dinv b, is written with it.  The thread per
// fine row (a thread per coarse row walked its rows one after another: 72 us at
// 500,000 rows, 22 now) and the sliced columns keep every load of the matrix
// contiguous.
__global__ void __launch_bounds__(256) amg_down(int64_t nq, int64_t nc, const int64_t* __restrict__ off,
                                                const int32_t* __restrict__ row, const int32_t* __restrict__ ci,
                                                const double* __restrict__ a, const double* __restrict__ b,
                                                const double* __restrict__ x, const double* __restrict__ dinvc,
                                                double* __restrict__ bc, double* __restrict__ xc)
{
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= nq) return;                            // nq is a multiple of 64: whole wavefronts
    const int32_t i = row[q];
    double r = 0;
    if (i >= 0) {
        r = b[i];
        const int64_t e1 = off[(q >> 6) + 1];
        int64_t e = off[q >> 6] + (q & 63);
        for (; e + 192 < e1; e += 256) {            // four entries in flight
            double av[4], xv[4];
            UNROLL for (int u = 0; u < 4; u++) { av[u] = a[e + 64 * u]; xv[u] = x[ci[e + 64 * u]]; }
            UNROLL for (int u = 0; u < 4; u++) r -= av[u] * xv[u];
        }
        for (; e < e1; e += 64) r -= a[e] * x[ci[e]];
    }
    r += __shfl_xor(r, 1);
    r += __shfl_xor(r, 2);
    const int64_t I = q >> 2;
    if ((q & 3) == 0 && I < nc) {
        bc[I] = r;
        xc[I] = OMEGA * dinvc[I] * r;
    }
}

// Up a level: x' = x + the coarse correction of the row's aggregate, then one
// weighted-Jacobi sweep, both in one pass (cagg: the aggregate of a column).
__global__ void __launch_bounds__(256) amg_up(int64_t nq, const int64_t* __restrict__ off,
                                              const int32_t* __restrict__ row, const int32_t* __restrict__ ci,
                                              const int32_t* __restrict__ cagg, const double* __restrict__ a,
                                              const double* __restrict__ dinv, const double* __restrict__ b,
                                              const double* __restrict__ x, const double* __restrict__ xc,
                                              double* __restrict__ xo)
{
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= nq) return;
    const int32_t i = row[q];
    if (i < 0) return;
    double r = b[i];
    const int64_t e1 = off[(q >> 6) + 1];
    int64_t e = off[q >> 6] + (q & 63);
    for (; e + 192 < e1; e += 256) {
        double av[4], xv[4];
        UNROLL for (int u = 0; u < 4; u++) { av[u] = a[e + 64 * u]; xv[u] = x[ci[e + 64 * u]] + xc[cagg[e + 64 * u]]; }
        UNROLL for (int u = 0; u < 4; u++) r -= av[u] * xv[u];
    }
    for (; e < e1; e += 64) r -= a[e] * (x[ci[e]] + xc[cagg[e]]);
    xo[i] = (x[i] + xc[q >> 2]) + OMEGA * dinv[i] * r;
}

// The part of the V-cycle from the first level of at most SM_TOP rows on (levels
// of at most SM_ROWS together) in one workgroup: every vector in LDS, the
// matrices read from L2, the coarsest level by its dense inverse.  Launched level
// by level, the levels below 2,000 rows took four launches each and a serial
// triangular solve (27 us), about 150 us of the cycle's 550 at 500,000 rows; this
// kernel takes 25.
constexpr int SM_ROWS = 1536, SM_TOP = 1024, SM_LEVELS = 14, SM_THREADS = 1024;
struct SmallLevel {
    int n, nc, nq;
    const int64_t* off;
    const int32_t *row, *ci, *cagg;
    const double *a, *dinv;
};
struct SmallHier {
    int nl, nd;                              // levels above the dense one, rows of the dense one
    const double *inv, *dinvd;
    SmallLevel lv[SM_LEVELS];
};

__global__ void __launch_bounds__(SM_THREADS) amg_small(SmallHier h, const double* __restrict__ b,
                                                        double* __restrict__ xo)
{
    constexpr int N = PressureAmg::DENSE_MAX;
    __shared__ double sb[SM_ROWS], sx[SM_ROWS], so[SM_TOP];
    const int t = threadIdx.x;
    const int n0 = h.nl ? h.lv[0].n : h.nd;
    const double* d0 = h.nl ? h.lv[0].dinv : h.dinvd;
    for (int i = t; i < n0; i += SM_THREADS) {
        const double v = b[i];
        sb[i] = v;
        sx[i] = OMEGA * d0[i] * v;
    }
    __syncthreads();
    int o = 0;
    for (int l = 0; l < h.nl; l++) {
        const SmallLevel& L = h.lv[l];
        const int on = o + L.n;
        const double* dn = l + 1 < h.nl ? h.lv[l + 1].dinv : h.dinvd;
        for (int q = t; q < L.nq; q += SM_THREADS) {         // nq is a multiple of 64: whole wavefronts
            const int i = L.row[q];
            double r = 0;
            if (i >= 0) {
                r = sb[o + i];
                const int e1 = (int)L.off[(q >> 6) + 1];
                int e = (int)L.off[q >> 6] + (q & 63);
                for (; e + 192 < e1; e += 256) {             // four entries in flight
                    double av[4];
                    int cv[4];
                    UNROLL for (int u = 0; u < 4; u++) { av[u] = L.a[e + 64 * u]; cv[u] = L.ci[e + 64 * u]; }
                    UNROLL for (int u = 0; u < 4; u++) r -= av[u] * sx[o + cv[u]];
                }
                for (; e < e1; e += 64) r -= L.a[e] * sx[o + L.ci[e]];
            }
            r += __shfl_xor(r, 1);
            r += __shfl_xor(r, 2);
            const int I = q >> 2;
            if ((q & 3) == 0 && I < L.nc) {
                sb[on + I] = r;
                sx[on + I] = OMEGA * dn[I] * r;
            }
        }
        __syncthreads();
        o = on;
    }
    {   // sixteen lanes per row of the dense inverse
        const int i = t >> 4, c = t & 15;
        double acc = 0;
        if (i < h.nd)
            for (int j = c; j < h.nd; j += 16) acc += h.inv[i * N + j] * sb[o + j];
        for (int m = 8; m > 0; m >>= 1) acc += __shfl_xor(acc, m);
        if (i < h.nd && c == 0) sx[o + i] = acc;
    }
    __syncthreads();
    for (int l = h.nl - 1; l >= 0; l--) {
        const SmallLevel& L = h.lv[l];
        const int on = o;
        o -= L.n;
        for (int q = t; q < L.nq; q += SM_THREADS) {
            const int i = L.row[q];
            if (i < 0) continue;
            double r = sb[o + i];
            const int e1 = (int)L.off[(q >> 6) + 1];
            int e = (int)L.off[q >> 6] + (q & 63);
            for (; e + 192 < e1; e += 256) {
                double av[4];
                int cv[4], gv[4];
                UNROLL for (int u = 0; u < 4; u++) { av[u] = L.a[e + 64 * u]; cv[u] = L.ci[e + 64 * u]; gv[u] = L.cagg[e + 64 * u]; }
                UNROLL for (int u = 0; u < 4; u++) r -= av[u] * (sx[o + cv[u]] + sx[on + gv[u]]);
            }
            for (; e < e1; e += 64) r -= L.a[e] * (sx[o + L.ci[e]] + sx[on + L.cagg[e]]);
            so[i] = (sx[o + i] + sx[on + (q >> 2)]) + OMEGA * L.dinv[i] * r;
        }
        __syncthreads();
        for (int i = t; i < L.n; i += SM_THREADS) sx[o + i] = so[i];
        __syncthreads();
    }
    for (int i = t; i < n0; i += SM_THREADS) xo[i] = sx[i];
}

// Dense LU with partial pivoting of the coarsest level (n <= 64), one
// 64-lane block; lane i holds row i.
__global__ void __launch_bounds__(64) amg_dense_lu(int n, const int64_t* __restrict__ rp,
                                                   const int32_t* __restrict__ ci, const double* __restrict__ a,
                                                   double* __restrict__ lu, int32_t* __restrict__ piv)
{
    constexpr int N = PressureAmg::DENSE_MAX;
    __shared__ double M[N][N + 1];
    __shared__ int prow;
    const int t = threadIdx.x;
    for (int j = 0; j < N; j++) M[t][j] = (t == j && t >= n) ? 1.0 : 0.0;
    if (t < n)
        for (int64_t s = rp[t]; s < rp[t + 1]; s++) M[t][ci[s]] += a[s];
    __syncthreads();
    for (int k = 0; k < n; k++) {
        if (t == 0) {
            int p = k;
            double best = fabs(M[k][k]);
            for (int i = k + 1; i < n; i++)
                if (fabs(M[i][k]) > best) { best = fabs(M[i][k]); p = i; }
            prow = p;
            piv[k] = p;
        }
        __syncthreads();
        const int p = prow;
        if (p != k && t < N) {           // lane t swaps column t of rows k and p
            const double v = M[k][t];
            M[k][t] = M[p][t];
            M[p][t] = v;
        }
        __syncthreads();
        const double d = M[k][k];
        if (t > k && t < n) {
            const double f = d != 0 ? M[t][k] / d : 0.0;
            M[t][k] = f;
            for (int j = k + 1; j < n; j++) M[t][j] -= f * M[k][j];
        }
        __syncthreads();
    }
    for (int j = 0; j < N; j++) lu[t * N + j] = M[t][j];
}

// The coarsest level's inverse from its LU, lane t = column t: once per solve,
// so each cycle's coarsest solve is one product.
__global__ void __launch_bounds__(64) amg_dense_inv(int n, const double* __restrict__ lu,
                                                    const int32_t* __restrict__ piv, double* __restrict__ inv)
{
    constexpr int N = PressureAmg::DENSE_MAX;
    __shared__ double M[N * N], Y[N * N];
    const int t = threadIdx.x;
    for (int i = 0; i < N; i++) { M[i * N + t] = lu[i * N + t]; Y[i * N + t] = i == t ? 1.0 : 0.0; }
    __syncthreads();
    for (int k = 0; k < n; k++) {
        const int p = piv[k];
        if (p != k) { const double v = Y[k * N + t]; Y[k * N + t] = Y[p * N + t]; Y[p * N + t] = v; }
    }
    for (int i = 0; i < n; i++) {        // L (unit diagonal); a lane reads and writes its own column only
        double v = Y[i * N + t];
        for (int k = 0; k < i; k++) v -= M[i * N + k] * Y[k * N + t];
        Y[i * N + t] = v;
    }
    for (int i = n - 1; i >= 0; i--) {   // U
        double v = Y[i * N + t];
        for (int k = i + 1; k < n; k++) v -= M[i * N + k] * Y[k * N + t];
        Y[i * N + t] = M[i * N + i] != 0 ? v / M[i * N + i] : 0.0;
    }
    for (int i = 0; i < N; i++) inv[i * N + t] = (i < n && t < n) ? Y[i * N + t] : 0.0;
}

// One colour of the block Gauss-Seidel sweep; a group of B lanes per row,
// lane r = column r of the blocks and row r of the result.  The diagonal slot is first in each row.
template <int B>
__global__ void __launch_bounds__(64) gs_color(const int32_t* __restrict__ rows, int64_t nrows,
                                               const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                               const double* __restrict__ val, const double* __restrict__ dinv,
                                               const double* __restrict__ rhat, double* __restrict__ x)
{
    constexpr int G = 64 / B;
    __shared__ double sh[64][B + 1];
    const int lane = threadIdx.x, g = lane / B, r = lane % B;
    const int64_t k = (int64_t)blockIdx.x * G + g;
    const bool valid = g < G && k < nrows;
    const int64_t i = valid ? rows[k] : 0;
    double acc[B];
    UNROLL for (int c = 0; c < B; c++) acc[c] = 0;
    if (valid)
        for (int64_t s = rowptr[i] + 1; s < rowptr[i + 1]; s++) block_column<B>(val + (size_t)s * B * B, r, x[(size_t)col[s] * B + r], acc);
    const double t = row_sums<B>(acc, sh);
    UNROLL for (int c = 0; c < B; c++) acc[c] = dinv[((size_t)i * B + c) * B + r] * t;
    const double y = row_sums<B>(acc, sh);
    if (valid) x[(size_t)i * B + r] = rhat[(size_t)i * B + r] - y;
}

// R = v - Dinv J x1 and z = R + x1 on the bulk rows for the pressure
// correction x1 (px in the pressure entries, 0 elsewhere).
template <int B>
__global__ void __launch_bounds__(64) cpr_resid(const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                                const double* __restrict__ d0, const double* __restrict__ px,
                                                const double* __restrict__ v, double* __restrict__ R,
                                                double* __restrict__ z, int64_t nb)
{
    constexpr int G = 64 / B;
    const int lane = threadIdx.x, g = lane / B, r = lane % B;
    const int64_t i = xcd_chunk(blockIdx.x, gridDim.x) * G + g;
    if (g >= G || i >= nb) return;
    double t = 0;
    for (int64_t s = rowptr[i]; s < rowptr[i + 1]; s++) t += d0[(size_t)s * B + r] * px[col[s]];
    const double y = v[(size_t)i * B + r] - t;
    R[(size_t)i * B + r] = y;
    z[(size_t)i * B + r] = r == 0 ? y + px[i] : y;
}

// The Gauss-Seidel sweep and the operator after it on a two-coloured graph,
// with the matrix read once.  g = the sweep from zero on D^{-1} J g = R: the
// first colour's rows keep R (their neighbours are still zero), the second
// colour's are g2 = R2 - Dinv A21 R1 (SECOND), z = g + x1.  Then w = D^{-1} J z =
// D^{-1} J g + (v - R); the sweep solved the second colour's rows exactly, so w2 =
// v2, and w1 = R1 + Dinv A12 g2 + v1 - R1 = v1 + Dinv A12 g2 (first colour).
// That takes Dinv D for the identity, which it is to eps cond(D); a product with
// D and then Dinv rounds by as much.
// R holds g afterwards.  One iteration reads the off-diagonal blocks once; the
// sweep over both colours, the residual before it and the product after it read
// the matrix three times (500,000 rows, B = 8: 0.47 + 0.36 + 0.36 ms, now 0.41, at
// 4.8 TB/s the rate of a large copy).
template <int B, bool SECOND>
__global__ void __launch_bounds__(64) cpr_half(const int32_t* __restrict__ rows, int64_t nrows,
                                               const int64_t* __restrict__ rowptr, const int32_t* __restrict__ col,
                                               const double* __restrict__ val, const double* __restrict__ dinv,
                                               const double* __restrict__ px, const double* __restrict__ v,
                                               double* R, double* __restrict__ z, double* __restrict__ w)
{
    constexpr int G = 64 / B;
    __shared__ double sh[64][B + 1];
    const int lane = threadIdx.x, g = lane / B, r = lane % B;
    const int64_t k = xcd_chunk(blockIdx.x, gridDim.x) * G + g;
    const bool valid = g < G && k < nrows;
    const int64_t i = valid ? rows[k] : 0;
    const size_t o = (size_t)i * B + r;
    double d[B], acc[B];                           // column r of Dinv, loaded beside the blocks
    UNROLL for (int c = 0; c < B; c++) { d[c] = dinv[((size_t)i * B + c) * B + r]; acc[c] = 0; }
    const double vo = v[o];
    if (valid)
        for (int64_t s = rowptr[i] + 1; s < rowptr[i + 1]; s++) block_column<B>(val + (size_t)s * B * B, r, R[(size_t)col[s] * B + r], acc);
    const double t = row_sums<B>(acc, sh);
    UNROLL for (int c = 0; c < B; c++) acc[c] = d[c] * t;
    const double y = row_sums<B>(acc, sh);
    if (!valid) return;
    if constexpr (SECOND) {
        const double gi = R[o] - y;
        R[o] = gi;
        z[o] = r == 0 ? gi + px[i] : gi;
        w[o] = vo;
    } else {
        w[o] = vo + y;
    }
}

// ------------------------------------------------- Gram-Schmidt of one vector
// Classical Gram-Schmidt with one reorthogonalisation against M vectors:
// h = V.w; w -= V h with h2 = V.w; w -= V h2 with w.w.  Each block writes its
// partial sums and a second kernel adds them in block order (letting the last
// block to finish add them needs a device-wide release in every block, which
// flushes the L2s: 130 us at 1,024 blocks).  Bandwidth-bound.  A thread takes E elements of a
// contiguous tile and walks the vectors one after another, M accumulators in
// registers: on 4M elements and M = 30, 6.4 TB/s for the product and 5.4 for
// the update with E = 8, against 2.5 for a thread that loads its element of
// all M vectors at once.  E = 1 for vectors that would leave the device idle.
// Up to ORTH_M vectors the first update and the second product are one
// kernel that reads the element's vectors again while they are near (M = 16:
// 145 us against 99 + 89; M = 30: 358 against 182 + 154, so two above).
constexpr int FG_THREADS = 256, FG_BLOCKS = 1024, FG_MAX = 31, FG_E = 8, ORTH_M = 16;

// the block's sums of acc into part[k][blockIdx.x] (FG_BLOCKS apart)
template <int M>
__device__ __forceinline__ void fg_partial(double (&acc)[M], double* part)
{
    __shared__ double sh[FG_THREADS / 64][32];
    const int t = threadIdx.x, wv = t >> 6, ln = t & 63;
    UNROLL for (int k = 0; k < M; k++) {
        double v = acc[k];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (ln == 0) sh[wv][k] = v;
    }
    __syncthreads();
    if (t < M) part[(size_t)t * FG_BLOCKS + blockIdx.x] = ((sh[0][t] + sh[1][t]) + sh[2][t]) + sh[3][t];
}

// total of product blockIdx.x over the n blocks' partials: h (and host, when
// given); with sum (one block) also host[k] = a[k] + b[k] for k < m, the total in
// host[m] and its inverse root in scale
__global__ void __launch_bounds__(FG_THREADS) fg_final(const double* __restrict__ part, int n, double* __restrict__ h,
                                                       double* host, bool sum, int m, const double* __restrict__ a,
                                                       const double* __restrict__ b, double* __restrict__ scale)
{
    __shared__ double sh[FG_THREADS];
    const int t = threadIdx.x, k = blockIdx.x;
    double v = 0;
    UNROLL for (int q = 0; q < FG_BLOCKS / FG_THREADS; q++) {
        const int i = q * FG_THREADS + t;
        v += i < n ? part[(size_t)k * FG_BLOCKS + i] : 0.0;
    }
    sh[t] = v;
    __syncthreads();
    for (int o = FG_THREADS / 2; o > 0; o >>= 1) {
        if (t < o) sh[t] += sh[t + o];
        __syncthreads();
    }
    if (!sum) {
        if (t == 0) {
            h[k] = sh[0];
            if (host) host[k] = sh[0];
        }
        return;
    }
    if (t < m) host[t] = a[t] + b[t];
    if (t == 0) {
        host[m] = sh[0];
        *scale = 1 / sqrt(sh[0]);
    }
}

// E elements of p at i + 256 e; FULL: the block's whole tile lies below len,
// else 0 past the end
template <int E, bool FULL>
__device__ __forceinline__ void fg_load(const double* __restrict__ p, int64_t i, int64_t len, double (&v)[E])
{
    UNROLL for (int e = 0; e < E; e++) v[e] = FULL || i + FG_THREADS * e < len ? p[i + FG_THREADS * e] : 0.0;
}

template <int M, int E, bool FULL>
__device__ __forceinline__ void fg_dot_tile(const double* __restrict__ V, int64_t ldv, const double* __restrict__ w,
                                            int64_t i, int64_t len, double (&acc)[M])
{
    double wi[E];
    fg_load<E, FULL>(w, i, len, wi);
    UNROLL for (int k = 0; k < M; k++) {
        double v[E];
        fg_load<E, FULL>(V + (size_t)k * ldv, i, len, v);
        UNROLL for (int e = 0; e < E; e++) acc[k] += v[e] * wi[e];
    }
}

template <int M, int E>
__global__ void __launch_bounds__(FG_THREADS) fg_dot(const double* __restrict__ V, int64_t ldv,
                                                     const double* __restrict__ w, int64_t len, double* part)
{
    constexpr int64_t TILE = (int64_t)FG_THREADS * E;
    double acc[M];
    UNROLL for (int k = 0; k < M; k++) acc[k] = 0;
    int64_t b = (int64_t)blockIdx.x * TILE;
    for (; b + TILE <= len; b += gridDim.x * TILE) fg_dot_tile<M, E, true>(V, ldv, w, b + threadIdx.x, len, acc);
    if (b < len) fg_dot_tile<M, E, false>(V, ldv, w, b + threadIdx.x, len, acc);
    fg_partial<M>(acc, part);
}

template <int M, int E, bool FULL>
__device__ __forceinline__ void fg_update_tile(double* __restrict__ w, const double* __restrict__ V, int64_t ldv,
                                               const double* cs, int64_t i, int64_t len, double& nn)
{
    double wi[E];
    fg_load<E, FULL>(w, i, len, wi);
    UNROLL for (int k = 0; k < M; k++) {
        double v[E];
        fg_load<E, FULL>(V + (size_t)k * ldv, i, len, v);
        UNROLL for (int e = 0; e < E; e++) wi[e] -= cs[k] * v[e];
    }
    UNROLL for (int e = 0; e < E; e++) {
        if (FULL || i + FG_THREADS * e < len) w[i + FG_THREADS * e] = wi[e];
        nn += wi[e] * wi[e];
    }
}

// w -= V c; with NORM, also the partials of w.w
template <int M, int E, bool NORM>
__global__ void __launch_bounds__(FG_THREADS) fg_update(double* __restrict__ w, const double* __restrict__ V,
                                                        int64_t ldv, const double* __restrict__ c, int64_t len,
                                                        double* part)
{
    constexpr int64_t TILE = (int64_t)FG_THREADS * E;
    __shared__ double cs[32];
    if (threadIdx.x < M) cs[threadIdx.x] = c[threadIdx.x];
    __syncthreads();
    double acc[1] = {0};
    int64_t b = (int64_t)blockIdx.x * TILE;
    for (; b + TILE <= len; b += gridDim.x * TILE)
        fg_update_tile<M, E, true>(w, V, ldv, cs, b + threadIdx.x, len, acc[0]);
    if (b < len) fg_update_tile<M, E, false>(w, V, ldv, cs, b + threadIdx.x, len, acc[0]);
    if constexpr (NORM) fg_partial<1>(acc, part);
}

template <int M>
__global__ void __launch_bounds__(FG_THREADS) fg_orth(double* __restrict__ w, const double* __restrict__ V,
                                                      int64_t ldv, const double* __restrict__ h, int64_t len,
                                                      double* part)
{
    __shared__ double hs[32];
    if (threadIdx.x < M) hs[threadIdx.x] = h[threadIdx.x];
    __syncthreads();
    double acc[M];
    UNROLL for (int k = 0; k < M; k++) acc[k] = 0;
    for (int64_t i = (int64_t)blockIdx.x * FG_THREADS + threadIdx.x; i < len; i += (int64_t)gridDim.x * FG_THREADS) {
        double v[M];
        UNROLL for (int k = 0; k < M; k++) v[k] = V[(size_t)k * ldv + i];
        double wi = w[i];
        UNROLL for (int k = 0; k < M; k++) wi -= hs[k] * v[k];
        w[i] = wi;
        UNROLL for (int k = 0; k < M; k++) acc[k] += v[k] * wi;
    }
    fg_partial<M>(acc, part);
}

template <int B>
__global__ void __launch_bounds__(256) fg_scale(double* __restrict__ v, const double* __restrict__ w,
                                                const double* __restrict__ scale, double s, int64_t nb, int64_t len,
                                                const double* __restrict__ dinv0, double* __restrict__ pb,
                                                double* __restrict__ px0)
{
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= len) return;
    const double y = w[k] * (scale ? *scale : s);
    v[k] = y;
    const int64_t i = k / B;
    if (k == i * B && i < nb) {
        pb[i] = y;
        px0[i] = OMEGA * dinv0[i] * y;
    }
}

__global__ void __launch_bounds__(256) fg_axpy(double* __restrict__ x, const double* __restrict__ Z, int64_t ldz,
                                               int m, FgCoef y, int64_t len)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= len) return;
    double acc = x[i];
    for (int k = 0; k < m; k++) acc += y.y[k] * Z[(size_t)k * ldz + i];
    x[i] = acc;
}

unsigned grid256(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// ------------------------------------------------------------- PressureAmg
// Buffers without host data are zeroed on the stream whose kernels use them: a
// caller's stream need not be ordered with the default one.  setup() waits once.
template <class T>
int PressureAmg::dev(T** p, size_t count, const T* host, std::string& err)
{
    void* q = nullptr;
    if (count == 0) count = 1;
    hipError_t e = hipMalloc(&q, count * sizeof(T));
    if (e != hipSuccess) { err = std::string("hipMalloc: ") + hipGetErrorString(e); return -1; }
    mem_.push_back(q);
    if (host) e = hipMemcpy(q, host, count * sizeof(T), hipMemcpyHostToDevice);
    else e = hipMemsetAsync(q, 0, count * sizeof(T), st_);
    if (e != hipSuccess) { err = std::string("hipMemcpy: ") + hipGetErrorString(e); return -1; }
    *p = (T*)q;
    return 0;
}

PressureAmg::~PressureAmg()
{
    for (void* p : mem_) (void)hipFree(p);
}

int PressureAmg::setup(int64_t n, const std::vector<int64_t>& rp, const std::vector<int32_t>& col,
                       const std::vector<double>& w, hipStream_t st, std::string& err)
{
    st_ = st;
    amg::Graph g;
    g.n = n;
    g.rp = rp;
    g.ci = col;
    g.w = w;
    while (true) {
        Level L;
        L.n = g.n;
        L.nnz = (int64_t)g.ci.size();
        if (dev(&L.rp, g.rp.size(), g.rp.data(), err) || dev(&L.ci, g.ci.size(), g.ci.data(), err) ||
            dev(&L.a, (size_t)L.nnz, (const double*)nullptr, err) ||
            dev(&L.dinv, (size_t)L.n, (const double*)nullptr, err) ||
            dev(&L.b, (size_t)L.n, (const double*)nullptr, err) ||
            dev(&L.x, (size_t)L.n, (const double*)nullptr, err) ||
            dev(&L.r, (size_t)L.n, (const double*)nullptr, err))
            return -1;
        amg::Graph gc;
        amg::LevelMaps M;
        if (g.n <= DENSE_MAX || (int)lv_.size() + 1 >= MAX_LEVELS || !amg::coarsen(g, gc, M)) {
            lv_.push_back(L);
            break;
        }
        amg::Sell S;
        amg::sell_layout(g, M, gc.n, S);
        L.nc = gc.n;
        L.nq = (int64_t)S.row.size();
        L.ne = S.off.back();
        if (dev(&L.gp, M.gp.size(), M.gp.data(), err) || dev(&L.gs, M.gs.size(), M.gs.data(), err) ||
            dev(&L.off, S.off.size(), S.off.data(), err) || dev(&L.row, S.row.size(), S.row.data(), err) ||
            dev(&L.agg, M.agg.size(), M.agg.data(), err) || dev(&L.sci, (size_t)L.ne, (const int32_t*)nullptr, err) ||
            dev(&L.cagg, (size_t)L.ne, (const int32_t*)nullptr, err) ||
            dev(&L.src, (size_t)L.ne, (const int32_t*)nullptr, err) ||
            dev(&L.sa, (size_t)L.ne, (const double*)nullptr, err))
            return -1;
        hipLaunchKernelGGL(amg_sell_fill, dim3(grid256(L.nq)), dim3(256), 0, st, L.nq, L.off, L.row, L.rp, L.ci,
                           L.agg, L.sci, L.cagg, L.src);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) {
            err = std::string("amg_sell_fill: ") + hipGetErrorString(e);
            return -1;
        }
        lv_.push_back(L);
        g = std::move(gc);
    }
    if (lv_.back().n <= DENSE_MAX) {
        if (dev(&lu_, (size_t)DENSE_MAX * DENSE_MAX, (const double*)nullptr, err) ||
            dev(&inv_, (size_t)DENSE_MAX * DENSE_MAX, (const double*)nullptr, err) ||
            dev(&piv_, (size_t)DENSE_MAX, (const int32_t*)nullptr, err))
            return -1;
        // the levels whose vectors fit one workgroup's LDS
        int64_t rows = 0;
        for (int l = (int)lv_.size() - 1; l >= 0; l--) {
            rows += lv_[l].n;
            if (lv_[l].n > SM_TOP || rows > SM_ROWS || (int)lv_.size() - 1 - l > SM_LEVELS) break;
            small_ = l;
        }
    }
    const hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) { err = std::string("hipStreamSynchronize: ") + hipGetErrorString(e); return -1; }
    return 0;
}

#define OCPX_B_SWITCH(X)                                                                            \
    switch (B) {                                                                                    \
    X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14)                                     \
    default: return hipErrorInvalidValue;                                                           \
    }

hipError_t PressureAmg::values(int B, const double* val, const double* dinv, double* d0, hipStream_t st)
{
    Level& L0 = lv_[0];
    const unsigned nblk = (unsigned)((L0.n + 64 / B - 1) / (64 / B));
#define X(N) case N: hipLaunchKernelGGL(cpr_columns<N>, dim3(nblk), dim3(64), 0, st, L0.n, L0.rp, val, dinv, d0, L0.a); break;
    OCPX_B_SWITCH(X)
#undef X
    for (size_t l = 0; l < lv_.size(); l++) {
        Level& L = lv_[l];
        hipLaunchKernelGGL(amg_dinv, dim3(grid256(L.n)), dim3(256), 0, st, L.n, L.rp, L.a, L.dinv);
        if (l + 1 < lv_.size()) {
            Level& C = lv_[l + 1];
            hipLaunchKernelGGL(amg_gather, dim3(grid256(C.nnz)), dim3(256), 0, st, C.nnz, L.gp, L.gs, L.a, C.a);
            if (L.ne) hipLaunchKernelGGL(amg_sell, dim3(grid256(L.ne)), dim3(256), 0, st, L.ne, L.src, L.a, L.sa);
        }
    }
    const Level& Lc = lv_.back();
    if (Lc.n <= DENSE_MAX) {
        hipLaunchKernelGGL(amg_dense_lu, dim3(1), dim3(64), 0, st, (int)Lc.n, Lc.rp, Lc.ci, Lc.a, lu_, piv_);
        hipLaunchKernelGGL(amg_dense_inv, dim3(1), dim3(64), 0, st, (int)Lc.n, lu_, piv_, inv_);
    }
    return hipGetLastError();
}

hipError_t PressureAmg::small_cycle(double* x, hipStream_t st)
{
    SmallHier h{};
    h.nl = (int)lv_.size() - 1 - small_;
    h.nd = (int)lv_.back().n;
    h.inv = inv_;
    h.dinvd = lv_.back().dinv;
    for (int k = 0; k < h.nl; k++) {
        const Level& L = lv_[small_ + k];
        h.lv[k] = SmallLevel{(int)L.n, (int)L.nc, (int)L.nq, L.off, L.row, L.sci, L.cagg, L.sa, L.dinv};
    }
    hipLaunchKernelGGL(amg_small, dim3(1), dim3(SM_THREADS), 0, st, h, lv_[small_].b, x);
    return hipGetLastError();
}

// Level l with its right-hand side in b and its first sweep in x; the result
// goes to xo, which is another array (a sweep reads its neighbours' x).
hipError_t PressureAmg::cycle(int l, double* xo, hipStream_t st)
{
    Level& L = lv_[l];
    if (l == small_) return small_cycle(xo, st);
    if (l + 1 == (int)lv_.size()) {           // no dense level: a few sweeps
        double *in = L.x, *out = L.r;
        for (int k = 0; k < 9; k++) {
            hipLaunchKernelGGL(amg_smooth, dim3(grid256(L.n)), dim3(256), 0, st, L.n, L.rp, L.ci, L.a, L.dinv, L.b, in, out);
            std::swap(in, out);
        }
        if (in != xo) return hipMemcpyAsync(xo, in, (size_t)L.n * sizeof(double), hipMemcpyDeviceToDevice, st);
        return hipGetLastError();
    }
    Level& C = lv_[l + 1];
    hipLaunchKernelGGL(amg_down, dim3(grid256(L.nq)), dim3(256), 0, st, L.nq, L.nc, L.off, L.row, L.sci, L.sa, L.b,
                       L.x, C.dinv, C.b, C.x);
    hipError_t e = cycle(l + 1, C.r, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(amg_up, dim3(grid256(L.nq)), dim3(256), 0, st, L.nq, L.off, L.row, L.sci, L.cagg, L.sa, L.dinv,
                       L.b, L.x, C.r, xo);
    return hipGetLastError();
}

hipError_t PressureAmg::vcycle(double* x, hipStream_t st)
{
    return cycle(0, x, st);
}

// --------------------------------------------------------------- launchers
hipError_t run_gs_color(int B, const int32_t* rows, int64_t nrows, const int64_t* rowptr, const int32_t* col,
                        const double* val, const double* dinv, const double* rhat, double* x, hipStream_t st)
{
    if (nrows == 0) return hipSuccess;
    const unsigned nblk = (unsigned)((nrows + 64 / B - 1) / (64 / B));
#define X(N) case N: hipLaunchKernelGGL(gs_color<N>, dim3(nblk), dim3(64), 0, st, rows, nrows, rowptr, col, val, \
                                        dinv, rhat, x); break;
    OCPX_B_SWITCH(X)
#undef X
    return hipGetLastError();
}

hipError_t run_cpr_resid(int B, const int64_t* rowptr, const int32_t* col, const double* d0, const double* px,
                         const double* v, double* R, double* z, int64_t nb, hipStream_t st)
{
    if (nb == 0) return hipSuccess;
    const unsigned nblk = (unsigned)((nb + 64 / B - 1) / (64 / B));
#define X(N) case N: hipLaunchKernelGGL(cpr_resid<N>, dim3(nblk), dim3(64), 0, st, rowptr, col, d0, px, v, R, z, nb); break;
    OCPX_B_SWITCH(X)
#undef X
    return hipGetLastError();
}

hipError_t run_cpr_half(int B, int which, const int32_t* rows, int64_t nrows, const int64_t* rowptr,
                        const int32_t* col, const double* val, const double* dinv, const double* px,
                        const double* v, double* R, double* z, double* w, hipStream_t st)
{
    if (nrows == 0) return hipSuccess;
    const unsigned nblk = (unsigned)((nrows + 64 / B - 1) / (64 / B));
#define X(N) case N: if (which) hipLaunchKernelGGL((cpr_half<N, true>), dim3(nblk), dim3(64), 0, st, rows, nrows, rowptr, col, val, dinv, px, v, R, z, w); \
        else hipLaunchKernelGGL((cpr_half<N, false>), dim3(nblk), dim3(64), 0, st, rows, nrows, rowptr, col, val, dinv, px, v, R, z, w); break;
    OCPX_B_SWITCH(X)
#undef X
    return hipGetLastError();
}

hipError_t run_fg_scale(int B, double* v, const double* w, const double* scale, double s, int64_t nb, int64_t len,
                        const double* dinv0, double* pb, double* px0, hipStream_t st)
{
    if (len == 0) return hipSuccess;
#define X(N) case N: hipLaunchKernelGGL(fg_scale<N>, dim3(grid256(len)), dim3(256), 0, st, v, w, scale, s, nb, len, dinv0, pb, px0); break;
    OCPX_B_SWITCH(X)
#undef X
    return hipGetLastError();
}
#undef OCPX_B_SWITCH

int fg_scratch_len() { return FG_BLOCKS * 32; }

// blocks of tiles of e elements per thread, and whether E = 8 fills the device
static unsigned fg_blocks(int64_t len, int e)
{
    const int64_t b = (len + (int64_t)FG_THREADS * e - 1) / ((int64_t)FG_THREADS * e);
    return (unsigned)(b < 1 ? 1 : (b > FG_BLOCKS ? FG_BLOCKS : b));
}
static bool fg_wide(int64_t len) { return len >= (int64_t)512 * FG_THREADS * FG_E; }

#define OCPX_M_LOW(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16)
#define OCPX_M_HIGH(X) X(17) X(18) X(19) X(20) X(21) X(22) X(23) X(24) X(25) X(26) X(27) X(28) X(29) X(30) X(31)
static_assert(FG_MAX == 31 && ORTH_M == 16, "the cases of OCPX_M_LOW and OCPX_M_HIGH");

static hipError_t fg_sum(const double* part, unsigned n, int m, double* h, double* host, hipStream_t st)
{
    hipLaunchKernelGGL(fg_final, dim3(m), dim3(FG_THREADS), 0, st, part, (int)n, h, host, false, 0, nullptr, nullptr, nullptr);
    return hipGetLastError();
}

hipError_t run_fg_dot(const double* V, int64_t ldv, int m, const double* w, int64_t len, double* part, double* h,
                      double* host, hipStream_t st)
{
    const unsigned nw = fg_blocks(len, FG_E), n1 = fg_blocks(len, 1);
#define X(M) case M: if (fg_wide(len)) hipLaunchKernelGGL((fg_dot<M, FG_E>), dim3(nw), dim3(FG_THREADS), 0, st, V, ldv, w, len, part); \
        else hipLaunchKernelGGL((fg_dot<M, 1>), dim3(n1), dim3(FG_THREADS), 0, st, V, ldv, w, len, part); break;
    switch (m) {
    OCPX_M_LOW(X) OCPX_M_HIGH(X)
    default: return hipErrorInvalidValue;
    }
#undef X
    return fg_sum(part, fg_wide(len) ? nw : n1, m, h, host, st);
}

hipError_t run_fg_orth(double* w, const double* V, int64_t ldv, int m, const double* h, int64_t len, double* part,
                       double* h2, hipStream_t st)
{
    const unsigned nw = fg_blocks(len, FG_E), n1 = fg_blocks(len, 1);
#define X(M) case M: hipLaunchKernelGGL(fg_orth<M>, dim3(n1), dim3(FG_THREADS), 0, st, w, V, ldv, h, len, part); \
        return fg_sum(part, n1, m, h2, nullptr, st);
#define Y(M) case M: if (fg_wide(len)) hipLaunchKernelGGL((fg_update<M, FG_E, false>), dim3(nw), dim3(FG_THREADS), 0, st, w, V, ldv, h, len, part); \
        else hipLaunchKernelGGL((fg_update<M, 1, false>), dim3(n1), dim3(FG_THREADS), 0, st, w, V, ldv, h, len, part); break;
    switch (m) {
    OCPX_M_LOW(X) OCPX_M_HIGH(Y)
    default: return hipErrorInvalidValue;
    }
#undef X
#undef Y
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? run_fg_dot(V, ldv, m, w, len, part, h2, nullptr, st) : e;
}

hipError_t run_fg_orth_norm(double* w, const double* V, int64_t ldv, int m, const double* h, const double* h2,
                            int64_t len, double* part, double* host, double* scale, hipStream_t st)
{
    const unsigned nw = fg_blocks(len, FG_E), n1 = fg_blocks(len, 1);
#define X(M) case M: if (fg_wide(len)) hipLaunchKernelGGL((fg_update<M, FG_E, true>), dim3(nw), dim3(FG_THREADS), 0, st, w, V, ldv, h2, len, part); \
        else hipLaunchKernelGGL((fg_update<M, 1, true>), dim3(n1), dim3(FG_THREADS), 0, st, w, V, ldv, h2, len, part); break;
    switch (m) {
    OCPX_M_LOW(X) OCPX_M_HIGH(X)
    default: return hipErrorInvalidValue;
    }
#undef X
    hipLaunchKernelGGL(fg_final, dim3(1), dim3(FG_THREADS), 0, st, part, (int)(fg_wide(len) ? nw : n1), nullptr, host, true, m, h,
                       h2, scale);
    return hipGetLastError();
}
#undef OCPX_M_LOW
#undef OCPX_M_HIGH

hipError_t run_fg_axpy(double* x, const double* Z, int64_t ldz, int m, const FgCoef& y, int64_t len, hipStream_t st)
{
    if (len == 0) return hipSuccess;
    if (m < 0 || m > 32) return hipErrorInvalidValue;
    hipLaunchKernelGGL(fg_axpy, dim3(grid256(len)), dim3(256), 0, st, x, Z, ldz, m, y, len);
    return hipGetLastError();
}

}  // namespace ocpx
