// cpr.hpp — the CPR-type preconditioner of the device linear solve and the
// FGMRES pieces around it (cpr.hip).
//
// The reference decouples the FIM system with ABF (each block row times the
// inverse of its diagonal block, src/Decoupling.cpp:23-57, 426-499) and
// solves it with FGMRES(30) preconditioned by FASP's two-stage pressure /
// full-system preconditioner (data/spe5/bsr.fasp: unsmoothed-aggregation AMG
// with pairwise matching on the pressure block, one V-cycle).  Here:
//
//  * PressureAmg: the pressure block of the decoupled system, A_p(i, j) =
//    row 0 of D_i^{-1} times column 0 of A_ij, made an M-matrix (positive
//    off-diagonal entries moved to the diagonal, the diagonal at least the
//    off-diagonal magnitudes' sum).  Its aggregation hierarchy is
//    built once per context on the host from the transmissibility graph
//    (pairwise matching on the strongest connection, twice per level, so
//    aggregates of up to four cells); every solve forms the level matrices
//    on the device (level 0 from the BSR, coarser ones by Galerkin sums over
//    a precomputed gather list) and applies one V-cycle: one weighted-Jacobi
//    sweep before and after the coarse correction, a product with the dense
//    inverse (formed once per solve) on the coarsest level.
//  * the second stage: one multicolour block Gauss-Seidel sweep on the
//    decoupled system (whose diagonal blocks are the identity), colours
//    from a greedy colouring of the block graph.  With two colours (any
//    Cartesian grid) the sweep and the operator that follows it share one
//    read of the matrix (cpr.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

namespace ocpx {

class PressureAmg {
public:
    PressureAmg() = default;
    PressureAmg(const PressureAmg&) = delete;
    PressureAmg& operator=(const PressureAmg&) = delete;
    ~PressureAmg();

    // Hierarchy from the level-0 pattern (block rows of the bulk system:
    // rowptr, col with the diagonal first in each row) and the weight of
    // every off-diagonal slot (its connection's transmissibility).  Buffers are
    // zeroed on st and ready on return.
    int setup(int64_t n, const std::vector<int64_t>& rp, const std::vector<int32_t>& col,
              const std::vector<double>& w, hipStream_t st, std::string& err);
    bool ready() const { return !lv_.empty(); }
    int levels() const { return (int)lv_.size(); }
    int64_t rows(int l) const { return lv_[l].n; }

    // Level matrices of the current system: val the bulk BSR (B x B blocks,
    // row-major), dinv the inverses of its diagonal blocks, d0 [nnzb][B] receives
    // column 0 of every decoupled block D_i^{-1} A_ij.
    hipError_t values(int B, const double* val, const double* dinv, double* d0, hipStream_t st);
    // x = one V-cycle applied to b; b is already in place: level0_b() and
    // level0_x() (= OMEGA Dinv b) hold the level-0 right-hand side and its first sweep
    hipError_t vcycle(double* x, hipStream_t st);
    double* level0_b() { return lv_[0].b; }
    double* level0_x() { return lv_[0].x; }
    const double* level0_dinv() const { return lv_[0].dinv; }

    static constexpr int DENSE_MAX = 64;     // the coarsest level is solved densely up to this size
    static constexpr double OMEGA = 2.0 / 3.0;   // weighted-Jacobi smoother

private:
    struct Level {
        int64_t n = 0, nnz = 0;
        int64_t* rp = nullptr;
        int32_t* ci = nullptr;
        double *a = nullptr, *dinv = nullptr, *b = nullptr, *x = nullptr, *r = nullptr;
        // to the next level (all but the last)
        int64_t *gp = nullptr, *gs = nullptr;   // coarse slot s = sum of a[gs[gp[s] .. gp[s+1])]
        // the level's matrix in V-cycle order (amg::Sell); ne entries
        int64_t nc = 0, nq = 0, ne = 0;
        int64_t* off = nullptr;
        int32_t *row = nullptr, *agg = nullptr, *sci = nullptr, *cagg = nullptr, *src = nullptr;
        double* sa = nullptr;
    };
    std::vector<Level> lv_;
    int small_ = -1;                         // first level of the one-workgroup part of the cycle, -1 none
    double *lu_ = nullptr, *inv_ = nullptr;  // dense LU and inverse of the coarsest level (DENSE_MAX^2)
    int32_t* piv_ = nullptr;
    std::vector<void*> mem_;
    hipStream_t st_ = nullptr;               // setup()'s stream
    template <class T>
    int dev(T** p, size_t count, const T* host, std::string& err);
    hipError_t cycle(int l, double* x, hipStream_t st);
    hipError_t small_cycle(double* x, hipStream_t st);
};

// x_i = rhat_i - Dinv_i sum_{j != i} A_ij x_j for the rows of one colour
hipError_t run_gs_color(int B, const int32_t* rows, int64_t nrows, const int64_t* rowptr, const int32_t* col,
                        const double* val, const double* dinv, const double* rhat, double* x, hipStream_t st);

// ---- FGMRES pieces on vectors of len doubles (partials are summed in block
// order, so results have the same bits on every run).  part: fg_scratch_len()
// doubles.
int fg_scratch_len();
// h[k] = V_k . w for k < m (V: m vectors, stride ldv; m <= 31); host (pinned, may be null) gets a copy
hipError_t run_fg_dot(const double* V, int64_t ldv, int m, const double* w, int64_t len, double* part, double* h,
                      double* host, hipStream_t st);
// w -= sum h[k] V_k, then h2[k] = V_k . w
hipError_t run_fg_orth(double* w, const double* V, int64_t ldv, int m, const double* h, int64_t len, double* part,
                       double* h2, hipStream_t st);
// w -= sum h2[k] V_k; host[k] = h[k] + h2[k], host[m] = w . w; *scale = 1 / |w|
hipError_t run_fg_orth_norm(double* w, const double* V, int64_t ldv, int m, const double* h, const double* h2,
                            int64_t len, double* part, double* host, double* scale, hipStream_t st);
// v = w * (scale ? *scale : s); for the nb bulk rows pb = v's pressure entries and px0 = OMEGA dinv0 pb
hipError_t run_fg_scale(int B, double* v, const double* w, const double* scale, double s, int64_t nb, int64_t len,
                        const double* dinv0, double* pb, double* px0, hipStream_t st);
struct FgCoef { double y[32]; };
// x += sum_{k < m} y[k] Z_k
hipError_t run_fg_axpy(double* x, const double* Z, int64_t ldz, int m, const FgCoef& y, int64_t len, hipStream_t st);

// R = v - Dinv J x1 and z = R + x1 on the bulk rows, x1 the pressure correction px (0 in the other entries)
hipError_t run_cpr_resid(int B, const int64_t* rowptr, const int32_t* col, const double* d0, const double* px,
                         const double* v, double* R, double* z, int64_t nb, hipStream_t st);
// the second and the first colour of a two-colour graph (which = 1, 0), see cpr.hip
hipError_t run_cpr_half(int B, int which, const int32_t* rows, int64_t nrows, const int64_t* rowptr,
                        const int32_t* col, const double* val, const double* dinv, const double* px,
                        const double* v, double* R, double* z, double* w, hipStream_t st);

}  // namespace ocpx
