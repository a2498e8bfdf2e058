// kf_direct.h -- direct solver of the shifted stencil, x = (L_h - c)^-1 b.
//
// kielflow's 7-point stencil (solver_poisson_jacobi_nlin.cpp:177-199) is a
// sum of one second difference per axis, each with coefficients of that
// axis alone.  With the eigenvectors of the three second differences,
// (L_h - c)^-1 is a transform along each axis, a division by
// lambda_x + lambda_y + lambda_z - c, and the transforms back (the fast
// diagonalisation method of Lynch, Rice and Thomas 1964).  On an
// equidistant grid the eigenvectors are Fourier modes and the transforms the
// library's FFT passes; on a stretched axis they are a dense matrix and the
// transforms matrix products on the matrix cores.
//
// It serves as the approximate inverse of J = L_h - diag(e): with c near e,
// an iteration leaves about |e - c| / (|lambda| + c) of the error (0.01 to
// 0.1 for a grain in a plasma; a V-cycle 0.1), for one pass of each axis
// forth and back instead of a V-cycle's sweeps on every level.  Measured
// against V-cycles (BiCGStab around them on stretched grids): the first solve
// of a run 6.2 -> 0.94 ms at 192x128x192 equidistant FP64 and 6.5 -> 0.34 ms
// at 64^3 hyperbolic; an RK4 step 14.8 -> 12.1 ms (256^3 mixed), 26.9 -> 19.4
// (256^3 FP64), 18.9 -> 7.9 (128^3 sine FP64).
#pragma once

#include <vector>

#include "kf_common.h"
#include "kf_fft.h"
#include "kf_axes.h"

namespace kf {

template <typename R>
class Direct {
  public:
    // h[d][i] = x_i - x_{i-1}, i = 0..n_d (the solver's spacings)
    // like: a plan of the grid's lengths that is there already, or null
    Direct(const AxisDesc ax[3], const std::vector<double> h[3], hipStream_t s, const fft::Plan<R> *like = nullptr);
    ~Direct();
    Direct(const Direct &) = delete;
    Direct &operator=(const Direct &) = delete;
    // whether the grid's axes admit it: equidistant, or spacings that mirror
    // about the axis' first point (the maps of SiSt and HySt with
    // l0 = -L/2): their even and odd modes are eigenvectors of tridiagonal
    // matrices
    static bool possible(const AxisDesc ax[3], const std::vector<double> h[3]);
    // x = (L_h - c)^-1 b, *c > 0 in device memory; every kernel returns at
    // once when ctl[0] is set; x may not be b
    void solve(const R *b, R *x, const double *c, const int *ctl, hipStream_t s);

  private:
    void release();
    void solve_fourier(const R *b, R *x, const double *c, const int *ctl, hipStream_t s);
    void x_pass(const double *c, const int *ctl, hipStream_t s);
    void solve_modal(const R *b, R *x, const double *c, const int *ctl, hipStream_t s);
    int n_[3];
    bool fourier_;
    fft::Plan<R> plan_{};  // equidistant grids
    R *pool_ = nullptr;    // the tables below
    const R *lam_[3] = {};  // eigenvalues of the axes (equidistant: of the half spectrum along z)
    // stretched grids: T^-1 and T of the x and y axes, their transposes for z
    const R *fwd_[3] = {}, *inv_[3] = {};
    R *tmp_ = nullptr;     // a real field between the products
};

}  // namespace kf
