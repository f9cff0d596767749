// Grouped truncated SVD and symmetric eigensolver on the device (FP64).
//
// Small problems (min(m, n) <= LMAX) are solved directly: two passes of Gram
// matrix on MFMA, k_precond, rotation, which leave graded, nearly orthogonal
// columns (whose Gram matrix is then relatively accurate), one of parallel-order
// Jacobi in LDS, column norms; the smallest by two Jacobi passes.  Larger problems run block subspace
// iteration (Y = M V, Z = M^T U; Y = M V for eigenpairs) with a pivoted
// Cholesky QR step after every product, until the top-k subspace has
// converged to working precision; the Ritz triplets (pairs) are then extracted
// by Gram/Jacobi steps.  All problems of a call advance together in grouped
// launches.
#pragma once

#include <vector>

#include "blocktensor.h"

namespace tnr {

struct SvdIn {
    const double* M;     // m x n, column-major, leading dim ld
    int m, n, ld;
    int kmax;            // triplets wanted, <= min(m, n)
    uint64_t seed;
};

struct SvdOut {
    Buf U, V, s;         // U: m x kmax (ld m), V: n x kmax (ld n), s: kmax
    int ldu = 0, ldv = 0;
    std::vector<double> s_host;
    int iters = 0;       // subspace iterations (0 = direct)
    double conv = 0.0;   // accumulated contraction bound of the top-k subspace
    int status = 0;      // TNR_OK, TNR_ERR_NOCONV or TNR_ERR_NONFINITE (see below)
};

void svd_grouped(Ctx& ctx, const std::vector<SvdIn>& in, std::vector<SvdOut>& out);

struct EighIn {
    double* M;           // n x n symmetric (symmetrised in place), leading dim ld
    int n, ld;
    int kmax;
    uint64_t seed;
};

struct EighOut {
    Buf U, lam;          // U: n x ncols (ld n), lam: ncols, by |lambda| descending
    int ncols = 0;       // n (direct) or the block size (iterative)
    std::vector<double> lam_host;
    bool direct = false; // all n eigenvalues available
    int iters = 0;
    double conv = 0.0;
    int status = 0;      // TNR_OK, TNR_ERR_NOCONV or TNR_ERR_NONFINITE (see below)
};

void eigh_grouped(Ctx& ctx, const std::vector<EighIn>& in, std::vector<EighOut>& out);

// Per-problem status: TNR_ERR_NOCONV for a problem whose block iteration
// reaches max_iters with the accumulated contraction bound still above
// conv_target, or any of whose Jacobi solves reaches its sweep cap with a
// rotation still due (the reference's LAPACK-backed svd_trunc and
// eigh_trunc! raise there); TNR_ERR_NONFINITE for a problem with a NaN or
// infinite singular value / eigenvalue, whose host values are then zeroed so
// the global truncation stays well defined.  Other problems of the group are
// unaffected.
//
// Solver knobs (the autotuner may override them).
struct SolverCfg {
    double jacobi_tol = 1e-15;   // relative off-diagonal threshold (final Ritz extraction, direct)
    int jacobi_sweeps = 40;
    // Rayleigh-Ritz inside the block iteration: the loop takes such steps, with
    // these thresholds and k_conv, only where cholqr_y, cholqr_z or cholqr_eigh
    // is 0.  Measured with them on BTRG chi = 32 beta
    // scans: looser thresholds or sweep caps here make the iteration
    // and the final extraction take longer than they save, so the loop
    // keeps a tight threshold; V is still rebuilt at full accuracy (1e-15)
    // once the loop ends.
    double jacobi_tol_iter = 1e-10;
    // The first iteration's Rayleigh-Ritz step only aligns the random start
    // basis; later steps refine it.  Measured on single BTRG chi = 32 runs
    // (beta 0.44): 1e-4 takes 3 % less time than 1e-10, 1e-6 .. 1e-2 2 %.
    double jacobi_tol_first = 1e-4;
    int jacobi_sweeps_iter = 40;
    double null_rtol = 1e-14;    // columns below this x sigma_max are null
    double conv_target = 1e-14;  // accumulated contraction of the top-k subspace angle
    double block_mult = 2.0;     // block width max(block_mult k, k + block_extra) <= LMAX
    // Block iteration orthonormalisation by pivoted Cholesky QR instead of
    // Rayleigh-Ritz: the Y side (cholqr_y), the Z side (cholqr_z; the
    // stopping rule then reads the pivots R_jj) and the eigensolver's loop
    // (cholqr_eigh).  Without Rayleigh-Ritz in the loop the iteration is a
    // simultaneous iteration: its basis vectors converge to the singular
    // vectors one by one, so the Gram matrices of the final extraction are
    // nearly diagonal and cheap for Jacobi.  Measured on single BTRG
    // chi = 32 runs: 17 % less time with the Z side on Cholesky QR.  The
    // eigensolver's steps keep every direction (span): its spectra are
    // squares, and after a random start whatever lies below 1e-8 of the
    // largest value is beyond the Gram matrix's resolution; dropped there, it
    // ended HOTRG chi = 48 solves early (1e-7 norm errors).  Rayleigh-Ritz ->
    // Cholesky QR in its loop: HOTRG chi 16 20.5 -> 14.6 ms, chi 32 59.1 ->
    // 41.5 (7 steps), the same number of iterations.
    bool cholqr_y = true;
    bool cholqr_z = true;
    bool cholqr_eigh = true;
    // Steps that rebuild V from the last Z and that extract the Ritz triplets
    // from Y = M V.  With Cholesky QR on the Z side V takes rv_passes Cholesky
    // QR steps (1 leaves it orthonormal to the Gram matrix's resolution only);
    // the basis vectors of the simultaneous iteration are close to the singular
    // vectors, so the columns of M V are graded and well conditioned after
    // scaling, and one Jacobi pass on them has the relative accuracy that a
    // second pass gives.  A Jacobi basis of Z instead costs two more solves:
    // BTRG chi 32 21.9 -> 20.2 ms, Z2 chi 64 69.5 -> 66.1, ATRG Z2 chi 16 21.7 ->
    // 20.1 without them, errors against LAPACK the same.
    int rv_passes = 2;
    int rf_passes = 1;
    int block_extra = 2;
    int min_iters = 2;
    int max_iters = 80;
    // from this iteration on, a block iteration of a matrix small enough to
    // be refactorised whole stops as soon as even twice its current
    // convergence rate could not reach conv_target by max_iters (it would
    // stall and be factorised whole anyway); 0 iterates to max_iters
    int stall_from = 8;
};
SolverCfg& solver_cfg();
// Defaults, then TNR_SOLVER_CFG, then `spec` ("key=value,...", see
// solver.cpp); not while other calls are running.
void set_solver_cfg(const char* spec);

}  // namespace tnr
