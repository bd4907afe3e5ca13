// f2d_modal.hpp -- direct solve of the 5-point Poisson/Helmholtz operator of
// a fully wet rectangle of any size by the eigenvectors of its two second
// differences (internal interface of the library).
//
// On a rectangle the operator of get_Laplacian_sparse (elliptic.py:114-195)
// is cx D_x + cy D_y - maindiag, D the second difference of one direction:
// its eigenvectors are sines on the n - 1 vertices between two Dirichlet
// lines ("wall"), Fourier modes on a periodic direction ("ring"), cosines on
// the n cells between two Neumann walls ("even").  With the orthonormal
// eigenvectors as the columns of Qx, Qy,
//   x = Qy ((Qy^T b Qx) / lambda) Qx^T,
// four dense products: no restriction to power-of-two sizes, no iteration.
// A zero eigenvalue (the constant of a singular operator) is dropped, which
// is the zero-mean solution of the zero-mean right-hand side.
#pragma once
#include "f2d_common.hpp"

namespace f2d {

struct ModalSolver;

// every vertex strictly inside the domain is an unknown (cells: every cell)
// and the sizes lie in [8, 4096] (a halo point is the image of one unknown)
bool modal_applicable(int64_t ny, int64_t nx, int xper, int yper, int64_t nwet, bool cells);

// single: FP32 solves are to be measured (modal_solve), from FP64 results
ModalSolver* modal_create(int64_t ny, int64_t nx, double dx, double dy, double maindiag,
                          int xper, int yper, bool cells, bool single = false);
void modal_destroy(ModalSolver* m);

// x = A^-1 b at the unknowns and their periodic halo images, on the padded
// layout; TB is b's and TX x's type, the arithmetic is FP64.  gmode 0: b
// given at the unknowns; 1 (vertices): b = centerstovertices of the cell
// field (operators.py:126-133, formed inside the first transform: the
// averaged eigenvectors).  measure: the relative residual goes to `stats` (8
// doubles, device), as the other direct solves record it, converged up to
// accept.  skip: a device
// flag; the passes of a solve enqueued behind a nonzero one do nothing.
// only: a mask on the padded layout; x is written where it is set, without
// halo images.
template <class TB, class TX>
void modal_solve(ModalSolver* m, const TB* b, int gmode, TX* x, bool measure, double accept,
                 double* stats, hipStream_t s, const double* skip = nullptr, const int8_t* only = nullptr);

}  // namespace f2d
