// f2d_modal_plan.hpp -- extents of the eigenvector solve's matrices and the
// choice of its tiles (f2d_modal.hip).  Host arithmetic only, without HIP: a
// CPU test walks every size, kind of direction and tile of it.
#pragma once
#include <cstdint>

namespace f2d {

enum { BC_RING = 0, BC_WALL = 1, BC_EVEN = 2 };

// Output tiles of a pass (rows = pairs) and the contraction pairs of a chunk.
struct ModalTile {
  int b, kc;
};
constexpr ModalTile MODAL_TILES[3] = {{64, 8}, {32, 16}, {16, 32}};

// A pass loads whole tiles of matrix columns and whole chunks of its rows,
// unclamped: the columns are padded to the widest tile, the rows to the
// longest chunk, with zeros.
constexpr int MODAL_PITCH = 64, MODAL_CHUNK = 32;

constexpr int modal_up(int v, int m) { return (v + m - 1) / m * m; }

// one direction of n cells
struct ModalSizes {
  int bc = 0, n = 0;              // kind, cells
  int pts = 0, refl = 0, nh = 0;  // unknowns, mirror of p is refl - p, mirror pairs
  int ne = 0, no = 0;             // even and odd modes
  int cpts = 0, crefl = 0, cnh = 0;  // points, mirror, pairs of a cell field
  // rows and pitch of the matrices: points to modes, modes to points, and
  // (KC rows, pitch LF) cells to modes
  int KF = 0, LF = 0, KB = 0, LB = 0, KC = 0;
};

inline ModalSizes modal_sizes(int bc, int n) {
  ModalSizes d;
  d.bc = bc;
  d.n = n;
  d.pts = bc == BC_WALL ? n - 1 : n;
  d.refl = bc == BC_WALL ? n - 2 : (bc == BC_EVEN ? n - 1 : n);
  d.nh = bc == BC_RING ? n / 2 + 1 : (d.pts + 1) / 2;
  d.ne = bc == BC_WALL ? n / 2 : (bc == BC_RING ? n / 2 + 1 : (n + 1) / 2);
  d.no = d.pts - d.ne;
  d.cpts = n;
  d.crefl = n - 1;
  d.cnh = (n + 1) / 2;
  d.KF = modal_up(d.nh, MODAL_CHUNK);
  d.LF = modal_up(d.ne, MODAL_PITCH);
  d.KB = modal_up(d.ne, MODAL_CHUNK);
  d.LB = modal_up(d.nh, MODAL_PITCH);
  d.KC = modal_up(d.cnh, MODAL_CHUNK);
  return d;
}

inline int64_t modal_tiles(int m, int nj, int b) {
  return (int64_t)((m + b - 1) / b) * ((nj + b - 1) / b);
}

// The tile of a pass of m rows and nj output pairs, an index of MODAL_TILES.
// Measured on closed n x n grids (us a solve): 64 x 64 tiles fill the chip
// from about 640 of them (3000 x 2000: 1129 against 1306 with 32 x 32;
// 1600^2, 325 tiles: 505 against 380), 32 x 32 from about 400 (1000^2, 512
// tiles: 119 against 150 with 16 x 16; 1000 x 600, 304 tiles: 97 against
// 87), below them 16 x 16 tiles whose four waves split the contraction
// (256^2: 19 against 29; 40^2: 13.5 against 15.2).
inline int modal_tile(int m, int nj) {
  if (modal_tiles(m, nj, 64) >= 640) return 0;
  return modal_tiles(m, nj, 32) >= 400 ? 1 : 2;
}

}  // namespace f2d
