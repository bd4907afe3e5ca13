// f2d_modal.hip -- eigenvector (dense transform) solve of the rectangle's
// 5-point operator for sizes the FFT solve does not take (f2d_modal.hpp has
// the mathematics).  It replaces, for those sizes, the factorisation and
// back-substitution of Poisson2D (elliptic.py:71-87).
//
// Every eigenvector is even or odd about the middle of its direction, so a
// transform of n points folds into two products of half the size: with
// e = v(p) + v(p'), o = v(p) - v(p') over the mirror pairs (p, p'), the even
// modes take e and the odd ones o; on the way back the pair is u_e + u_o and
// u_e - u_o.  That halves the operations.  All four passes are one kernel,
// "contract the contiguous index, store the result transposed":
//   pass 1  b (padded, or the cell field with the averaged eigenvectors)
//           -> modes of x, rows of y
//   pass 2  -> modes of y, scaled by 1 / lambda
//   pass 3  -> points of x
//   pass 4  -> x (padded, with its periodic halo images)
// The products run on v_mfma_f64_16x16x4 from LDS tiles; even and odd parts
// travel as one pair, so one 16-byte LDS read feeds two MFMAs.
//
// What bounds it: the FP64 matrix rate from about 1000 points a side (a
// square solve is 2 n^3 multiply-adds: 1000^2 119 us, 34 TFLOP/s; 4096^2
// 4.65 ms, 59 TFLOP/s of the 71 a large library product reaches), launch and
// load latency below (four launches: 40^2 13.5 us, 256^2 19 us, 800 x 304
// 38 us).  An even/odd operand pair is an ext_vector and not a HIP struct:
// as double2 the prefetched pairs went through scratch memory, 3 times slower.
#include <cmath>
#include <vector>

#include "f2d_modal.hpp"
#include "f2d_modal_plan.hpp"

namespace f2d {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d4 __attribute__((ext_vector_type(4)));

// one pass: out(j, m) = sum_k mat[k][j] in(m, k), even and odd parts at once
struct ModalPass {
  const d2* mat;  // [K][LJ], {even, odd}, zero beyond its rows and columns
  const void* in;      // row m at in + m * ldi
  void* out;
  int64_t ldi, ldo;
  int M;               // rows of the input
  int K, LJ;           // padded contraction length, pitch of mat (ModalSizes)
  int nk;              // contraction pairs (forward: mirror pairs; back: modes)
  int npts, refl;      // forward: points of the direction, mirror of p is refl - p
  int ne, no;          // even and odd modes
  int nj;              // output pairs (forward: modes; back: mirror pairs)
  // pass 2: eigenvalues lam_m[m] + lam_j[mode]
  const double *lam_m, *lam_j;
  // pass 4: first unknown of the padded array, wrap sizes (0: closed)
  int64_t x0;
  int wx, wy;          // periods for the halo images of columns and rows
  const int8_t* only;  // pass 4: write at the set points only (may be NULL)
  const double* skip;  // device flag: nonzero, the pass does nothing (may be NULL)
};

enum { EPI_MODES = 0, EPI_SCALED = 1, EPI_POINTS = 2, EPI_PADDED = 3 };

__device__ __forceinline__ double inv_lam(double l) { return l != 0.0 ? 1.0 / l : 0.0; }

// value v of the unknown in padded row/column order (r, c) and its periodic
// images; a closed direction has none
template <class T>
__device__ __forceinline__ void put_wrapped(T* x, const ModalPass& a, int r, int c, T v) {
  const int64_t k = a.x0 + (int64_t)r * a.ldo + c;
  if (a.only) {
    if (a.only[k]) x[k] = v;
    return;
  }
  const int64_t sx = !a.wx ? 0 : (c < 3 ? a.wx : (c >= a.wx - 3 ? -a.wx : 0));
  const int64_t sy = !a.wy ? 0 : (r < 3 ? (int64_t)a.wy * a.ldo
                                        : (r >= a.wy - 3 ? -(int64_t)a.wy * a.ldo : 0));
  x[k] = v;
  if (sx) x[k + sx] = v;
  if (sy) x[k + sy] = v;
  if (sx && sy) x[k + sx + sy] = v;
}

// Workgroup tile: BM rows x BN output pairs, 256 threads as WM x WN x WK
// waves of 16 MT rows x 16 NT pairs; the WK waves of a tile split each
// chunk's contraction steps and are summed through LDS at the end (fixed
// order).  A chunk is KC contraction pairs.  The loads of D chunks are in
// flight in registers (an operand comes from another XCD's writes, 1-2 us
// away, several times a chunk's MFMAs), a chunk is staged into one of two LDS
// buffers and used after one barrier.
// FOLD: the input holds points (pairs p, refl - p), else modes.  Rows beyond
// M and pairs beyond nk are read at clamped places: a row's result is not
// stored, a pair meets a zero row of the matrix.
template <int BM, int BN, int MT, int NT, int WK, int KC, int D, bool FOLD, int EPI, class TI,
          class TO>
__global__ __launch_bounds__(256, 2) void k_modal(ModalPass a) {
  constexpr int WN = BN / (16 * NT), WM = BM / (16 * MT);
  static_assert(WM * WN * WK == 4, "four waves");
  constexpr int IN_PT = BM * KC / 256, MAT_PT = BN * KC / 256;
  static_assert(IN_PT >= 1 && MAT_PT >= 1, "every thread stages");
  constexpr int BS = BM + 1;  // padded: the staging writes walk the contraction index
  __shared__ d2 sb[2][KC * BS];
  __shared__ d2 sa[2][KC * BN];
  const int njt = (a.nj + BN - 1) / BN, nmt = (a.M + BM - 1) / BM;
  // XCD b mod 8 takes a contiguous run of tiles, output tiles fastest: its
  // workgroups share a few input rows and stream the matrix together
  const int per = (int)(gridDim.x >> 3);
  const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= njt * nmt) return;
  if (a.skip && *a.skip != 0.0) return;
  const int m0 = (tile / njt) * BM, j0 = (tile % njt) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wk = wave % WK, wn = (wave / WK) % WN, wm = wave / (WK * WN);
  const int kin = tid % KC, min0 = tid / KC;    // staging: input element
  const int jmat = tid % BN, kmat0 = tid / BN;  // staging: matrix element
  const TI* row[IN_PT];
#pragma unroll
  for (int i = 0; i < IN_PT; i++)
    row[i] = reinterpret_cast<const TI*>(a.in) +
             (int64_t)min(m0 + min0 + i * (256 / KC), a.M - 1) * a.ldi;
  const d2* mat = a.mat + (int64_t)kmat0 * a.LJ + j0 + jmat;

  TI ru[D][IN_PT], rw[D][IN_PT];
  d2 ra[D][MAT_PT];
  auto fetch = [&](int d, int k0) {
    int p0, p1;
    if (FOLD) {
      p0 = min(k0 + kin, a.nk - 1);
      p1 = min(a.refl - p0, a.npts - 1);
    } else {
      p0 = min(k0 + kin, a.ne - 1);
      p1 = a.ne + min(k0 + kin, a.no - 1);
    }
#pragma unroll
    for (int i = 0; i < IN_PT; i++) {
      ru[d][i] = row[i][p0];
      rw[d][i] = row[i][p1];
    }
#pragma unroll
    for (int i = 0; i < MAT_PT; i++)
      ra[d][i] = mat[(int64_t)(k0 + i * (256 / BN)) * a.LJ];
  };
  auto stage = [&](int d, int buf, int k0) {
    // a point on the mirror line is its own pair: counted once, no odd part
    const int p0 = k0 + kin;
    const bool self = FOLD && (a.refl - p0 == p0 || a.refl - p0 >= a.npts);
#pragma unroll
    for (int i = 0; i < IN_PT; i++) {
      const double u = (double)ru[d][i], w = (double)rw[d][i];
      d2 v;
      v.x = FOLD ? (self ? u : u + w) : u;
      v.y = FOLD ? (self ? 0.0 : u - w) : w;
      sb[buf][kin * BS + min0 + i * (256 / KC)] = v;
    }
#pragma unroll
    for (int i = 0; i < MAT_PT; i++) sa[buf][(kmat0 + i * (256 / BN)) * BN + jmat] = ra[d][i];
  };

  d4 ce[NT][MT], co[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int t = 0; t < MT; t++) ce[n][t] = co[n][t] = d4{0.0, 0.0, 0.0, 0.0};
  // (loads are never under a condition: a clamped chunk is loaded past the
  // end, so that no register copy waits for a load in flight)
  const int last = a.K - KC;
#pragma unroll
  for (int d = 0; d < D; d++) {
    fetch(d, min(d * KC, last));
    __builtin_amdgcn_sched_barrier(0);  // in order: a wait counts the later sets out
  }
  int buf = 0;
  for (int kb = 0; kb < a.K; kb += D * KC) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int k0 = kb + d * KC;
      if (k0 >= a.K) break;  // uniform
      {
        // (buf was last read two chunks ago, before the previous barrier)
        stage(d, buf, k0);
        // the next loads take the registers just staged: not moved above
        __builtin_amdgcn_sched_barrier(0);
        fetch(d, min(k0 + D * KC, last));
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < KC / (4 * WK); q++) {
          const int kr = (q * WK + wk) * 4 + (lane >> 4);
          d2 av[NT];
#pragma unroll
          for (int n = 0; n < NT; n++)
            av[n] = sa[buf][kr * BN + (wn * NT + n) * 16 + (lane & 15)];
#pragma unroll
          for (int t = 0; t < MT; t++) {
            const d2 bv = sb[buf][kr * BS + (wm * MT + t) * 16 + (lane & 15)];
#pragma unroll
            for (int n = 0; n < NT; n++) {
              ce[n][t] =
                  __builtin_amdgcn_mfma_f64_16x16x4f64(av[n].x, bv.x, ce[n][t], 0, 0, 0);
              co[n][t] =
                  __builtin_amdgcn_mfma_f64_16x16x4f64(av[n].y, bv.y, co[n][t], 0, 0, 0);
            }
          }
        }
        buf ^= 1;
      }
    }
  }
  if (WK > 1) {
    static_assert(WK == 1 || (MT == 1 && NT == 1), "split tiles hold one block a wave");
    double* red = reinterpret_cast<double*>(&sb[0][0]);
    static_assert((WK - 1) * WM * WN * 8 * 64 * 8 <= (int)sizeof(sb), "reduction space");
    const int slot = wm * WN + wn;
    __syncthreads();  // the last chunk's reads of sb
    if (wk > 0) {
      double* r = red + ((wk - 1) * WM * WN + slot) * 8 * 64 + lane;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        r[q * 64] = ce[0][0][q];
        r[(4 + q) * 64] = co[0][0][q];
      }
    }
    __syncthreads();
    if (wk > 0) return;
    for (int w = 0; w < WK - 1; w++) {
      const double* r = red + (w * WM * WN + slot) * 8 * 64 + lane;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        ce[0][0][q] += r[q * 64];
        co[0][0][q] += r[(4 + q) * 64];
      }
    }
  }
  TO* out = reinterpret_cast<TO*>(a.out);
#pragma unroll
  for (int t = 0; t < MT; t++) {
    const int m = m0 + (wm * MT + t) * 16 + (lane & 15);
    if (m >= a.M) continue;
    const double lm = EPI == EPI_SCALED ? a.lam_m[m] : 0.0;
#pragma unroll
    for (int nq = 0; nq < 4 * NT; nq++) {
      const int n = nq >> 2, q = nq & 3;
      const int j = j0 + (wn * NT + n) * 16 + (lane >> 4) + 4 * q;
      if (j >= a.nj) continue;
      const double e = ce[n][t][q], o = co[n][t][q];
      if (EPI == EPI_MODES || EPI == EPI_SCALED) {
        if (j < a.ne)
          out[(int64_t)j * a.ldo + m] =
              EPI == EPI_SCALED ? e * inv_lam(lm + a.lam_j[j]) : e;
        if (j < a.no)
          out[(int64_t)(a.ne + j) * a.ldo + m] =
              EPI == EPI_SCALED ? o * inv_lam(lm + a.lam_j[a.ne + j]) : o;
      } else {
        const int p1 = a.refl - j;
        const bool pair = p1 != j && p1 < a.npts;
        if (EPI == EPI_POINTS) {
          out[(int64_t)j * a.ldo + m] = e + o;
          if (pair) out[(int64_t)p1 * a.ldo + m] = e - o;
        } else {
          put_wrapped<TO>(out, a, j, m, TO(e + o));
          if (pair) put_wrapped<TO>(out, a, p1, m, TO(e - o));
        }
      }
    }
  }
}

// The pair matrices of one direction of n cells, from a table t of
// cos(pi j / (2 n)), j = 0 .. 4 n - 1 (exact index reduction).  form 0: rows
// are mirror pairs of points, columns modes (forward); 1: the transpose
// (back); 2: forward from a cell field, the eigenvectors averaged from the
// two vertices of each cell.
__global__ __launch_bounds__(256) void k_modal_mat(int bc, int n, int form, int ne, int no,
                                                   int nh, int K, int LJ,
                                                   const double* __restrict__ t,
                                                   d2* __restrict__ mat) {
  const int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (w >= (int64_t)K * LJ) return;
  const int row = (int)(w / LJ), col = (int)(w - (int64_t)row * LJ);
  const int h = form == 1 ? col : row, j = form == 1 ? row : col;
  const int n4 = 4 * n;
  // cos or sin of (pi / (2 n)) a, a reduced modulo 4 n
  auto cs = [&](int64_t a) { return t[(int)(a % n4)]; };
  auto sn = [&](int64_t a) { return t[(int)((a + 3 * (int64_t)n) % n4)]; };  // cos(x - pi/2)
  auto value = [&](bool odd, int pos) -> double {  // mode j of a parity at point pos
    const double r2 = sqrt(2.0 / (double)n);
    if (bc == BC_WALL)  // sin(pi k pos / n): symmetric for odd k
      return r2 * sn(2 * (int64_t)(odd ? 2 * j + 2 : 2 * j + 1) * pos);
    if (bc == BC_RING) {
      if (odd) return r2 * sn(4 * (int64_t)(j + 1) * pos);
      const double c = (j == 0 || 2 * j == n) ? sqrt(1.0 / (double)n) : r2;
      return c * cs(4 * (int64_t)j * pos);
    }
    const int k = odd ? 2 * j + 1 : 2 * j;  // cos(pi k (2 pos + 1) / (2 n))
    return (k == 0 ? sqrt(1.0 / (double)n) : r2) * cs((int64_t)k * (2 * pos + 1));
  };
  d2 v = {0.0, 0.0};
  if (h < nh) {
    if (form == 2) {
      if (j < ne) v.x = 0.5 * (value(false, h) + value(false, h + 1));
      if (j < no) v.y = 0.5 * (value(true, h) + value(true, h + 1));
    } else {
      const int pos = bc == BC_WALL ? h + 1 : h;
      if (j < ne) v.x = value(false, pos);
      if (j < no) v.y = value(true, pos);
    }
  }
  mat[w] = v;
}

// ---------------------------------------------------------------------------
// measured residual (host-checked solves)
// ---------------------------------------------------------------------------
struct ModalRes {
  int ny, nx, NXP;  // the problem's points (unknowns) and the padded pitch
  int64_t k0;       // padded index of the first unknown
  int bcx, bcy;
  double cx, cy, md;
  int gmode;
};

template <class T>
__device__ __forceinline__ double modal_b(const ModalRes& g, const T* b, int64_t k) {
  if (!g.gmode) return (double)b[k];
  return 0.25 * ((((double)b[k - g.NXP - 1] + (double)b[k - 1]) + (double)b[k - g.NXP]) +
                 (double)b[k]);
}

// one direction's second difference at position p of n points, neighbours by
// the direction's kind (a wall's beyond is 0, an even wall drops its term)
template <class T>
__device__ __forceinline__ double modal_d2(int bc, int p, int n, const T* x, int64_t k,
                                           int64_t st) {
  const double c = (double)x[k];
  const bool lo = p == 0, hi = p == n - 1;
  double l, r;
  if (bc == BC_RING) {
    l = (double)x[lo ? k + (int64_t)(n - 1) * st : k - st];
    r = (double)x[hi ? k - (int64_t)(n - 1) * st : k + st];
  } else {
    const double edge = bc == BC_EVEN ? c : 0.0;
    l = lo ? edge : (double)x[k - st];
    r = hi ? edge : (double)x[k + st];
  }
  return l + r - 2.0 * c;
}

__device__ __forceinline__ double modal_sum(double v, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const double r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return r;
}

constexpr int MODAL_NB = 512;  // blocks of the residual sums

// block sums of b; then (mean given) of r^2, r, (b - mean)^2 with
// r = (b - mean) - A x
template <class T>
__global__ __launch_bounds__(256) void k_modal_bsum(ModalRes g, const T* __restrict__ b,
                                                    double* __restrict__ part) {
  __shared__ double sh[4];
  double v = 0.0;
  const int64_t n = (int64_t)g.ny * g.nx;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += MODAL_NB * 256) {
    const int64_t r = i / g.nx;
    v += modal_b(g, b, g.k0 + r * g.NXP + (i - r * g.nx));
  }
  v = modal_sum(v, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

template <class TB, class TX>
__global__ __launch_bounds__(256) void k_modal_norms(ModalRes g, const TB* __restrict__ b,
                                                     const TX* __restrict__ x, int singular,
                                                     const double* __restrict__ bpart,
                                                     double* __restrict__ part) {
  __shared__ double sh[4];
  const int64_t n = (int64_t)g.ny * g.nx;
  double mb = 0.0;
  if (singular) {
    for (int i = threadIdx.x; i < MODAL_NB; i += 256) mb += bpart[i];
    mb = modal_sum(mb, sh) / (double)n;
  }
  double rr = 0.0, rs = 0.0, bb = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += MODAL_NB * 256) {
    const int r = (int)(i / g.nx), c = (int)(i - (int64_t)r * g.nx);
    const int64_t k = g.k0 + (int64_t)r * g.NXP + c;
    const double ax = g.cx * modal_d2(g.bcx, c, g.nx, x, k, 1) +
                      g.cy * modal_d2(g.bcy, r, g.ny, x, k, g.NXP) - g.md * (double)x[k];
    const double bv = modal_b(g, b, k) - mb, rv = bv - ax;
    rr += rv * rv;
    rs += rv;
    bb += bv * bv;
  }
  rr = modal_sum(rr, sh);
  rs = modal_sum(rs, sh);
  bb = modal_sum(bb, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = rr;
    part[MODAL_NB + blockIdx.x] = rs;
    part[2 * MODAL_NB + blockIdx.x] = bb;
  }
}

// relative residual of the (projected) system into the solve statistics
// [iterations, relres, converged, refinements | failed, max, solves]
__global__ __launch_bounds__(256) void k_modal_stats(const double* __restrict__ part, double n,
                                                     int singular, double accept,
                                                     double* __restrict__ st) {
  __shared__ double sh[4];
  double v[3];
  for (int c = 0; c < 3; c++) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < MODAL_NB; i += 256) acc += part[c * MODAL_NB + i];
    v[c] = modal_sum(acc, sh);
  }
  if (threadIdx.x != 0) return;
  double rr = v[0];
  if (singular) rr -= v[1] * v[1] / n;
  const bool finite = rr - rr == 0.0 && v[2] - v[2] == 0.0;
  const double rel = !finite ? NAN : (v[2] > 0.0 && rr > 0.0 ? sqrt(rr / v[2]) : 0.0);
  const double conv = rel <= accept ? 1.0 : 0.0;
  st[0] = 1.0;
  st[1] = rel;
  st[2] = conv;
  st[3] = 0.0;
  st[4] += conv > 0.0 ? 0.0 : 1.0;
  st[6] += 1.0;
  if (st[7] == st[7] && !(rel <= st[7])) st[7] = rel;  // a NaN stays
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct ModalDir : ModalSizes {  // one direction
  d2 *fwd = nullptr, *back = nullptr, *cell = nullptr;
  double* lam = nullptr;  // even modes, then odd modes
};

struct ModalSolver {
  ModalDir x, y;
  ModalRes res{};
  int64_t NXP = 0, k0 = 0, c0 = 0;  // padded index of the first unknown, cell
  int singular = 0;
  double *t1 = nullptr, *t2 = nullptr;
  double* part = nullptr;
  double* x64 = nullptr;  // FP64 result of a measured FP32 solve
  std::vector<void*> allocs;
};

bool modal_applicable(int64_t ny, int64_t nx, int xper, int yper, int64_t nwet, bool cells) {
  const int64_t wx = cells || xper ? nx : nx - 1, wy = cells || yper ? ny : ny - 1;
  return nx >= 8 && ny >= 8 && nx <= 4096 && ny <= 4096 && nwet == wx * wy;
}

template <class P>
static P* malloc_dev(ModalSolver* m, size_t bytes) {
  void* p = nullptr;
  F2D_HIP(hipMalloc(&p, bytes < 256 ? 256 : bytes));
  m->allocs.push_back(p);
  return reinterpret_cast<P*>(p);
}

static void dir_create(ModalSolver* m, ModalDir& d, int bc, int n, double c, double md) {
  static_cast<ModalSizes&>(d) = modal_sizes(bc, n);
  const long double pi = 3.14159265358979323846264338327950288L;
  std::vector<double> t(4 * (size_t)n), lam(d.pts);
  for (int j = 0; j < 4 * n; j++) t[j] = (double)cosl(pi * j / (2.0L * n));
  t[n] = t[3 * (size_t)n] = 0.0;
  for (int j = 0; j < d.pts; j++) {
    const bool odd = j >= d.ne;
    const int q = odd ? j - d.ne : j;
    // the angle of the mode's second difference
    long double a;
    if (bc == BC_WALL) a = pi * (odd ? 2 * q + 2 : 2 * q + 1) / n;
    else if (bc == BC_RING) a = 2.0L * pi * (odd ? q + 1 : q) / n;
    else a = pi * (odd ? 2 * q + 1 : 2 * q) / n;
    // 2 (cos a - 1) without cancellation
    const long double h = sinl(0.5L * a);
    lam[j] = (double)(-4.0L * c * h * h) - md;
  }
  double* td = nullptr;
  F2D_HIP(hipMalloc(&td, sizeof(double) * t.size()));
  m->allocs.push_back(td);
  F2D_HIP(hipMemcpy(td, t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice));
  d.lam = malloc_dev<double>(m, sizeof(double) * d.pts);
  F2D_HIP(hipMemcpy(d.lam, lam.data(), sizeof(double) * d.pts, hipMemcpyHostToDevice));
  auto mat = [&](int form, int nh, int K, int LJ) {
    d2* p = malloc_dev<d2>(m, sizeof(d2) * (size_t)K * LJ);
    k_modal_mat<<<grid1d((int64_t)K * LJ, 256), 256>>>(bc, n, form, d.ne, d.no, nh, K, LJ, td,
                                                       p);
    F2D_HIP(hipGetLastError());
    return p;
  };
  d.fwd = mat(0, d.nh, d.KF, d.LF);
  d.back = mat(1, d.nh, d.KB, d.LB);
  if (bc != BC_EVEN) d.cell = mat(2, d.cnh, d.KC, d.LF);
}

ModalSolver* modal_create(int64_t ny, int64_t nx, double dx, double dy, double maindiag,
                          int xper, int yper, bool cells, bool single) {
  ModalSolver* m = new ModalSolver();
  try {
    const int closed = cells ? BC_EVEN : BC_WALL;
    const double cx = dy / dx, cy = dx / dy;
    dir_create(m, m->x, xper ? BC_RING : closed, (int)nx, cx, 0.0);
    dir_create(m, m->y, yper ? BC_RING : closed, (int)ny, cy, maindiag);
    m->NXP = nx + 6;
    m->c0 = 3 * m->NXP + 3;
    m->k0 = (m->y.bc == BC_WALL ? 4 : 3) * m->NXP + (m->x.bc == BC_WALL ? 4 : 3);
    m->singular = maindiag == 0.0 && m->x.bc != BC_WALL && m->y.bc != BC_WALL;
    m->res = ModalRes{m->y.pts, m->x.pts, (int)m->NXP, m->k0, m->x.bc, m->y.bc,
                      cx, cy, maindiag, 0};
    const size_t n = (size_t)nx * ny;
    m->t1 = malloc_dev<double>(m, sizeof(double) * n);
    m->t2 = malloc_dev<double>(m, sizeof(double) * n);
    m->part = malloc_dev<double>(m, sizeof(double) * 4 * MODAL_NB);
    if (single) m->x64 = malloc_dev<double>(m, sizeof(double) * (size_t)(nx + 6) * (ny + 6));
    F2D_HIP(hipDeviceSynchronize());
  } catch (...) {
    modal_destroy(m);
    throw;
  }
  return m;
}

void modal_destroy(ModalSolver* m) {
  if (!m) return;
  (void)hipDeviceSynchronize();
  for (void* p : m->allocs) (void)hipFree(p);
  delete m;
}

template <int T, int MT, int NT, int WK, bool FOLD, int EPI, class TI, class TO>
static void launch_tile(const ModalPass& a, hipStream_t s) {
  constexpr int B = MODAL_TILES[T].b, KC = MODAL_TILES[T].kc;
  // the loads of whole tiles and chunks stay inside the matrix
  F2D_REQUIRE(modal_up(a.nj, B) <= a.LJ && a.K % KC == 0, "tile does not fit the matrix");
  const int64_t t = (modal_tiles(a.M, a.nj, B) + 7) / 8 * 8;
  k_modal<B, B, MT, NT, WK, KC, 2, FOLD, EPI, TI, TO><<<(unsigned)t, 256, 0, s>>>(a);
}

template <bool FOLD, int EPI, class TI, class TO>
static void launch_pass(const ModalPass& a, hipStream_t s) {
  switch (modal_tile(a.M, a.nj)) {
    case 0: launch_tile<0, 2, 2, 1, FOLD, EPI, TI, TO>(a, s); break;
    case 1: launch_tile<1, 1, 1, 1, FOLD, EPI, TI, TO>(a, s); break;
    default: launch_tile<2, 1, 1, 4, FOLD, EPI, TI, TO>(a, s);
  }
}

template <class TB, class TX>
void modal_solve(ModalSolver* m, const TB* b, int gmode, TX* x, bool measure, double accept,
                 double* stats, hipStream_t s, const double* skip, const int8_t* only) {
  const ModalDir &dx = m->x, &dy = m->y;
  F2D_REQUIRE(!gmode || (dx.cell && dy.cell), "the cell operator takes b on the cells");
  // 1: rows of b -> modes of x (t1: one row per mode)
  ModalPass a{};
  a.skip = skip;
  a.mat = gmode ? dx.cell : dx.fwd;
  a.in = b + (gmode ? m->c0 : m->k0);
  a.out = m->t1;
  a.ldi = m->NXP;
  a.M = gmode ? dy.cpts : dy.pts;
  a.ldo = a.M;
  a.K = gmode ? dx.KC : dx.KF;
  a.LJ = dx.LF;
  a.nk = gmode ? dx.cnh : dx.nh;
  a.npts = gmode ? dx.cpts : dx.pts;
  a.refl = gmode ? dx.crefl : dx.refl;
  a.ne = dx.ne;
  a.no = dx.no;
  a.nj = dx.ne;
  launch_pass<true, EPI_MODES, TB, double>(a, s);
  // 2: -> modes of y, divided by the eigenvalues (t2)
  ModalPass p{};
  p.skip = skip;
  p.mat = gmode ? dy.cell : dy.fwd;
  p.in = m->t1;
  p.out = m->t2;
  p.ldi = a.ldo;
  p.M = dx.pts;
  p.ldo = dx.pts;
  p.K = gmode ? dy.KC : dy.KF;
  p.LJ = dy.LF;
  p.nk = gmode ? dy.cnh : dy.nh;
  p.npts = gmode ? dy.cpts : dy.pts;
  p.refl = gmode ? dy.crefl : dy.refl;
  p.ne = dy.ne;
  p.no = dy.no;
  p.nj = dy.ne;
  p.lam_m = dx.lam;
  p.lam_j = dy.lam;
  launch_pass<true, EPI_SCALED, double, double>(p, s);
  // 3: modes of x -> points of x (t1)
  ModalPass q{};
  q.skip = skip;
  q.mat = dx.back;
  q.in = m->t2;
  q.out = m->t1;
  q.ldi = dx.pts;
  q.M = dy.pts;
  q.ldo = dy.pts;
  q.K = dx.KB;
  q.LJ = dx.LB;
  q.nk = dx.ne;
  q.npts = dx.pts;
  q.refl = dx.refl;
  q.ne = dx.ne;
  q.no = dx.no;
  q.nj = dx.nh;
  launch_pass<false, EPI_POINTS, double, double>(q, s);
  // 4: modes of y -> x
  ModalPass r{};
  r.skip = skip;
  r.mat = dy.back;
  r.in = m->t1;
  r.out = x;
  r.ldi = dy.pts;
  r.M = dx.pts;
  r.ldo = m->NXP;
  r.K = dy.KB;
  r.LJ = dy.LB;
  r.nk = dy.ne;
  r.npts = dy.pts;
  r.refl = dy.refl;
  r.ne = dy.ne;
  r.no = dy.no;
  r.nj = dy.nh;
  r.x0 = m->k0;
  r.wx = dx.bc == BC_RING ? dx.n : 0;
  r.wy = dy.bc == BC_RING ? dy.n : 0;
  r.only = only;
  launch_pass<false, EPI_PADDED, double, TX>(r, s);
  if (measure && stats) {
    ModalRes g = m->res;
    g.gmode = gmode;
    double* sum = m->part + 3 * MODAL_NB;
    if (m->singular) k_modal_bsum<TB><<<MODAL_NB, 256, 0, s>>>(g, b, sum);
    if constexpr (sizeof(TX) == 4) {
      // the residual of x rounded to FP32 (1e-3 at 1024^2, the operator
      // amplifies the rounding) says nothing: that of the FP64 result
      F2D_REQUIRE(m->x64, "eigenvector solver built without its FP64 result");
      r.out = m->x64;
      r.only = nullptr;
      launch_pass<false, EPI_PADDED, double, double>(r, s);
      k_modal_norms<TB, double><<<MODAL_NB, 256, 0, s>>>(g, b, m->x64, m->singular, sum,
                                                         m->part);
    } else {
      k_modal_norms<TB, double><<<MODAL_NB, 256, 0, s>>>(g, b, x, m->singular, sum, m->part);
    }
    k_modal_stats<<<1, 256, 0, s>>>(m->part, (double)g.ny * g.nx, m->singular, accept,
                                   stats);
  }
}

template void modal_solve(ModalSolver*, const double*, int, double*, bool, double, double*,
                          hipStream_t, const double*, const int8_t*);
template void modal_solve(ModalSolver*, const float*, int, float*, bool, double, double*,
                          hipStream_t, const double*, const int8_t*);
template void modal_solve(ModalSolver*, const double*, int, float*, bool, double, double*,
                          hipStream_t, const double*, const int8_t*);

}  // namespace f2d
