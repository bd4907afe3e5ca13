// f2d_fft.hip -- direct spectral solve of the fully wet, doubly periodic
// Poisson/Helmholtz operator (see f2d_fft.hpp for the mathematics).
//
// Three passes over the data, each one kernel:
//   rows:    two real rows packed as one complex row, length-nx FFT in LDS,
//            unpacked to the two half spectra (kx = 0 .. nx/2), written
//            column-major (each kx column contiguous in y)
//   columns: length-ny FFT, division by the eigenvalue (and 1/(nx ny)),
//            inverse FFT, all in LDS; written back in place
//   rows:    the two half spectra of a row pair repacked into one complex
//            row, inverse FFT, real/imaginary parts stored as the two rows
//            together with their periodic halo images
// Lengths up to 1024 run as mixed radix-4/2 Stockham passes through LDS
// (fft_lds: self-sorting, ping-pong between two buffers); 2048 and 4096, and
// FP64 columns from 256 (plan_blocks), as radix-8 passes in registers with LDS
// exchanges between them (RegFft).  Twiddles come from tables in pass order;
// inverse transforms conjugate on the way in and out.
#include <cmath>
#include <type_traits>
#include <vector>

#include "f2d_fft.hpp"

namespace f2d {

template <class T> struct CplxOf;
template <> struct CplxOf<double> { using type = double2; };
template <> struct CplxOf<float> { using type = float2; };
template <class T> using cplx = typename CplxOf<T>::type;

template <class T>
__device__ __forceinline__ cplx<T> mk(T a, T b) {
  cplx<T> r;
  r.x = a;
  r.y = b;
  return r;
}
template <class T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) {
  return mk<T>(a.x + b.x, a.y + b.y);
}
template <class T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) {
  return mk<T>(a.x - b.x, a.y - b.y);
}
template <class T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
  return mk<T>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Row workgroups are mapped XCD-aware: the hardware places workgroup b on
// XCD b % 8, so workgroup b takes row block (b % 8) * (G / 8) + b / 8 and
// each XCD handles one contiguous run of rows.  The column-major writes of
// neighbouring rows then meet in the same L2 and leave it as whole lines.
__device__ __forceinline__ int row_block(int b, int G) {
  return (G & 7) ? b : (b & 7) * (G >> 3) + (b >> 3);
}

struct FftArgs {
  int nx, ny, lgx, lgy;
  int nk;        // nx / 2 + 1 spectral columns
  int ncu;       // column-pass units: nk complex columns, or (odd x) the
                 // pairs of real columns, (nk + 1) / 2
  int NXP;       // padded row stride
  int P;         // row pairs per workgroup (row passes)
  int Q;         // spectral columns per workgroup (column pass)
  double cx, cy, d;
  int singular;
  int real0;     // drop the imaginary parts of the modes kx = 0, nx / 2
  // Closed directions (ex, ey nonzero): the problem's onx x ony interior is
  // solved as its extension on the periodic doubled grid (nx = 2 onx when
  // ex, ny = 2 ony when ey): 1 odd (vertex unknowns, Dirichlet boundary
  // lines), 2 even (cell unknowns, Neumann walls); onx / ony are the
  // problem's sizes, NXP its padded row length.
  int ex, ey;
  int onx, ony;
};
// Passes behind a device flag (nonzero: they do nothing) take arguments and
// instantiations of their own: with the flag and its test in every pass a
// 1024^2 FP64 step takes 1.5% longer.
struct FftSkipArgs : FftArgs {
  const double* skip;
};
template <bool SKIP> using FftPassArgs = std::conditional_t<SKIP, FftSkipArgs, FftArgs>;

// Forward DFTs of `nf` contiguous length-N sequences held in LDS buffer `a`
// (`b` is scratch of the same size).  Returns the buffer with the result.
template <class T>
__device__ cplx<T>* fft_lds(cplx<T>* a, cplx<T>* b, int N, int lgN, int nf,
                            const cplx<T>* tw) {
  const int tid = threadIdx.x, nth = blockDim.x;
  int Ns = 1;
  if (lgN & 1) {  // one radix-2 pass (Ns = 1: no twiddles)
    const int nb = N >> 1;
    for (int w = tid; w < nf * nb; w += nth) {
      const int f = w >> (lgN - 1), j = w & (nb - 1);
      const cplx<T>* s = a + f * N;
      cplx<T>* o = b + f * N;
      const cplx<T> a0 = s[j], a1 = s[j + nb];
      o[2 * j] = cadd<T>(a0, a1);
      o[2 * j + 1] = csub<T>(a0, a1);
    }
    __syncthreads();
    cplx<T>* t = a;
    a = b;
    b = t;
    Ns = 2;
  }
  const int Ns0 = Ns;
  while (Ns < N) {  // radix-4 passes
    const int nb = N >> 2;
    for (int w = tid; w < nf * nb; w += nth) {
      const int f = w >> (lgN - 2), j = w & (nb - 1);
      const cplx<T>* s = a + f * N;
      cplx<T>* o = b + f * N;
      const int jm = j & (Ns - 1);
      // this pass's twiddles: three contiguous runs of Ns (conflict-free)
      const cplx<T>* tp = tw + (Ns - Ns0);
      const cplx<T> a0 = s[j];
      const cplx<T> a1 = cmul<T>(s[j + nb], tp[jm]);
      const cplx<T> a2 = cmul<T>(s[j + 2 * nb], tp[Ns + jm]);
      const cplx<T> a3 = cmul<T>(s[j + 3 * nb], tp[2 * Ns + jm]);
      const cplx<T> b0 = cadd<T>(a0, a2), b1 = csub<T>(a0, a2);
      const cplx<T> b2 = cadd<T>(a1, a3), b3 = csub<T>(a1, a3);
      const int base = ((j - jm) << 2) + jm;
      o[base] = cadd<T>(b0, b2);
      o[base + Ns] = mk<T>(b1.x + b3.y, b1.y - b3.x);      // b1 - i b3
      o[base + 2 * Ns] = csub<T>(b0, b2);
      o[base + 3 * Ns] = mk<T>(b1.x - b3.y, b1.y + b3.x);  // b1 + i b3
    }
    __syncthreads();
    cplx<T>* t = a;
    a = b;
    b = t;
    Ns <<= 2;
  }
  return a;
}

// Register transforms of N = 2^LG points, LG 8 .. 12: N / 8 threads a
// sequence, 8 points a thread.  Thread j takes points j + m N/8 (m = 0 .. 7)
// and returns entries j + q N/8, so a pass's global loads and stores are
// coalesced without LDS, and a column's forward transform hands its entries
// straight to the inverse one.  Passes: one of radix 2 or 4 where LG is not
// a multiple of 3, then radix 8; between two passes the entries go through
// LDS (index i at i + i / 8: the stride-8 writes of the first passes then
// spread over the banks).  Against radix-4 passes through LDS (fft_lds) a
// 1024-point row makes 3 LDS exchanges instead of 5 and a column 6 instead
// of 11.  Every twiddle comes from the table (no products of twiddles: the
// FP32 rounding is that of one factor a pass), loaded ahead of the exchange.
// Bound by HBM from 2048 points: a FP64 4096^2 solve takes 301 us for the
// 1.2 GB that its passes read and write (4.0 TB/s), 2048^2 83 us (fft_lds
// 111 us), closed 1024^2 44 us (63), channel 1024^2 40 us (49); FP32 4096^2
// 214 us (346), closed 2048^2 127 us (199).
template <class T> struct Vec2 {
  typedef T type __attribute__((ext_vector_type(2)));  // (a struct in an
  // array held over a loop is kept in scratch memory, an ext_vector is not)
};
template <class T> using vec2 = typename Vec2<T>::type;

__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }
// (fused: one rounding less a component)
template <class T>
__device__ __forceinline__ vec2<T> vmul(vec2<T> a, vec2<T> b) {
  return vec2<T>{fma_t(a.x, b.x, -(a.y * b.y)), fma_t(a.x, b.y, a.y * b.x)};
}
// a / sqrt 2 to half an ulp: the constant with its rounding error
template <class T>
__device__ __forceinline__ T half_sqrt(T a) {
  const T hi = T(0.70710678118654752440);
  const T lo = T(sizeof(T) == 4 ? 0.70710678118654752440 - (double)0.70710678118654752440f
                                : -4.8336466567264567e-17);
  return fma_t(hi, a, lo * a);
}
// a times -i
template <class T>
__device__ __forceinline__ vec2<T> vmi(vec2<T> a) {
  return vec2<T>{a.y, -a.x};
}

__device__ __forceinline__ constexpr int pad8(int i) { return i + (i >> 3); }

template <int LG> struct RegFft {
  static constexpr int N = 1 << LG, TPF = N / 8, R0 = 1 << (LG % 3), PN = N + N / 8;
  // offset of the twiddles of the radix-8 pass of sub-length NS
  static constexpr int off(int ns) {
    int o = 0;
    for (int m = R0 == 1 ? 8 : R0; m < ns; m *= 8) o += 7 * m;
    return o;
  }
  // LDS exchanges of one transform
  static constexpr int exchanges = (LG / 3) + (R0 > 1 ? 1 : 0) - 1;
  // FP64 4096: one LDS buffer (two would leave a CU one workgroup)
  template <class T> static constexpr bool one() { return sizeof(T) == 8 && LG == 12; }
};

// the threads of a sequence meet: a wave's LDS operations are in order
template <int TPF>
__device__ __forceinline__ void seq_sync() {
  if (TPF > 64) {
    __syncthreads();
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

template <class T>
__device__ __forceinline__ void dft8(vec2<T>* v) {
  typedef vec2<T> V;
  const V a0 = v[0] + v[4], a4 = v[0] - v[4], a1 = v[1] + v[5], a5 = v[1] - v[5];
  const V a2 = v[2] + v[6], a6 = v[2] - v[6], a3 = v[3] + v[7], a7 = v[3] - v[7];
  const V b0 = a0 + a2, b2 = a0 - a2, b1 = a1 + a3, b3 = vmi<T>(a1 - a3);
  v[0] = b0 + b1;
  v[4] = b0 - b1;
  v[2] = b2 + b3;
  v[6] = b2 - b3;
  const V c1 = V{half_sqrt(a5.x + a5.y), half_sqrt(a5.y - a5.x)};  // times (1 - i) / sqrt 2
  const V c2 = vmi<T>(a6);
  const V c3 = V{half_sqrt(a7.y - a7.x), -half_sqrt(a7.x + a7.y)};  // (-1 - i) / sqrt 2
  const V d0 = a4 + c2, d2 = a4 - c2, d1 = c1 + c3, d3 = vmi<T>(c1 - c3);
  v[1] = d0 + d1;
  v[5] = d0 - d1;
  v[3] = d2 + d3;
  v[7] = d2 - d3;
}

// LDS regions of one sequence: buffer e & 1 of exchange e (one buffer: the
// same, after a wait for its readers)
template <class T, int LG>
__device__ __forceinline__ vec2<T>* xbuf(vec2<T>* b0, vec2<T>* b1, int e) {
  return RegFft<LG>::template one<T>() || !(e & 1) ? b0 : b1;
}
template <class T, int LG>
__device__ __forceinline__ void xwait() {
  if (RegFft<LG>::template one<T>()) seq_sync<RegFft<LG>::TPF>();
}
template <class T, int LG>
__device__ __forceinline__ void xread(vec2<T>* v, const vec2<T>* b, int j) {
  constexpr int st = RegFft<LG>::TPF + RegFft<LG>::TPF / 8;
  const vec2<T>* p = b + pad8(j);
#pragma unroll
  for (int m = 0; m < 8; m++) v[m] = p[m * st];
}
// entries j + q N/8 to their places (natural order, padded)
template <class T, int LG>
__device__ __forceinline__ void xwrite(const vec2<T>* v, vec2<T>* b, int j) {
  constexpr int st = RegFft<LG>::TPF + RegFft<LG>::TPF / 8;
  vec2<T>* p = b + pad8(j);
#pragma unroll
  for (int m = 0; m < 8; m++) p[m * st] = v[m];
}

template <class T, int LG, int NS>
__device__ __forceinline__ void load_tw(vec2<T>* t, const vec2<T>* __restrict__ tw, int j) {
  const vec2<T>* p = tw + RegFft<LG>::off(NS) + (j & (NS - 1));
#pragma unroll
  for (int q = 0; q < 7; q++) t[q] = p[q * NS];
}

// the radix-8 pass of sub-length NS and those after it; E: its exchange
template <class T, int LG, int NS, int E>
__device__ __forceinline__ void pass8(vec2<T>* v, vec2<T>* t, vec2<T>* b0, vec2<T>* b1, int j,
                                      const vec2<T>* __restrict__ tw) {
  typedef RegFft<LG> R;
  if (NS > 1) {
#pragma unroll
    for (int q = 1; q < 8; q++) v[q] = vmul<T>(v[q], t[q - 1]);
  }
  dft8<T>(v);
  if constexpr (NS * 8 < R::N) {
    load_tw<T, LG, NS * 8>(t, tw, j);
    const int jm = j & (NS - 1), base = ((j - jm) << 3) + jm;
    vec2<T>* b = xbuf<T, LG>(b0, b1, E);
    xwait<T, LG>();
    if (NS >= 8) {
      vec2<T>* p = b + pad8(base);
#pragma unroll
      for (int q = 0; q < 8; q++) p[q * (NS + NS / 8)] = v[q];
    } else {
#pragma unroll
      for (int q = 0; q < 8; q++) b[pad8(base + q * NS)] = v[q];
    }
    seq_sync<R::TPF>();
    xread<T, LG>(v, b, j);
    pass8<T, LG, NS * 8, E + 1>(v, t, b0, b1, j, tw);
  }
}

// forward transform, its exchanges numbered from E
template <class T, int LG, int E>
__device__ __forceinline__ void fft_regs(vec2<T>* v, vec2<T>* b0, vec2<T>* b1, int j,
                                         const vec2<T>* __restrict__ tw) {
  typedef RegFft<LG> R;
  typedef vec2<T> V;
  V t[7];
  if constexpr (R::R0 == 1) {
    pass8<T, LG, 1, E>(v, t, b0, b1, j, tw);
  } else {
    load_tw<T, LG, R::R0>(t, tw, j);
    V* b = xbuf<T, LG>(b0, b1, E);
    xwait<T, LG>();
    if constexpr (R::R0 == 2) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        V* p = b + pad8(2 * (j + q * R::TPF));
        p[0] = v[q] + v[q + 4];
        p[1] = v[q] - v[q + 4];
      }
    } else {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        V* p = b + pad8(4 * (j + q * R::TPF));
        const V s0 = v[q] + v[q + 4], s1 = v[q] - v[q + 4];
        const V s2 = v[q + 2] + v[q + 6], s3 = vmi<T>(v[q + 2] - v[q + 6]);
        p[0] = s0 + s2;
        p[1] = s1 + s3;
        p[2] = s0 - s2;
        p[3] = s1 - s3;
      }
    }
    seq_sync<R::TPF>();
    xread<T, LG>(v, b, j);
    pass8<T, LG, R::R0, E + 1>(v, t, b0, b1, j, tw);
  }
}

// right-hand side at interior vertex k (padded index): b itself, or
// centerstovertices (operators.py:126-133) of the cell field
template <class TB>
__device__ __forceinline__ double gval(const TB* __restrict__ b, int64_t k,
                                       int NXP, int gmode) {
  if (gmode == 0) return (double)b[k];
  return 0.25 * ((((double)b[k - NXP - 1] + (double)b[k - 1]) +
                  (double)b[k - NXP]) + (double)b[k]);
}

// sum of v over the threads of the workgroup (a multiple of 64, at most
// 1024), the same on every thread: butterflies within each 64-lane wave,
// then the wave sums in a fixed order (deterministic); sh holds at least
// 16 doubles
__device__ __forceinline__ double bsum256(double v, double* sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  const int nw = blockDim.x >> 6;
  double r;
  if (nw == 4) {
    r = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  } else {
    r = 0.0;
    for (int i = 0; i < nw; i++) r += sh[i];
  }
  __syncthreads();
  return r;
}

// right-hand side of a refinement: (b - mb) - A x64 at padded index k
template <class TB>
__device__ __forceinline__ double rval(const FftArgs& a, const TB* __restrict__ b,
                                       int gmode, const double* __restrict__ x,
                                       int64_t k, double mb) {
  const int64_t P = a.NXP;
  const double Ax = a.cx * (x[k - 1] + x[k + 1]) + a.cy * (x[k - P] + x[k + P]) -
                    a.d * x[k];
  return (gval(b, k, a.NXP, gmode) - mb) - Ax;
}

// right-hand side of a warm-started refinement: (g - mb) - A x32 at
// interior point (y, n), g the right-hand side there, x32 a caller's FP32
// initial guess read with periodic (wrapped) interior indices, so that its
// halo is not read
__device__ __forceinline__ double rval32(const FftArgs& a, double g,
                                         const float* __restrict__ x, int y, int n,
                                         double mb) {
  const int64_t P = a.NXP;
  const int64_t r = (int64_t)(y + 3) * P + 3;
  const int64_t rs = (int64_t)(y == 0 ? a.ny - 1 : y - 1) + 3;
  const int64_t rn = (int64_t)(y == a.ny - 1 ? 0 : y + 1) + 3;
  const int nw = n == 0 ? a.nx - 1 : n - 1, ne = n == a.nx - 1 ? 0 : n + 1;
  const double Ax = a.cx * ((double)x[r + nw] + (double)x[r + ne]) +
                    a.cy * ((double)x[rs * P + n + 3] + (double)x[rn * P + n + 3]) -
                    a.d * (double)x[r + n];
  return (g - mb) - Ax;
}

// Closed directions.  Odd (1): the Dirichlet problem on a closed direction
// of length on (vertex unknowns at points 1 .. on-1, zero at 0 and on) is
// the restriction of the periodic problem on the doubled length 2 on to
// the odd extension of its data: doubled point n is the problem's point n
// for n < on, the point 2 on - n with the opposite sign above on, and 0 at
// 0 and on.  Even (2): the Neumann problem on on cells (elliptic.py:186-190:
// a wall drops its neighbour from the row and from the diagonal) is the
// restriction of the periodic problem to the even extension about the
// walls: doubled point n is the problem's cell n for n < on and cell
// 2 on - 1 - n above, with the same sign.  The 5-point operator commutes
// with both reflections.  ext_of returns the sign (0 on a boundary line)
// and the problem's point.
__device__ __forceinline__ int ext_of(const FftArgs& a, int y, int n, int& yo, int& xo) {
  int sg = 1;
  yo = y;
  xo = n;
  if (a.ey == 1) {
    if (y == 0 || y == a.ony) return 0;
    if (y > a.ony) {
      yo = 2 * a.ony - y;
      sg = -sg;
    }
  } else if (a.ey == 2 && y >= a.ony) {
    yo = 2 * a.ony - 1 - y;
  }
  if (a.ex == 1) {
    if (n == 0 || n == a.onx) return 0;
    if (n > a.onx) {
      xo = 2 * a.onx - n;
      sg = -sg;
    }
  } else if (a.ex == 2 && n >= a.onx) {
    xo = 2 * a.onx - 1 - n;
  }
  return sg;
}

// the problem's unknowns among the doubled grid's points: the first
// quadrant, less the boundary lines of an odd direction
__device__ __forceinline__ bool ext_unknown(const FftArgs& a, int y, int n) {
  if (a.ey && (y >= a.ony || (a.ey == 1 && y == 0))) return false;
  if (a.ex && (n >= a.onx || (a.ex == 1 && n == 0))) return false;
  return true;
}

// x at the problem's point (yo, xo) of an array of the padded layout, as
// the stencil of an unknown reads it: 0 on the boundary lines of an odd
// direction, the mirror cell across the wall of an even one, wrapped in a
// periodic one (the halo is not read)
template <class TX>
__device__ __forceinline__ double xat(const FftArgs& a, const TX* __restrict__ x, int yo,
                                      int xo) {
  if (a.ex == 1) {
    if (xo <= 0 || xo >= a.onx) return 0.0;
  } else if (a.ex == 2) {
    xo = xo < 0 ? -1 - xo : (xo >= a.onx ? 2 * a.onx - 1 - xo : xo);
  } else {
    xo = xo < 0 ? xo + a.onx : (xo >= a.onx ? xo - a.onx : xo);
  }
  if (a.ey == 1) {
    if (yo <= 0 || yo >= a.ony) return 0.0;
  } else if (a.ey == 2) {
    yo = yo < 0 ? -1 - yo : (yo >= a.ony ? 2 * a.ony - 1 - yo : yo);
  } else {
    yo = yo < 0 ? yo + a.ony : (yo >= a.ony ? yo - a.ony : yo);
  }
  return (double)x[(int64_t)(yo + 3) * a.NXP + xo + 3];
}

// A x at the problem's unknown (yo, xo), x read through xat
template <class TX>
__device__ __forceinline__ double ax_ext(const FftArgs& a, const TX* __restrict__ x, int yo,
                                         int xo) {
  return a.cx * (xat(a, x, yo, xo - 1) + xat(a, x, yo, xo + 1)) +
         a.cy * (xat(a, x, yo - 1, xo) + xat(a, x, yo + 1, xo)) - a.d * xat(a, x, yo, xo);
}

// value v at the problem's unknown (y, n) and its periodic halo image
// (closed directions have no image; at most one direction is periodic)
template <class TX>
__device__ __forceinline__ void put_ext(TX* x, int y, int n, const FftArgs& a, TX v) {
  const int64_t P = a.NXP;
  const int64_t k = (int64_t)(y + 3) * P + n + 3;
  x[k] = v;
  if (!a.ex) {
    const int64_t d = n < 3 ? a.onx : (n >= a.onx - 3 ? -a.onx : 0);
    if (d) x[k + d] = v;
  }
  if (!a.ey) {
    const int64_t d = y < 3 ? (int64_t)a.ony * P : (y >= a.ony - 3 ? -(int64_t)a.ony * P : 0);
    if (d) x[k + d] = v;
  }
}

// b - A x at padded point (j, i) of the operator masked to m (x read at the
// masked unknowns only, 0 elsewhere; periodic directions wrapped), with the
// arithmetic of the capacitance solve's residual (f2d_capacitance.hip)
__device__ __forceinline__ double xm_at(const FftArgs& a, const int8_t* m, const float* x,
                                        int j, int i) {
  if (!a.ex) i = i < 3 ? i + a.onx : (i >= a.onx + 3 ? i - a.onx : i);
  if (!a.ey) j = j < 3 ? j + a.ony : (j >= a.ony + 3 ? j - a.ony : j);
  const int64_t k = (int64_t)j * a.NXP + i;
  return m[k] ? (double)x[k] : 0.0;
}
// (j, i): the padded point k = j NXP + i, as the caller knows it
__device__ __forceinline__ double masked_res(const FftArgs& a, double g, const int8_t* m,
                                             const float* x, int j, int i) {
  const int64_t k = (int64_t)j * a.NXP + i;
  if (!m[k]) return 0.0;
  const double ax = a.cx * (xm_at(a, m, x, j, i - 1) + xm_at(a, m, x, j, i + 1)) +
                    a.cy * (xm_at(a, m, x, j - 1, i) + xm_at(a, m, x, j + 1, i)) -
                    a.d * (double)x[k];
  return g - ax;
}

// Rows forward.  Without x64/x32: the rows of b (or of c2v(b)); with bpart
// non-NULL each workgroup also writes the FP64 sum of its values of b (the
// mean of b for the singular operator).  With x64 (or x32): the rows of
// the residual (b - mb) - A x, mb = (sum of the nbp partials bpin) / (nx ny);
// bpart, if given, still receives the sums of b.
template <class T, class TB, int LG, bool SKIP>
__global__ __launch_bounds__(LG ? 512 : 1024) void k_fft_rows_fwd(
    FftPassArgs<SKIP> a, const TB* __restrict__ b, int gmode, cplx<T>* __restrict__ S,
    const cplx<T>* __restrict__ tw, double* __restrict__ bpart,
    const double* __restrict__ x64, const double* __restrict__ bpin, int nbp,
    const float* __restrict__ x32, FftMask fm = FftMask(),
    const FftBatchPtrs* __restrict__ bt = nullptr) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double sh[16];
  if constexpr (SKIP)
    if (*a.skip != 0.0) return;
  if (bt) {  // a batch: this member's b, spectrum and masks
    b = reinterpret_cast<const TB*>(bt[blockIdx.y].b);
    S = reinterpret_cast<cplx<T>*>(bt[blockIdx.y].S);
    fm = bt[blockIdx.y].m;
  }
  const int nx = a.nx, P = a.P, lg = a.lgx;
  cplx<T>* b0 = reinterpret_cast<cplx<T>*>(smem);
  cplx<T>* b1 = b0 + P * nx;
  cplx<T>* tl = b1 + P * nx;  // twiddles, staged in LDS
  if (!LG)
    for (int w = threadIdx.x; w < nx; w += blockDim.x) tl[w] = tw[w];
  const int y0 = row_block(blockIdx.x, gridDim.x) * 2 * P;
  double mb = 0.0;
  if ((x64 || x32) && bpin) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < nbp; i += blockDim.x) acc += bpin[i];
    mb = bsum256(acc, sh) / ((double)a.onx * (double)a.ony);
  }
  double sum = 0.0;
  // rows y0 + 2p, y0 + 2p + 1 of a periodic grid at column n
  auto pair_at = [&](int p, int n, double& va, double& vb) {
    const int64_t ka = (int64_t)(y0 + 2 * p + 3) * a.NXP + n + 3;
    if (x32) {
      const double ga = gval(b, ka, a.NXP, gmode), gb = gval(b, ka + a.NXP, a.NXP, gmode);
      sum += ga + gb;
      va = rval32(a, ga, x32, y0 + 2 * p, n, mb);
      vb = rval32(a, gb, x32, y0 + 2 * p + 1, n, mb);
    } else if (x64) {
      va = rval(a, b, gmode, x64, ka, mb);
      vb = rval(a, b, gmode, x64, ka + a.NXP, mb);
    } else {
      va = gval(b, ka, a.NXP, gmode);
      vb = gval(b, ka + a.NXP, a.NXP, gmode);
      if (fm.in) {
        if (fm.xr) {
          va = masked_res(a, va, fm.in, fm.xr, y0 + 2 * p + 3, n + 3);
          vb = masked_res(a, vb, fm.in, fm.xr, y0 + 2 * p + 4, n + 3);
        } else {
          if (!fm.in[ka]) va = 0.0;
          if (!fm.in[ka + a.NXP]) vb = 0.0;
        }
        reinterpret_cast<TB*>(fm.out)[ka] = TB(va);
        reinterpret_cast<TB*>(fm.out)[ka + a.NXP] = TB(vb);
      }
      sum += va + vb;
    }
  };
  // extension of a closed direction: the value (or residual) at each of
  // the problem's points once, written to its doubled-grid point and,
  // in a closed x, to the mirror point with the reflection's sign (0 on
  // an odd extension's boundary lines).  Component h of the complex row
  // pair holds row y0 + 2p + h.
  const bool ext = a.ex | a.ey;
  if (ext) {
    const int nh = a.ex ? a.onx : nx;
    const int lg2 = a.ex ? lg : lg + 1;  // 2 nh = 2^lg2
    T* bs = reinterpret_cast<T*>(b0);
    for (int w = threadIdx.x; w < P * 2 * nh; w += blockDim.x) {
      const int p = w >> lg2, r = w & ((1 << lg2) - 1);
      const int h = r >= nh ? 1 : 0, n = r - h * nh;
      const int y = y0 + 2 * p + h;
      int yo, xo;
      const int sg = ext_of(a, y, n, yo, xo);
      double v = 0.0;
      if (sg) {
        const int64_t k = (int64_t)(yo + 3) * a.NXP + xo + 3;
        double g = gval(b, k, a.NXP, gmode);
        if (fm.in) {  // b (or the residual) at the masked unknowns only, kept
          g = fm.xr ? masked_res(a, g, fm.in, fm.xr, yo + 3, xo + 3) : (fm.in[k] ? g : 0.0);
          reinterpret_cast<TB*>(fm.out)[k] = TB(g);
        }
        // sums of b over the problem's points (the singular even case)
        if (ext_unknown(a, y, n)) sum += g;
        v = g;
        if (x32)
          v = (g - mb) - ax_ext<float>(a, x32, yo, xo);
        else if (x64)
          v = (g - mb) - ax_ext<double>(a, x64, yo, xo);
        if (sg < 0) v = -v;
      }
      const int q = p * nx;
      bs[2 * (q + n) + h] = T(v);
      if (a.ex == 1) {
        if (n > 0) bs[2 * (q + 2 * a.onx - n) + h] = T(-v);
        else bs[2 * (q + a.onx) + h] = T(0);  // the boundary line
      } else if (a.ex == 2) {
        bs[2 * (q + 2 * a.onx - 1 - n) + h] = T(v);
      }
    }
  } else if (!LG) {
    for (int w = threadIdx.x; w < P * nx; w += blockDim.x) {
      double va, vb;
      pair_at(w >> lg, w & (nx - 1), va, vb);
      b0[w] = mk<T>(T(va), T(vb));
    }
  }
  auto store_sum = [&]() {
    if (bpart) {
      sum = bsum256(sum, sh);
      if (threadIdx.x == 0) bpart[blockIdx.x] = sum;
    }
  };
  // half spectra of the two rows: Xa = (C + D) / 2, Xb = -i (C - D) / 2 with
  // C = F(k), D = conj(F(nx - k))
  // (closed y: the workgroups cover rows 0 .. ony-1; the column pass forms
  // the reflected rows itself)
  auto unpack = [&](int p, int k, T Cx, T Cy, T Dx, T Dy) {  // D0 = F(nx - k)
    const int64_t at = (int64_t)k * a.ny + y0 + 2 * p;
    const cplx<T> Xa = mk<T>(T(0.5) * (Cx + Dx), T(0.5) * (Cy - Dy));
    const cplx<T> Xb = mk<T>(T(0.5) * (Cy + Dy), T(-0.5) * (Cx - Dx));
    if (a.ex == 1) {  // odd x: the spectrum of an odd real row is imaginary
      reinterpret_cast<T*>(S)[at] = Xa.y;
      reinterpret_cast<T*>(S)[at + 1] = Xb.y;
    } else {
      S[at] = Xa;
      S[at + 1] = Xb;
    }
  };
  const int lgP = __ffs(P) - 1;  // P is a power of two
  if constexpr (LG > 0) {
    typedef RegFft<LG> R;
    typedef vec2<T> V;
    V* base = reinterpret_cast<V*>(smem);
    const int seq = threadIdx.x / R::TPF, j = threadIdx.x & (R::TPF - 1);
    V* x0 = base + seq * R::PN;
    V* x1 = base + (P + seq) * R::PN;
    const V* twv = reinterpret_cast<const V*>(tw);
    V v[8];
    constexpr int E = R::exchanges;
    if (ext) {
      __syncthreads();
#pragma unroll
      for (int m = 0; m < 8; m++) v[m] = base[seq * R::N + j + m * R::TPF];
      __syncthreads();  // (the staged rows lie unpadded over all regions)
    } else {
#pragma unroll
      for (int m = 0; m < 8; m++) {
        double va, vb;
        pair_at(seq, j + m * R::TPF, va, vb);
        v[m] = V{T(va), T(vb)};
      }
    }
    store_sum();
    fft_regs<T, LG, 0>(v, x0, x1, j, twv);
    V* xo = xbuf<T, LG>(x0, x1, E);
    xwait<T, LG>();
    xwrite<T, LG>(v, xo, j);
    __syncthreads();
    V* xs = xbuf<T, LG>(base, base + P * R::PN, E);
    for (int w = threadIdx.x; w < a.nk * P; w += blockDim.x) {
      const int p = w & (P - 1), k = w >> lgP;
      const V C = xs[p * R::PN + pad8(k)];
      const V D = xs[p * R::PN + pad8((R::N - k) & (R::N - 1))];
      unpack(p, k, C.x, C.y, D.x, D.y);
    }
  } else {
    store_sum();
    __syncthreads();
    const cplx<T>* r = fft_lds<T>(b0, b1, nx, lg, P, tl);
    for (int w = threadIdx.x; w < a.nk * P; w += blockDim.x) {
      const int p = w & (P - 1), k = w >> lgP;
      const cplx<T> C = r[p * nx + k], D = r[p * nx + ((nx - k) & (nx - 1))];
      unpack(p, k, C.x, C.y, D.x, D.y);
    }
  }
}

// Column pass of an odd (Dirichlet) x: the spectrum of an odd real row is
// imaginary (x[nx - n] = -x[n] gives X = -conj(X)), so its imaginary part
// is stored and two columns k1 = 2u, k2 = 2u + 1 travel as one complex
// column z = s1 + i s2.  (An even extension's spectrum carries a phase
// e^(i pi k / nx): those columns stay complex.)
// With Z = F(z) and Zc(ky) = conj(Z(ny - ky)), F(s1) = (Z + Zc) / 2 and
// F(s2) = (Z - Zc) / (2i); after the division by the eigenvalues (even in
// ky, so both stay spectra of real columns) the inverse of
// F(s1) c1 + i F(s2) c2 = Z (c1 + c2) / 2 + Zc (c1 - c2) / 2 returns the two
// solved columns as its real and imaginary parts.
template <class T, int LG>
__device__ __forceinline__ void cols_real_pairs(const FftArgs& a, T* __restrict__ Sr,
                                                const cplx<T>* __restrict__ tw,
                                                const double* __restrict__ lamx,
                                                const double* __restrict__ lamy) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int ny = a.ny, lg = a.lgy, on = a.ony;
  const int u0 = blockIdx.x * a.Q;
  const int nq = min(a.Q, a.ncu - u0);
  // value of stored column k at doubled row y (closed y: reflected rows)
  auto sval = [&](int k, int y) -> T {
    const T* c = Sr + (int64_t)k * ny;
    if (!a.ey || y < on) return c[y];
    if (a.ey == 1) return y > on ? -c[2 * on - y] : T(0);
    return c[2 * on - 1 - y];
  };
  const double inv = 1.0 / ((double)a.nx * (double)a.ny);
  // the divided spectrum of unit u0 + q at ky, conjugated: inverse by forward
  auto divided = [&](int q, int ky, T Zx, T Zy, T Mx, T My, T& zx, T& zy) {
    const int k1 = 2 * (u0 + q), k2 = k1 + 1;
    const double l1 = lamx[k1] + lamy[ky];
    const T c1 = l1 != 0.0 ? T(inv / l1) : T(0);
    T c2 = T(0);
    if (k2 < a.nk) {
      const double l2 = lamx[k2] + lamy[ky];
      c2 = l2 != 0.0 ? T(inv / l2) : T(0);
    }
    if (LG > 0 && a.ey == 1) {
      // odd columns: an imaginary odd spectrum each, column k2 in the real
      // part of Z and column k1 in the imaginary one; their even parts are
      // rounding (k_fft_cols)
      zx = T(0.5) * (Zx - Mx) * c2;
      zy = -(T(0.5) * (Zy - My) * c1);
      return;
    }
    const T hp = T(0.5) * (c1 + c2), hm = T(0.5) * (c1 - c2);
    zx = Zx * hp + Mx * hm;
    zy = -(Zy * hp - My * hm);
  };
  // (closed y: the row pass reads the problem's rows only)
  auto put = [&](int q, int y, T vx, T vy) {
    if (a.ey && y >= on) return;
    const int k1 = 2 * (u0 + q), k2 = k1 + 1;
    Sr[(int64_t)k1 * ny + y] = vx;
    if (k2 < a.nk) Sr[(int64_t)k2 * ny + y] = -vy;
  };
  if constexpr (LG > 0) {
    typedef RegFft<LG> R;
    typedef vec2<T> V;
    V* base = reinterpret_cast<V*>(smem);
    const int seq = threadIdx.x / R::TPF, j = threadIdx.x & (R::TPF - 1);
    V* x0 = base + seq * R::PN;
    V* x1 = base + (a.Q + seq) * R::PN;
    const V* twv = reinterpret_cast<const V*>(tw);
    const bool live = seq < nq;
    const int k1 = 2 * (u0 + seq), k2 = k1 + 1;
    V v[8];
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const int y = j + m * R::TPF;
      v[m] = V{live ? sval(k1, y) : T(0), live && k2 < a.nk ? sval(k2, y) : T(0)};
    }
    constexpr int E = R::exchanges;
    fft_regs<T, LG, 0>(v, x0, x1, j, twv);
    V* xo = xbuf<T, LG>(x0, x1, E);
    xwait<T, LG>();
    xwrite<T, LG>(v, xo, j);
    seq_sync<R::TPF>();
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const int ky = j + m * R::TPF;
      const V Zm = xo[pad8((R::N - ky) & (R::N - 1))];
      T zx = T(0), zy = T(0);
      if (live) divided(seq, ky, v[m].x, v[m].y, Zm.x, Zm.y, zx, zy);
      v[m] = V{zx, zy};
    }
    fft_regs<T, LG, E + 1>(v, x0, x1, j, twv);
    if (!live) return;
#pragma unroll
    for (int m = 0; m < 8; m++) put(seq, j + m * R::TPF, v[m].x, v[m].y);
  } else {
    cplx<T>* b0 = reinterpret_cast<cplx<T>*>(smem);
    cplx<T>* b1 = b0 + a.Q * ny;
    cplx<T>* tl = b1 + a.Q * ny;
    for (int w = threadIdx.x; w < nq * ny; w += blockDim.x) {
      const int q = w >> lg, y = w & (ny - 1);
      const int k1 = 2 * (u0 + q), k2 = k1 + 1;
      b0[w] = mk<T>(sval(k1, y), k2 < a.nk ? sval(k2, y) : T(0));
    }
    for (int w = threadIdx.x; w < ny; w += blockDim.x) tl[w] = tw[w];
    __syncthreads();
    cplx<T>* r = fft_lds<T>(b0, b1, ny, lg, nq, tl);
    cplx<T>* o = r == b0 ? b1 : b0;
    for (int w = threadIdx.x; w < nq * ny; w += blockDim.x) {
      const int q = w >> lg, ky = w & (ny - 1);
      const cplx<T> Z = r[w], Zm = r[q * ny + ((ny - ky) & (ny - 1))];
      T zx, zy;
      divided(q, ky, Z.x, Z.y, Zm.x, Zm.y, zx, zy);
      o[w] = mk<T>(zx, zy);
    }
    __syncthreads();
    const cplx<T>* z = fft_lds<T>(o, r, ny, lg, nq, tl);
    for (int w = threadIdx.x; w < nq * ny; w += blockDim.x) put(w >> lg, w & (ny - 1), z[w].x, z[w].y);
  }
}

template <class T, int LG, bool SKIP>
__global__ __launch_bounds__(LG ? 512 : 1024) void k_fft_cols(
    FftPassArgs<SKIP> a, cplx<T>* __restrict__ S, const cplx<T>* __restrict__ tw,
    const double* __restrict__ lamx, const double* __restrict__ lamy,
    const FftBatchPtrs* __restrict__ bt = nullptr) {
  extern __shared__ __align__(16) unsigned char smem[];
  if constexpr (SKIP)
    if (*a.skip != 0.0) return;
  if (bt) S = reinterpret_cast<cplx<T>*>(bt[blockIdx.y].S);
  if (a.ex == 1) {
    cols_real_pairs<T, LG>(a, reinterpret_cast<T*>(S), tw, lamx, lamy);
    return;
  }
  const int ny = a.ny, lg = a.lgy, on = a.ony;
  const int k0 = blockIdx.x * a.Q;
  const int nq = min(a.Q, a.nk - k0);
  cplx<T>* col = S + (int64_t)k0 * ny;
  // entry y of column k0 + q.  Closed y: rows 0 .. ony-1 are stored; row
  // 2 ony - y is row y with the opposite sign and row ony a boundary line
  // (odd), or row 2 ony - 1 - y is row y (even)
  auto cval = [&](int q, int y) -> cplx<T> {
    const cplx<T>* c = col + q * ny;
    if (!a.ey || y < on) return c[y];
    if (a.ey == 1) {
      const cplx<T> u = y > on ? c[2 * on - y] : mk<T>(T(0), T(0));
      return mk<T>(-u.x, -u.y);
    }
    return c[2 * on - 1 - y];
  };
  const double inv = 1.0 / ((double)a.nx * (double)a.ny);
  auto factor = [&](int q, int ky) -> T {
    const double lam = lamx[k0 + q] + lamy[ky];
    return lam != 0.0 ? T(inv / lam) : T(0);
  };
  if constexpr (LG > 0) {
    typedef RegFft<LG> R;
    typedef vec2<T> V;
    V* base = reinterpret_cast<V*>(smem);
    const int seq = threadIdx.x / R::TPF, j = threadIdx.x & (R::TPF - 1);
    V* x0 = base + seq * R::PN;
    V* x1 = base + (a.Q + seq) * R::PN;
    const V* twv = reinterpret_cast<const V*>(tw);
    const bool live = seq < nq;
    V v[8];
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const cplx<T> c = live ? cval(seq, j + m * R::TPF) : mk<T>(T(0), T(0));
      v[m] = V{c.x, c.y};
    }
    constexpr int E = R::exchanges;
    fft_regs<T, LG, 0>(v, x0, x1, j, twv);
    // (without the next exchange, exchange E + 1 goes where E would)
    constexpr bool swap = !R::template one<T>();
    V *c0 = swap ? x1 : x0, *c1 = swap ? x0 : x1;
    if (a.ey == 1) {
      // the spectrum of an odd extension is odd: what rounding leaves of an
      // even part would be amplified by 1/lambda and is no solution of the
      // Dirichlet problem
      V* xo = xbuf<T, LG>(x0, x1, E);
      xwait<T, LG>();
      xwrite<T, LG>(v, xo, j);
      seq_sync<R::TPF>();
#pragma unroll
      for (int m = 0; m < 8; m++)
        v[m] = T(0.5) * (v[m] - xo[pad8((R::N - (j + m * R::TPF)) & (R::N - 1))]);
      c0 = x0;
      c1 = x1;
    }
#pragma unroll
    for (int m = 0; m < 8; m++) {  // conjugate: inverse by forward
      const T f = live ? factor(seq, j + m * R::TPF) : T(0);
      v[m] = V{v[m].x * f, -(v[m].y * f)};
    }
    fft_regs<T, LG, E + 1>(v, c0, c1, j, twv);
    if (!live) return;
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const int y = j + m * R::TPF;
      if (a.ey && y >= on) continue;  // the row pass reads the problem's rows only
      col[seq * ny + y] = mk<T>(v[m].x, -v[m].y);
    }
  } else {
    cplx<T>* b0 = reinterpret_cast<cplx<T>*>(smem);
    cplx<T>* b1 = b0 + a.Q * ny;
    cplx<T>* tl = b1 + a.Q * ny;
    for (int w = threadIdx.x; w < nq * ny; w += blockDim.x) b0[w] = cval(w >> lg, w & (ny - 1));
    for (int w = threadIdx.x; w < ny; w += blockDim.x) tl[w] = tw[w];
    __syncthreads();
    cplx<T>* r = fft_lds<T>(b0, b1, ny, lg, nq, tl);
    cplx<T>* o = r == b0 ? b1 : b0;
    for (int w = threadIdx.x; w < nq * ny; w += blockDim.x) {
      const T f = factor(w >> lg, w & (ny - 1));
      const cplx<T> v = r[w];
      r[w] = mk<T>(v.x * f, -(v.y * f));  // conjugate: inverse by forward
    }
    __syncthreads();
    const cplx<T>* z = fft_lds<T>(r, o, ny, lg, nq, tl);
    for (int w = threadIdx.x; w < nq * ny; w += blockDim.x) {
      if (a.ey && (w & (ny - 1)) >= on) continue;
      const cplx<T> v = z[w];
      col[w] = mk<T>(v.x, -v.y);
    }
  }
}

// value v at interior point (y, n) and its periodic halo images
template <class TX>
__device__ __forceinline__ void put_images(TX* x, int y, int n, const FftArgs& a,
                                           TX v) {
  const int64_t P = a.NXP;
  const int64_t k = (int64_t)(y + 3) * P + n + 3;
  const int64_t dxs = n < 3 ? a.nx : (n >= a.nx - 3 ? -a.nx : 0);
  const int64_t dys = y < 3 ? (int64_t)a.ny * P : (y >= a.ny - 3 ? -(int64_t)a.ny * P : 0);
  x[k] = v;
  if (dxs) x[k + dxs] = v;
  if (dys) x[k + dys] = v;
  if (dxs && dys) x[k + dxs + dys] = v;
}

// MODE 0: x = result (TX); 1: x = result and x64 = result; 2: x64 += result,
// x = (TX) x64; 3: x += result in FP64 (x = (TX)(x + result)), also into x64
// when given (each interior point is read and written by one thread; the
// halo images written are never read)
template <class T, class TX, int MODE, int LG, bool SKIP>
__global__ __launch_bounds__(LG ? 512 : 1024) void k_fft_rows_inv(
    FftPassArgs<SKIP> a, const cplx<T>* __restrict__ S, const cplx<T>* __restrict__ tw,
    TX* __restrict__ x, double* __restrict__ x64, const double* __restrict__ rs_src = nullptr,
    double* __restrict__ rs_dst = nullptr, FftMask fm = FftMask(),
    const FftBatchPtrs* __restrict__ bt = nullptr) {
  extern __shared__ __align__(16) unsigned char smem[];
  if constexpr (SKIP)
    if (*a.skip != 0.0) return;
  if (bt) {  // a batch: this member's spectrum, solution and mask
    S = reinterpret_cast<const cplx<T>*>(bt[blockIdx.y].S);
    x = reinterpret_cast<TX*>(bt[blockIdx.y].x);
    fm = bt[blockIdx.y].m;
  }
  // the row sums of this call's b become the next call's (one per workgroup;
  // the forward row pass has the same grid)
  if (rs_dst && threadIdx.x == 0) rs_dst[blockIdx.x] = rs_src[blockIdx.x];
  const int nx = a.nx, P = a.P, lg = a.lgx, h = nx >> 1;
  cplx<T>* b0 = reinterpret_cast<cplx<T>*>(smem);
  cplx<T>* b1 = b0 + P * nx;
  cplx<T>* tl = b1 + P * nx;
  if (!LG)
    for (int w = threadIdx.x; w < nx; w += blockDim.x) tl[w] = tw[w];
  const int y0 = row_block(blockIdx.x, gridDim.x) * 2 * P;
  // conj(C) with C(k) = Xa(k) + i Xb(k) and C(nx - k) = conj(Xa(k)) +
  // i conj(Xb(k)), k = 0 .. nx/2: a thread reads both rows' entries of its k
  const int lgP = __ffs(P) - 1;  // P is a power of two
  for (int w = threadIdx.x; w < a.nk * P; w += blockDim.x) {
    const int p = w & (P - 1), k = w >> lgP;
    const int64_t at = (int64_t)k * a.ny + y0 + 2 * p;
    cplx<T> Xa, Xb;
    if (a.ex == 1) {  // odd x: the imaginary part stored
      Xa = mk<T>(T(0), reinterpret_cast<const T*>(S)[at]);
      Xb = mk<T>(T(0), reinterpret_cast<const T*>(S)[at + 1]);
    } else {
      Xa = S[at];
      Xb = S[at + 1];
    }
    // The imaginary parts of a real row's modes 0 and nx/2 are 0, through the
    // column pass too (the spectrum of a real column is symmetric): fft_lds
    // keeps that to the last bit, the register transforms (fused products) do
    // not, and what rounding leaves there, amplified by 1/lambda in the low
    // column modes, would go to the paired row (an FP32 refinement at 1024^2
    // then contracts by 1e-3 a pass, not 1e-6)
    if (a.real0 && (k == 0 || k == h)) Xa.y = Xb.y = T(0);
    cplx<T>* c = b0 + p * (LG ? nx + nx / 8 : nx);
    c[LG ? pad8(k) : k] = mk<T>(Xa.x - Xb.y, -(Xa.y + Xb.x));
    if (k > 0 && k < h)
      c[LG ? pad8(nx - k) : nx - k] = mk<T>(Xa.x + Xb.y, -(Xb.x - Xa.y));
  }
  __syncthreads();
  // rows ya, ya + 1 at column n (va, vb: conj of the result's parts)
  auto store = [&](int ya, int n, double va, double vb) {
    if (a.ex | a.ey) {
      // closed direction: only the problem's unknowns are written
      for (int h = 0; h < 2; h++) {
        const int y = ya + h;
        if (!ext_unknown(a, y, n)) continue;
        const double val = h ? vb : va;
        const int64_t k = (int64_t)(y + 3) * a.NXP + n + 3;
        if (MODE == 3 && fm.res) {
          if (fm.res[k]) x[k] = TX((double)x[k] + val);  // the masked unknowns only
        } else if (MODE == 3) {
          const double nv = (double)x[k] + val;
          if (x64) put_ext<double>(x64, y, n, a, nv);
          put_ext<TX>(x, y, n, a, TX(nv));
        } else if (MODE == 2) {
          const double nv = x64[k] + val;
          put_ext<double>(x64, y, n, a, nv);
          put_ext<TX>(x, y, n, a, TX(nv));
        } else if (MODE == 0 && fm.res) {
          if (fm.res[k]) x[k] = TX(val);  // the masked unknowns only
        } else {
          put_ext<TX>(x, y, n, a, TX(val));
          if (MODE == 1) put_ext<double>(x64, y, n, a, val);
        }
      }
      return;
    }
    if (MODE == 3 && fm.res) {
      const int64_t ka = (int64_t)(ya + 3) * a.NXP + n + 3;
      if (fm.res[ka]) x[ka] = TX((double)x[ka] + va);  // the masked unknowns only
      if (fm.res[ka + a.NXP]) x[ka + a.NXP] = TX((double)x[ka + a.NXP] + vb);
    } else if (MODE == 3) {
      const int64_t ka = (int64_t)(ya + 3) * a.NXP + n + 3;
      const double na = (double)x[ka] + va, nb = (double)x[ka + a.NXP] + vb;
      if (x64) {
        put_images<double>(x64, ya, n, a, na);
        put_images<double>(x64, ya + 1, n, a, nb);
      }
      put_images<TX>(x, ya, n, a, TX(na));
      put_images<TX>(x, ya + 1, n, a, TX(nb));
    } else if (MODE == 2) {
      const int64_t ka = (int64_t)(ya + 3) * a.NXP + n + 3;
      const double na = x64[ka] + va, nb = x64[ka + a.NXP] + vb;
      put_images<double>(x64, ya, n, a, na);
      put_images<double>(x64, ya + 1, n, a, nb);
      put_images<TX>(x, ya, n, a, TX(na));
      put_images<TX>(x, ya + 1, n, a, TX(nb));
    } else if (MODE == 0 && fm.res) {
      const int64_t ka = (int64_t)(ya + 3) * a.NXP + n + 3;
      if (fm.res[ka]) x[ka] = TX(va);  // the masked unknowns only
      if (fm.res[ka + a.NXP]) x[ka + a.NXP] = TX(vb);
    } else {
      put_images<TX>(x, ya, n, a, TX(va));
      put_images<TX>(x, ya + 1, n, a, TX(vb));
      if (MODE == 1) {
        put_images<double>(x64, ya, n, a, va);
        put_images<double>(x64, ya + 1, n, a, vb);
      }
    }
  };
  if constexpr (LG > 0) {
    typedef RegFft<LG> R;
    typedef vec2<T> V;
    V* base = reinterpret_cast<V*>(smem);
    const int seq = threadIdx.x / R::TPF, j = threadIdx.x & (R::TPF - 1);
    V* x0 = base + seq * R::PN;
    V* x1 = base + (P + seq) * R::PN;
    V v[8];
    xread<T, LG>(v, x0, j);
    fft_regs<T, LG, 1>(v, x0, x1, j, reinterpret_cast<const V*>(tw));
#pragma unroll
    for (int m = 0; m < 8; m++)
      store(y0 + 2 * seq, j + m * R::TPF, (double)v[m].x, -(double)v[m].y);
  } else {
    const cplx<T>* r = fft_lds<T>(b0, b1, nx, lg, P, tl);
    for (int w = threadIdx.x; w < P * nx; w += blockDim.x) {
      const cplx<T> v = r[w];
      store(y0 + 2 * (w >> lg), w & (nx - 1), (double)v.x, -(double)v.y);
    }
  }
}


// partial sums of b over the interior (FP64)
template <class TB>
__global__ __launch_bounds__(256) void k_fft_bsum(FftArgs a, const TB* __restrict__ b,
                                                  int gmode, double* __restrict__ part) {
  __shared__ double sh[256];
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  double v = 0.0;
  if (idx < (int64_t)a.nx * a.ny) {
    const int y = (int)(idx >> a.lgx), q = (int)(idx & (a.nx - 1));
    if (ext_unknown(a, y, q)) v = gval(b, (int64_t)(y + 3) * a.NXP + q + 3, a.NXP, gmode);
  }
  v = bsum256(v, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = v;
}

__global__ __launch_bounds__(256) void k_fft_mean(const double* __restrict__ part,
                                                  int nb, double n,
                                                  double* __restrict__ mean) {
  __shared__ double sh[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < nb; i += 256) acc += part[i];
  acc = bsum256(acc, sh);
  if (threadIdx.x == 0) *mean = acc / n;
}

// r = (b - mb) - A x64 at the interior (FP64), partial sums of r^2, r, b^2,
// b; mb (may be NULL: 0) is the mean of b for the singular operator, taken
// out before the squares are summed (no cancellation in the projected norm)
template <class TB>
__global__ __launch_bounds__(256) void k_fft_res(FftArgs a, const TB* __restrict__ b,
                                                 int gmode,
                                                 const double* __restrict__ x,
                                                 double* __restrict__ r,
                                                 double* __restrict__ part,
                                                 const double* __restrict__ mb) {
  __shared__ double sh[256];
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = (int64_t)a.nx * a.ny;
  const double m0 = mb ? *mb : 0.0;
  double rr = 0.0, rs = 0.0, bb = 0.0, bs = 0.0;
  if (idx < n) {
    const int y = (int)(idx >> a.lgx), q = (int)(idx & (a.nx - 1));
    const int64_t P = a.NXP;
    const int64_t k = (int64_t)(y + 3) * P + q + 3;
    // closed directions: the problem's unknowns only (the rest of the
    // doubled grid is the extension)
    const bool unk = ext_unknown(a, y, q);
    if (unk) {
      const double bv = gval(b, k, a.NXP, gmode) - m0;
      const double Ax = (a.ex | a.ey) ? ax_ext<double>(a, x, y, q)
                                      : a.cx * (x[k - 1] + x[k + 1]) +
                                            a.cy * (x[k - P] + x[k + P]) - a.d * x[k];
      const double rv = bv - Ax;
      if (r) r[k] = rv;
      rr = rv * rv;
      rs = rv;
      bb = bv * bv;
      bs = bv;
    }
  }
  rr = bsum256(rr, sh);
  rs = bsum256(rs, sh);
  bb = bsum256(bb, sh);
  bs = bsum256(bs, sh);
  if (threadIdx.x == 0) {
    const int nb = gridDim.x;
    part[blockIdx.x] = rr;
    part[nb + blockIdx.x] = rs;
    part[2 * nb + blockIdx.x] = bb;
    part[3 * nb + blockIdx.x] = bs;
  }
}

// one block: relative residual of the (projected) system into the solve
// statistics [iterations, relres, converged, refinements | failed, max, solves]
__global__ __launch_bounds__(256) void k_fft_stats(const double* __restrict__ part,
                                                   int nb, double n, int singular,
                                                   double accept, int nref,
                                                   int measured,
                                                   double* __restrict__ st) {
  __shared__ double sh[256];
  double v[4];
  for (int c = 0; c < 4; c++) {
    double acc = 0.0;
    if (measured)
      for (int i = threadIdx.x; i < nb; i += 256) acc += part[c * nb + i];
    v[c] = bsum256(acc, sh);
  }
  if (threadIdx.x != 0) return;
  double rel = 0.0, conv = 1.0;
  if (measured) {
    double rr = v[0], bb = v[2];
    if (singular) {
      rr -= v[1] * v[1] / n;
      bb -= v[3] * v[3] / n;
    }
    // (a norm that is not finite is reported as NaN)
    if (!(rr - rr == 0.0 && bb - bb == 0.0))
      rel = NAN;
    else
      rel = bb > 0.0 && rr > 0.0 ? sqrt(rr / bb) : 0.0;
    // a direct solve is exact up to rounding: its true residual sits at
    // eps times the condition number (about 1e-11 at 1024^2 in FP64); accept
    // is f2d_poisson_accept's
    conv = (rel <= accept) ? 1.0 : 0.0;
  }
  st[0] = (double)(nref + 1);
  st[1] = rel;
  st[2] = conv;
  st[3] = (double)nref;
  st[4] += conv > 0.0 ? 0.0 : 1.0;
  if ((double)nref > st[5]) st[5] = (double)nref;
  st[6] += 1.0;
  if (st[7] == st[7] && !(rel <= st[7])) st[7] = rel;  // a NaN stays
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct FftPlan {
  int P = 1, Q = 1;      // row pairs, columns (units) per workgroup
  int lgr = 0, lgc = 0;  // register transforms of rows, columns (0: fft_lds)
  int thr = 0, thc = 0;  // threads
  size_t lr = 0, lc = 0; // LDS
};

struct FftSolver {
  FftArgs a{};
  FftPlan p64, p32;
  double* lamx = nullptr;
  double* lamy = nullptr;
  double2* twx64 = nullptr;
  double2* twy64 = nullptr;
  float2* twx32 = nullptr;
  float2* twy32 = nullptr;
  double2* S64 = nullptr;
  float2* S32 = nullptr;
  double* x64 = nullptr;
  double* part = nullptr;
  double* part_b = nullptr;
  double* mean_b = nullptr;
  // per row-workgroup FP64 sums of b: [1] this call's, [0] the previous
  // call's (a warm-started solve reads [0] while it writes [1])
  double* rowsum[2] = {nullptr, nullptr};
  bool solved = false;  // a warm start needs an earlier solve of this handle
  double* bench_buf = nullptr;  // padded scratch for kernel timing
  int nbres = 0;
  std::vector<void*> allocs;
};

static int ilog2(int64_t v) {
  int l = 0;
  while ((int64_t(1) << l) < v) l++;
  return l;
}

static bool pow2(int64_t v) { return v > 0 && (v & (v - 1)) == 0; }

// log2 of the points of a register transform (RegFft), 0: fft_lds
static int reg_lg(int64_t n, int64_t from) {
  int l = 0;
  while ((int64_t(1) << l) < n) l++;
  return n >= from && l <= 12 ? l : 0;
}

bool fft_fits(int64_t ny, int64_t nx, int xper, int yper, bool f64, bool two_buffers) {
  // one row (column) per workgroup, two FFT buffers and the twiddles, in LDS;
  // or FP64 4096 points of a periodic direction in one buffer (RegFft)
  const size_t c = f64 ? 16 : 8;
  const int64_t tx = xper ? nx : 2 * nx, ty = yper ? ny : 2 * ny;
  auto lds = [&](int64_t n) { return 3 * (size_t)n * c <= 160 * 1024; };
  auto one = [&](int64_t n) { return !two_buffers && f64 && n == 4096; };
  const bool okx = lds(tx) || (one(tx) && xper);
  const bool oky = lds(ty) || (one(ty) && xper && yper);
  return okx && oky;
}

bool fft_applicable_cells(int64_t ny, int64_t nx, int xper, int yper, int64_t nwet) {
  const int ex = xper ? 0 : 1, ey = yper ? 0 : 1;
  return pow2(nx) && pow2(ny) && nx >= 8 && ny >= 8 && (nx << ex) <= 4096 &&
         (ny << ey) <= 4096 && nwet == nx * ny;
}

bool fft_applicable(int64_t ny, int64_t nx, int xper, int yper, int64_t nwet) {
  const int ex = xper ? 0 : 1, ey = yper ? 0 : 1;
  return pow2(nx) && pow2(ny) && nx >= 8 && ny >= 8 && (nx << ex) <= 4096 &&
         (ny << ey) <= 4096 && nwet == (nx - ex) * (ny - ey);
}

template <class P>
static P* falloc(FftSolver* f, size_t bytes) {
  void* p = nullptr;
  F2D_HIP(hipMalloc(&p, bytes < 256 ? 256 : bytes));
  F2D_HIP(hipMemset(p, 0, bytes < 256 ? 256 : bytes));
  f->allocs.push_back(p);
  return reinterpret_cast<P*>(p);
}

// Twiddles in the order the radix-4 passes read them: for the pass of
// sub-length Ns (Ns0 = 1 for even log2 N, 2 after the odd radix-2 pass),
// three runs of Ns entries at offset Ns - Ns0, run q holding
// exp(-2 pi i q jm / (4 Ns)), jm = 0 .. Ns-1.  A wavefront then reads
// consecutive (or identical) entries: no LDS bank conflicts.  N entries in all.
template <class C>
static C* twiddles(FftSolver* f, int N) {
  std::vector<C> t(N);
  int lg = 0;
  while ((1 << lg) < N) lg++;
  const int Ns0 = (lg & 1) ? 2 : 1;
  for (int Ns = Ns0; Ns < N; Ns <<= 2)
    for (int q = 1; q <= 3; q++)
      for (int jm = 0; jm < Ns; jm++) {
        const long double ang = -2.0L * 3.14159265358979323846264338327950288L *
                                (long double)(q * jm) / (long double)(4 * Ns);
        C c;
        c.x = (decltype(c.x))cosl(ang);
        c.y = (decltype(c.y))sinl(ang);
        t[(Ns - Ns0) + (q - 1) * Ns + jm] = c;
      }
  C* d = falloc<C>(f, sizeof(C) * N);
  F2D_HIP(hipMemcpy(d, t.data(), sizeof(C) * N, hipMemcpyHostToDevice));
  return d;
}

// The same for the register transforms: the radix-8 pass of sub-length Ns
// (from the first that has twiddles) reads seven runs of Ns entries, run q
// holding exp(-2 pi i q jm / (8 Ns)).
template <class C>
static C* reg_twiddles(FftSolver* f, int N, int lg) {
  std::vector<C> t;
  t.reserve(N);
  for (int Ns = lg % 3 ? 1 << (lg % 3) : 8; Ns < N; Ns *= 8)
    for (int q = 1; q < 8; q++)
      for (int jm = 0; jm < Ns; jm++) {
        const long double ang = -2.0L * 3.14159265358979323846264338327950288L *
                                (long double)(q * jm) / (long double)(8 * Ns);
        C c;
        c.x = (decltype(c.x))cosl(ang);
        c.y = (decltype(c.y))sinl(ang);
        t.push_back(c);
      }
  C* d = falloc<C>(f, sizeof(C) * t.size());
  F2D_HIP(hipMemcpy(d, t.data(), sizeof(C) * t.size(), hipMemcpyHostToDevice));
  return d;
}

static const size_t LDS_CAP = 64 * 1024;

// sequences per workgroup of a register transform of 2^lg points: one wave
// at least
static int reg_seqs(int lg) { return lg >= 9 ? 1 : 2; }

// Register transforms (RegFft) or passes through LDS (fft_lds).  Registers
// (us a pass, fft_lds first): from 2048 points in every pass (FP64 2048^2
// periodic: rows 30.5 -> 29.5, columns 44.5 -> 25.5, inverse rows 31.3 ->
// 23.1; FP32 17.8 -> 14.4, 21.4 -> 15.9, 19.4 -> 16.6), and FP64 columns from
// 256 points (256^2 6.4 -> 5.3, 1024^2 11.3 -> 8.5), from 1024 where y is
// closed (512^2 closed 9.3 -> 8.4; 256^2 closed 6.9 -> 6.9).  Shorter rows
// are bound by their strided stores and lose with 8 points a thread (1024^2
// FP64 8.0 -> 9.6, closed 512^2 6.7 -> 8.3); shorter FP32 columns gain 1 us
// alone and nothing in a step (1024^2: 49.3 us with either; two solves side
// by side, 512^2: 1% slower).
// One row pair (one spectral column) per workgroup, more for short rows
// (columns): many workgroups keep all CUs busy.  Threads a workgroup (fft_lds:
// 512 from 1024 points per workgroup, 256 below) and its LDS.
template <class T>
static void plan_blocks(const FftArgs& a, FftPlan& p) {
  const size_t c = sizeof(T) * 2;
  p.lgr = reg_lg(a.nx, 2048);
  p.lgc = reg_lg(a.ny, sizeof(T) == 4 ? 2048 : a.ey ? 1024 : 256);
  auto reg = [&](int n, int lg, int k, int& th, size_t& lds) {
    th = k * (n / 8);
    const int bufs = sizeof(T) == 8 && lg == 12 ? 1 : 2;
    lds = (size_t)bufs * k * (n + n / 8) * c;
  };
  p.P = p.lgr ? reg_seqs(p.lgr) : (a.nx >= 1024 ? 1 : 1024 / a.nx);
  // (closed y: the row passes cover the first half of the doubled rows)
  while (p.P > 1 && ((a.ny / 2) % p.P || (a.ey && (a.ny / 4) % p.P) ||
                     (2 * p.P + 1) * a.nx * c > LDS_CAP))
    p.P >>= 1;
  p.Q = p.lgc ? reg_seqs(p.lgc) : (a.ny >= 1024 ? 1 : 1024 / a.ny);
  // (odd x: a unit is a pair of columns; as many workgroups as unpaired)
  if (!p.lgc && a.ex == 1 && p.Q > 1) p.Q >>= 1;
  while (p.Q > 1 && !p.lgc && (2 * p.Q + 1) * a.ny * c > LDS_CAP) p.Q >>= 1;
  if (p.lgr) {
    reg(a.nx, p.lgr, p.P, p.thr, p.lr);
  } else {
    p.thr = p.P * a.nx >= 1024 ? 512 : 256;
    p.lr = (2 * (size_t)p.P + 1) * a.nx * c;
  }
  if (p.lgc) {
    reg(a.ny, p.lgc, p.Q, p.thc, p.lc);
  } else {
    p.thc = p.Q * a.ny >= 1024 ? 512 : 256;
    p.lc = (2 * (size_t)p.Q + 1) * a.ny * c;
  }
}

template <class K>
static void lds_limit(K* kernel, size_t lds) {
  // (the row passes hold some static LDS besides)
  if (lds > 62 * 1024)
    F2D_HIP(hipFuncSetAttribute((const void*)kernel,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
}

// the three passes on a plan, each kernel's instantiation by its length
template <class T, class TB, bool SKIP = false, class... A>
static void rows_fwd(const FftPlan& p, dim3 grid, hipStream_t s, A... args) {
  auto go = [&](auto* k) {
    lds_limit(k, p.lr);
    k<<<grid, p.thr, p.lr, s>>>(args...);
  };
  switch (p.lgr) {
    case 11: go(k_fft_rows_fwd<T, TB, 11, SKIP>); break;
    case 12: go(k_fft_rows_fwd<T, TB, 12, SKIP>); break;
    default: go(k_fft_rows_fwd<T, TB, 0, SKIP>);
  }
}
template <class T, bool SKIP = false, class... A>
static void cols(const FftPlan& p, dim3 grid, hipStream_t s, A... args) {
  auto go = [&](auto* k) {
    lds_limit(k, p.lc);
    k<<<grid, p.thc, p.lc, s>>>(args...);
  };
  if constexpr (sizeof(T) == 8) {  // (plan_blocks)
    if (p.lgc == 8) return go(k_fft_cols<T, 8, SKIP>);
    if (p.lgc == 9) return go(k_fft_cols<T, 9, SKIP>);
    if (p.lgc == 10) return go(k_fft_cols<T, 10, SKIP>);
  }
  switch (p.lgc) {
    case 11: go(k_fft_cols<T, 11, SKIP>); break;
    case 12: go(k_fft_cols<T, 12, SKIP>); break;
    default: go(k_fft_cols<T, 0, SKIP>);
  }
}
template <class T, class TX, int MODE, bool SKIP = false, class... A>
static void rows_inv(const FftPlan& p, dim3 grid, hipStream_t s, A... args) {
  auto go = [&](auto* k) {
    lds_limit(k, p.lr);
    k<<<grid, p.thr, p.lr, s>>>(args...);
  };
  switch (p.lgr) {
    case 11: go(k_fft_rows_inv<T, TX, MODE, 11, SKIP>); break;
    case 12: go(k_fft_rows_inv<T, TX, MODE, 12, SKIP>); break;
    default: go(k_fft_rows_inv<T, TX, MODE, 0, SKIP>);
  }
}

FftSolver* fft_create(int64_t ny, int64_t nx, double dx, double dy,
                      double maindiag, bool f64, bool f32, int xper, int yper,
                      bool cells) {
  FftSolver* f = new FftSolver();
  try {
    FftArgs& a = f->a;
    const int closed = cells ? 2 : 1;
    a.ex = xper ? 0 : closed;
    a.ey = yper ? 0 : closed;
    a.onx = (int)nx;
    a.ony = (int)ny;
    const int64_t onx = nx, ony = ny;
    nx = a.ex ? 2 * onx : onx;  // the transformed (doubled when closed) sizes
    ny = a.ey ? 2 * ony : ony;
    a.nx = (int)nx;
    a.ny = (int)ny;
    a.lgx = ilog2(nx);
    a.lgy = ilog2(ny);
    a.nk = (int)(nx / 2 + 1);
    a.ncu = a.ex == 1 ? (a.nk + 1) / 2 : a.nk;
    a.NXP = (int)(onx + 6);
    a.cx = dy / dx;
    a.cy = dx / dy;
    a.d = 2.0 * (a.cx + a.cy) + maindiag;
    // a Dirichlet direction makes the problem non-singular (its odd
    // extension has no mean); an even one keeps the constant null vector
    a.singular = (maindiag == 0.0 && a.ex != 1 && a.ey != 1) ? 1 : 0;
    const long double pi = 3.14159265358979323846264338327950288L;
    std::vector<double> lx(a.nk), ly(ny);
    for (int k = 0; k < a.nk; k++)
      lx[k] = (double)(2.0L * a.cx * (std::cos(2.0L * pi * k / nx) - 1.0L));
    for (int k = 0; k < ny; k++)
      ly[k] = (double)(2.0L * a.cy * (std::cos(2.0L * pi * k / ny) - 1.0L)) - maindiag;
    f->lamx = falloc<double>(f, sizeof(double) * a.nk);
    f->lamy = falloc<double>(f, sizeof(double) * ny);
    F2D_HIP(hipMemcpy(f->lamx, lx.data(), sizeof(double) * a.nk, hipMemcpyHostToDevice));
    F2D_HIP(hipMemcpy(f->lamy, ly.data(), sizeof(double) * ny, hipMemcpyHostToDevice));
    const size_t nspec = (size_t)a.nk * ny;
    const size_t npad = (size_t)(ony + 6) * (onx + 6);
    f->nbres = (int)((nx * ny + 255) / 256);
    f->part = falloc<double>(f, sizeof(double) * 4 * f->nbres);
    f->part_b = falloc<double>(f, sizeof(double) * f->nbres);
    f->mean_b = falloc<double>(f, sizeof(double));
    f->rowsum[0] = falloc<double>(f, sizeof(double) * (ny / 2 + 1));
    f->rowsum[1] = falloc<double>(f, sizeof(double) * (ny / 2 + 1));
    auto table = [&](auto zero, int n, int lg) {
      typedef decltype(zero) C;
      return lg ? reg_twiddles<C>(f, n, lg) : twiddles<C>(f, n);
    };
    if (f64) {
      plan_blocks<double>(a, f->p64);
      F2D_REQUIRE(f->p64.lr <= 160 * 1024 && f->p64.lc <= 160 * 1024,
                  "FFT rows do not fit in LDS");
      f->twx64 = table(double2{}, (int)nx, f->p64.lgr);
      f->twy64 = table(double2{}, (int)ny, f->p64.lgc);
      f->S64 = falloc<double2>(f, sizeof(double2) * nspec);
    }
    if (f32) {
      plan_blocks<float>(a, f->p32);
      f->twx32 = table(float2{}, (int)nx, f->p32.lgr);
      f->twy32 = table(float2{}, (int)ny, f->p32.lgc);
      f->S32 = falloc<float2>(f, sizeof(float2) * nspec);
      f->x64 = falloc<double>(f, sizeof(double) * npad);
    }
    F2D_HIP(hipDeviceSynchronize());
  } catch (...) {
    fft_destroy(f);
    throw;
  }
  return f;
}

void fft_destroy(FftSolver* f) {
  if (!f) return;
  (void)hipDeviceSynchronize();
  for (void* p : f->allocs) (void)hipFree(p);
  delete f;
}

// one spectral solve: rows forward, columns, rows inverse.  rs_out: write
// the per-workgroup sums of b there; xres (FP64) or xres32 (a caller's FP32
// guess): transform the residual b - A x instead of b, with the mean of b
// taken from the sums rs_in (singular operator only; any constant does,
// since the solve drops the mean, and the closer to the mean of b the less
// FP32 rounding of the residual)
template <class T, class TB, class TX, int MODE, bool SKIP = false>
static void spectral(FftSolver* f, const TB* b, int gmode, TX* x, double* x64,
                     hipStream_t s, double* rs_out = nullptr,
                     const double* xres = nullptr, const float* xres32 = nullptr,
                     const double* rs_in = nullptr, bool keep_sums = false,
                     const double* skip = nullptr) {
  FftPassArgs<SKIP> a;
  static_cast<FftArgs&>(a) = f->a;
  if constexpr (SKIP) a.skip = skip;
  const bool d = sizeof(T) == 8;
  const FftPlan& p = d ? f->p64 : f->p32;
  a.P = p.P;
  a.Q = p.Q;
  a.real0 = p.lgc > 0;
  cplx<T>* S = d ? (cplx<T>*)f->S64 : (cplx<T>*)f->S32;
  const cplx<T>* twx = d ? (const cplx<T>*)f->twx64 : (const cplx<T>*)f->twx32;
  const cplx<T>* twy = d ? (const cplx<T>*)f->twy64 : (const cplx<T>*)f->twy32;
  // closed y: rows 0 .. ony-1 only (the rest mirror them, see k_fft_rows_fwd)
  const int gr = (a.ey ? a.ony : a.ny) / (2 * a.P), gc = (a.ncu + a.Q - 1) / a.Q;
  const double* bpin = ((xres || xres32) && a.singular) ? rs_in : nullptr;
  const FftBatchPtrs* none = nullptr;
  rows_fwd<T, TB, SKIP>(p, dim3(gr), s, a, b, gmode, S, twx, rs_out, xres, bpin, gr, xres32,
                  FftMask(), none);
  cols<T, SKIP>(p, dim3(gc), s, a, S, twy, (const double*)f->lamx, (const double*)f->lamy, none);
  rows_inv<T, TX, MODE, SKIP>(p, dim3(gr), s, a, (const cplx<T>*)S, twx, x, x64,
                        (const double*)(keep_sums ? f->rowsum[1] : nullptr),
                        keep_sums ? f->rowsum[0] : (double*)nullptr, FftMask(), none);
}

template <class TB>
static void residual(FftSolver* f, const TB* b, int gmode, const double* x,
                     double* r, hipStream_t s, const double* mb = nullptr) {
  k_fft_res<TB><<<f->nbres, 256, 0, s>>>(f->a, b, gmode, x, r, f->part, mb);
}

// FP64 mean of b (singular operator), for the measured residual
template <class TB>
static const double* mean_of(FftSolver* f, const TB* b, int gmode, hipStream_t s) {
  if (!f->a.singular) return nullptr;
  k_fft_bsum<TB><<<f->nbres, 256, 0, s>>>(f->a, b, gmode, f->part_b);
  k_fft_mean<<<1, 256, 0, s>>>(f->part_b, f->nbres, (double)f->a.onx * f->a.ony,
                               f->mean_b);
  return f->mean_b;
}

void fft_solve_f64(FftSolver* f, const double* b, int gmode, double* x,
                   double accept, bool measure, double* stats, hipStream_t s,
                   const double* skip) {
  F2D_REQUIRE(f->S64, "FFT solver built without FP64 buffers");
  if (skip)
    spectral<double, double, double, 0, true>(f, b, gmode, x, nullptr, s, nullptr, nullptr,
                                              nullptr, nullptr, false, skip);
  else
    spectral<double, double, double, 0>(f, b, gmode, x, nullptr, s);
  if (measure) residual<double>(f, b, gmode, x, nullptr, s, mean_of(f, b, gmode, s));
  if (stats && measure)
    k_fft_stats<<<1, 256, 0, s>>>(f->part, f->nbres, (double)f->a.onx * f->a.ony,
                                  f->a.singular, accept, 0, measure ? 1 : 0, stats);
}

void fft_solve_f32_refine(FftSolver* f, const float* b, int gmode, float* x,
                          int nref, bool warm, double accept, bool measure,
                          double* stats, hipStream_t s) {
  F2D_REQUIRE(f->S32, "FFT solver built without FP32 buffers");
  if (nref <= 0) {
    spectral<float, float, float, 0>(f, b, gmode, x, nullptr, s);
    if (measure) {
      // the FP32 result measured in FP64 needs an FP64 copy of it
      spectral<float, float, float, 1>(f, b, gmode, x, f->x64, s);
      residual<float>(f, b, gmode, f->x64, nullptr, s, mean_of(f, b, gmode, s));
    }
  } else if (!warm || !f->solved) {
    // The residual fed to the FP32 transforms is formed in FP64 inside the
    // row pass, and must not carry the mean of b (singular operator): next
    // to it the FP32 rounding would erase the residual itself.  The first
    // row pass records the FP64 row sums (rowsum[1]) the later ones take the
    // mean from; the last pass keeps them for the next call (rowsum[0]).
    double* rs = f->rowsum[1];
    spectral<float, float, float, 1>(f, b, gmode, x, f->x64, s, rs, nullptr, nullptr,
                                     nullptr, nref == 0);
    for (int i = 0; i < nref; i++)
      spectral<float, float, float, 2>(f, b, gmode, x, f->x64, s, nullptr, f->x64, nullptr,
                                       rs, i == nref - 1);
    if (measure) residual<float>(f, b, gmode, f->x64, nullptr, s, mean_of(f, b, gmode, s));
  } else {
    // Warm start: the first refinement starts from the caller's x.  Its
    // row pass takes the mean from the previous call's row sums (rowsum[0];
    // a stale mean is harmless, see spectral) and records this b's sums
    // (rowsum[1]) for the later passes; the last pass keeps them for the
    // next call.  Fixed buffers: a captured graph replays the same.
    const bool keep64 = measure || nref > 1;
    spectral<float, float, float, 3>(f, b, gmode, x, keep64 ? f->x64 : nullptr, s,
                                     f->rowsum[1], nullptr, x, f->rowsum[0], nref == 1);
    for (int i = 1; i < nref; i++)
      spectral<float, float, float, 2>(f, b, gmode, x, f->x64, s, nullptr, f->x64, nullptr,
                                       f->rowsum[1], i == nref - 1);
    if (measure) residual<float>(f, b, gmode, f->x64, nullptr, s, mean_of(f, b, gmode, s));
  }
  f->solved = true;
  if (stats && measure)
    k_fft_stats<<<1, 256, 0, s>>>(f->part, f->nbres, (double)f->a.onx * f->a.ony,
                                  f->a.singular, accept, nref, measure ? 1 : 0, stats);
}

// One FP32 spectral solve (rows forward, columns, rows inverse; x = the
// result) for each of `nm` same-size members, `f` the plan of one of them
// (its args, twiddles and eigenvalues), `table` (device) their arrays.
void fft_solve_f32_batch(FftSolver* f, int nm, const FftBatchPtrs* table, hipStream_t s,
                         bool acc) {
  F2D_REQUIRE(f->S32, "FFT solver built without FP32 buffers");
  FftArgs a = f->a;
  const FftPlan& p = f->p32;
  a.P = p.P;
  a.Q = p.Q;
  a.real0 = p.lgc > 0;
  const int gr = (a.ey ? a.ony : a.ny) / (2 * a.P), gc = (a.ncu + a.Q - 1) / a.Q;
  const dim3 grr(gr, nm), grc(gc, nm);
  const float* nof = nullptr;
  const double* nod = nullptr;
  rows_fwd<float, float>(p, grr, s, a, nof, 0, (float2*)nullptr, (const float2*)f->twx32,
                         (double*)nullptr, nod, nod, gr, nof, FftMask(), table);
  cols<float>(p, grc, s, a, (float2*)nullptr, (const float2*)f->twy32, (const double*)f->lamx,
              (const double*)f->lamy, table);
  auto inv = [&](auto mode) {
    rows_inv<float, float, decltype(mode)::value>(
        p, grr, s, a, (const float2*)nullptr, (const float2*)f->twx32, (float*)nullptr,
        (double*)nullptr, nod, (double*)nullptr, FftMask(), table);
  };
  if (acc)
    inv(std::integral_constant<int, 3>());
  else
    inv(std::integral_constant<int, 0>());
}

// (acc: FP32 only)
template <class T>
static void solve_masked(FftSolver* f, const T* b, int gmode, T* x, const FftMask& m,
                         hipStream_t s, bool acc) {
  F2D_REQUIRE(!m.in || m.out, "a masked right-hand side needs its output array");
  FftArgs a = f->a;
  constexpr bool d = sizeof(T) == 8;
  const FftPlan& p = d ? f->p64 : f->p32;
  a.P = p.P;
  a.Q = p.Q;
  a.real0 = p.lgc > 0;
  cplx<T>* S = d ? (cplx<T>*)f->S64 : (cplx<T>*)f->S32;
  const cplx<T>* twx = d ? (const cplx<T>*)f->twx64 : (const cplx<T>*)f->twx32;
  const cplx<T>* twy = d ? (const cplx<T>*)f->twy64 : (const cplx<T>*)f->twy32;
  const int gr = (a.ey ? a.ony : a.ny) / (2 * a.P), gc = (a.ncu + a.Q - 1) / a.Q;
  FftMask mf = m, mi = m;
  mf.res = nullptr;
  mi.in = nullptr;
  mi.out = nullptr;
  mi.xr = nullptr;
  F2D_REQUIRE(!acc || (mi.res && !d), "an accumulating masked solve: FP32, with its mask");
  const FftBatchPtrs* none = nullptr;
  const double* nod = nullptr;
  rows_fwd<T, T>(p, dim3(gr), s, a, b, gmode, S, twx, (double*)nullptr, nod, nod, gr,
                 (const float*)nullptr, mf, none);
  cols<T>(p, dim3(gc), s, a, S, twy, (const double*)f->lamx, (const double*)f->lamy, none);
  if constexpr (!d) {
    if (acc) {
      rows_inv<T, T, 3>(p, dim3(gr), s, a, (const cplx<T>*)S, twx, x, (double*)nullptr, nod,
                        (double*)nullptr, mi, none);
      return;
    }
  }
  rows_inv<T, T, 0>(p, dim3(gr), s, a, (const cplx<T>*)S, twx, x, (double*)nullptr, nod,
                    (double*)nullptr, mi, none);
}

void fft_solve_f32_masked(FftSolver* f, const float* b, int gmode, float* x, const FftMask& m,
                          hipStream_t s, bool acc) {
  F2D_REQUIRE(f->S32, "FFT solver built without FP32 buffers");
  solve_masked<float>(f, b, gmode, x, m, s, acc);
}

void fft_solve_f64_masked(FftSolver* f, const double* b, int gmode, double* x, const FftMask& m,
                          hipStream_t s) {
  F2D_REQUIRE(f->S64, "FFT solver built without FP64 buffers");
  solve_masked<double>(f, b, gmode, x, m, s, false);
}

// whether two plans solve the same operator (same args and eigenvalues)
bool fft_same_plan(const FftSolver* f, const FftSolver* g) {
  const FftArgs &a = f->a, &b = g->a;
  return a.nx == b.nx && a.ny == b.ny && a.ex == b.ex && a.ey == b.ey && a.onx == b.onx &&
         a.ony == b.ony && a.cx == b.cx && a.cy == b.cy && a.d == b.d &&
         a.singular == b.singular && f->p32.P == g->p32.P && f->p32.Q == g->p32.Q &&
         f->S32 != nullptr && g->S32 != nullptr;
}

float2* fft_spectrum32(FftSolver* f) { return f->S32; }

}  // namespace f2d

namespace f2d {

// Mean launch time (us, HIP events on `s`) of one pass of the spectral solve
// on scratch data, and its algorithmic bytes: kind 0 rows forward (1: the
// refinement's residual form, FP32 only), 2 columns, 3 rows inverse (4: the
// refinement's accumulating form, FP32 only); FP32 warm start: 5 rows
// forward of the residual of an FP32 guess with the row sums of b, 6 rows
// inverse accumulating onto the FP32 guess.
double fft_bench(FftSolver* f, bool f64, int kind, int reps, hipStream_t s,
                 double* bytes) {
  F2D_REQUIRE(f64 ? f->S64 != nullptr : f->S32 != nullptr,
              "FFT solver has no buffers of this precision");
  F2D_REQUIRE(f64 ? (kind == 0 || kind == 2 || kind == 3) : (kind >= 0 && kind <= 6),
              "FFT bench kind");
  const size_t npad = (size_t)(f->a.ony + 6) * (f->a.onx + 6);
  if (!f->bench_buf) f->bench_buf = falloc<double>(f, sizeof(double) * npad);
  FftArgs a = f->a;
  const FftPlan& p = f64 ? f->p64 : f->p32;
  a.P = p.P;
  a.Q = p.Q;
  a.real0 = p.lgc > 0;
  // closed y: rows 0 .. ony-1 only (the rest mirror them, see k_fft_rows_fwd)
  const int gr = (a.ey ? a.ony : a.ny) / (2 * a.P), gc = (a.ncu + a.Q - 1) / a.Q;
  const double N = (double)a.nx * a.ny, NS = (double)a.nk * a.ny;
  const double w = f64 ? 8.0 : 4.0;  // real word
  hipEvent_t e0, e1;
  F2D_HIP(hipEventCreate(&e0));
  F2D_HIP(hipEventCreate(&e1));
  const FftBatchPtrs* none = nullptr;
  const double* nod = nullptr;
  const float* nof = nullptr;
  double* out = nullptr;
  const double *lx = f->lamx, *ly = f->lamy;
  auto launch = [&]() {
    if (f64) {
      double* buf = f->bench_buf;
      const double2 *tx = f->twx64, *ty = f->twy64, *S = f->S64;
      if (kind == 0)
        rows_fwd<double, double>(p, dim3(gr), s, a, (const double*)buf, 0, f->S64, tx, out, nod,
                                 nod, gr, nof, FftMask(), none);
      else if (kind == 2)
        cols<double>(p, dim3(gc), s, a, f->S64, ty, lx, ly, none);
      else
        rows_inv<double, double, 0>(p, dim3(gr), s, a, S, tx, buf, out, nod, out, FftMask(),
                                    none);
    } else {
      float* buf = reinterpret_cast<float*>(f->bench_buf);
      const float2 *tx = f->twx32, *ty = f->twy32, *S = f->S32;
      const double* x64 = f->x64;
      if (kind == 0 || kind == 1)
        rows_fwd<float, float>(p, dim3(gr), s, a, (const float*)buf, 0, f->S32, tx, out,
                               kind == 1 ? x64 : nod, nod, gr, nof, FftMask(), none);
      else if (kind == 2)
        cols<float>(p, dim3(gc), s, a, f->S32, ty, lx, ly, none);
      else if (kind == 3)
        rows_inv<float, float, 0>(p, dim3(gr), s, a, S, tx, buf, out, nod, out, FftMask(), none);
      else if (kind == 4)
        rows_inv<float, float, 2>(p, dim3(gr), s, a, S, tx, buf, f->x64, nod, out, FftMask(),
                                  none);
      else if (kind == 5)
        rows_fwd<float, float>(p, dim3(gr), s, a, (const float*)buf, 0, f->S32, tx,
                               f->rowsum[1], nod,
                               (const double*)(a.singular ? f->rowsum[0] : nullptr), gr,
                               (const float*)buf, FftMask(), none);
      else
        rows_inv<float, float, 3>(p, dim3(gr), s, a, S, tx, buf, out, nod, out, FftMask(), none);
    }
  };
  launch();
  F2D_HIP(hipEventRecord(e0, s));
  for (int i = 0; i < reps; i++) launch();
  F2D_HIP(hipEventRecord(e1, s));
  F2D_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  F2D_HIP(hipEventElapsedTime(&ms, e0, e1));
  F2D_HIP(hipEventDestroy(e0));
  F2D_HIP(hipEventDestroy(e1));
  const double spec = NS * 2.0 * w;  // one pass over the half spectrum
  double by = 0.0;
  switch (kind) {
    case 0: by = N * w + spec; break;
    case 1: by = N * w + N * 8.0 + spec; break;
    case 2: by = 2.0 * spec; break;
    case 3: by = spec + N * w; break;
    case 4: by = spec + N * 8.0 * 2.0 + N * w; break;
    case 5: by = 2.0 * N * w + spec; break;
    default: by = spec + 2.0 * N * w; break;
  }
  *bytes = by;
  return 1e3 * (double)ms / reps;
}

}  // namespace f2d
