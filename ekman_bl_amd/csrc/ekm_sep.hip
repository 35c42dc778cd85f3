// ekm_sep.hip -- separable solver of the consistent projection (proj_mode 2
// on grids without cross terms; no counterpart in the reference).
//
// On a rectilinear grid the finest operator, row-scaled by 1/J, is to 1e-3 (33
// rows) or 1e-5 (385 rows) the sum Lz + Ly - kx^2 of a tridiagonal operator in z
// and one in y (the interior rows' metrics, the boundary rows of MUDPACK's
// discretisation and J differ from the products of one-dimensional ones by that
// much).  The separable operator is therefore solved directly in place of a V cycle, in
// the cycle precision (FP32), inside the same FP64 residual iterations:
//
//   r^ = Q' S^1/2 M^-1 r            product over the rows j, one GEMM for all solves
//   (Lz + lambda_k - kx^2) z^ = W^-1 r^   one tridiagonal line in z per (k, kx)
//   z = S^-1/2 Q z^                 product over the eigenmodes k
//   phi += z;  r -= A z             FP64, with max|r| per solve
//
// with Ly = S^-1/2 Q Lambda Q' S^1/2 (a tridiagonal matrix with positive
// products of its off-diagonals is similar to a symmetric one) and J = W(i) M(j).
// One pass divides the residual by 1e3 (33 rows) to 1e5 for every kx alike (a
// V(1,1) cycle by 20..1000), so the solves of a projection end together after 3
// passes and none of them is a chain of one workgroup's memory round trips:
// 1024x385x769 is 684 solves of 4 to 8 V cycles otherwise.  A pass counts as one cycle.
// Measured per projection against the V cycles: 1024x385x769 12.0 ms instead
// of 68.8, 256x193x257 0.50 instead of 4.95.  Against a solve to 2e-14, a step
// that stops at 1e-12 is 3 to 90 times closer in every field than with V cycles
// (planes of 65x65 to 385x769, and the reference run's periodic singular set): the
// passes leave less of the smooth error, and end further below the tolerance in
// most solves.
//
// The decomposition is tried at set-up (sep_plan_build) and used where every
// coefficient lies within kSepDev of the separable operator's; what has not
// met the tolerance after kSepIter passes goes on with V cycles from there.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "ekm_scan.h"
#include "ekm_sep.h"

namespace {

// A pass reduces the residual by about the largest relative deviation.  The rows
// of both operators sum to zero without the kx^2 term, so a deviation acts on
// differences of neighbours only and is not amplified on smooth modes: passes in
// FP64 on sine, geometric, jumping and noisy spacings, 33 to 769 columns, every
// kind of sides and kx = 0, reduce max|r| to at most 1.1 times the deviation each
// (the first to at most 11 times it).  0.02 keeps a pass at least as fast as the
// V(1,1) cycle's worst rate (about 1/20).
constexpr double kSepDev = 0.02;
// Lines whose shift lambda_k - kx^2 is below this fraction of the z operator's
// diagonal are solved in FP64: the rounding of an FP32 factor (6e-8 of the
// diagonal) would otherwise change the solution of the smoothest modes by
// more than 1e-3.
constexpr double kSepFp64Shift = 6e-5;
constexpr double kSepPin = 1e20;

constexpr int kCols = 128;   // columns per workgroup of the products: 4 wavefronts of 32
// Residual passes: points per thread and solves per workgroup, by pick_upd.
struct UpdSplit {
  int rows, solves;
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline bool solved(const unsigned long long* rm, int s, double tol) {
  return __longlong_as_double((long long)rm[s]) <= tol;
}

// Y[s][m][i] = alpha * sum_k A[m][k] X[s][k][i], A square, for all solves at once: column c
// of the product is (s, i) = (c / nx, c % nx), so no column is padding.
// v_mfma_f32_16x16x4f32: lane l holds A[l%16][l/16], B[l/16][l%16] and
// D[4*(l/16)+v][l%16].  Bound by the FP32 matrix rate; a wavefront keeps MT x 2
// tiles (MT*16 rows x 32 columns), so every element of X is read once per
// MT*16 rows and every operand of A (staged through LDS, packed so that a
// wavefront reads 64 consecutive words) feeds two matrix instructions.
// Workgroups of the same columns are placed on one XCD, where the second
// finds X in L2.
template <int MT, typename TI>
__global__ void __launch_bounds__(256) k_sep_gemm(const float* __restrict__ A, int mtt, int nchunk, int M, int nx,
                                                  int ncols, long ld, const TI* __restrict__ X, float alpha,
                                                  float* __restrict__ Y, const unsigned long long* __restrict__ rm,
                                                  double tol, int nmb) {
  __shared__ float sA[2][4 * MT * 64];
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int mb = slot % nmb, cb = (slot / nmb) * 8 + xcd;
  const int c0 = cb * kCols;
  if (c0 >= ncols) return;
  const int cl = min(c0 + kCols, ncols) - 1;
  bool all = true;
  for (int s = c0 / nx; s <= cl / nx; ++s) all = all && solved(rm, s, tol);
  if (all) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane >> 4, lc = lane & 15;
  const TI* xp[2];
  float* yp[2];
  bool in[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = c0 + wave * 32 + t * 16 + lc;
    in[t] = c < ncols;
    const int cc = in[t] ? c : ncols - 1;
    const int s = cc / nx, i = cc - s * nx;
    xp[t] = X + (size_t)s * ld + i;
    yp[t] = Y + (size_t)s * ld + i;
  }
  f32x4 acc[MT][2];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float b[4][2], bn[4][2], an[MT];
  auto load_b = [&](int ch, float (&v)[4][2]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // rows past M meet zero columns of A
      const int k = min(ch * 16 + q * 4 + lr, M - 1);
#pragma unroll
      for (int t = 0; t < 2; ++t) v[q][t] = (float)xp[t][(size_t)k * nx];
    }
  };
  auto load_a = [&](int ch) {
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      const int e = u * 256 + tid;          // element of the chunk: [4][MT][64]
      const int q = e / (MT * 64), w = e - q * (MT * 64);
      an[u] = A[((size_t)(ch * 4 + q) * mtt + (size_t)mb * MT) * 64 + w];
    }
  };
  load_a(0);
  load_b(0, b);
#pragma unroll
  for (int u = 0; u < MT; ++u) sA[0][u * 256 + tid] = an[u];
  __syncthreads();
  for (int ch = 0; ch < nchunk; ++ch) {
    const bool more = ch + 1 < nchunk;
    if (more) {
      load_a(ch + 1);
      load_b(ch + 1, bn);
    }
    const float* a = sA[ch & 1] + lane;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float av = a[(q * MT + m) * 64];
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, b[q][t], acc[m][t], 0, 0, 0);
      }
    if (more) {
#pragma unroll
      for (int u = 0; u < MT; ++u) sA[(ch + 1) & 1][u * 256 + tid] = an[u];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int t = 0; t < 2; ++t) b[q][t] = bn[q][t];
      __syncthreads();
    }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = (mb * MT + m) * 16 + 4 * lr + v;
      if (row < M) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          if (in[t]) yp[t][(size_t)row * nx] = alpha * acc[m][t][v];
      }
    }
}

// Factor layout of one (mode, eigenmode) line: f1, a, c [3][nx]; periodic ends
// add the wrap vectors W1, W2 [2][nx] and the 2x2 matrix [4].
__host__ __device__ inline long line_stride(int nx, bool per) { return per ? 5L * nx + 4 : 3L * nx; }

// Thomas factors of the lines of modes m0..m0+nm-1, one thread per (mode,
// eigenmode): f1 = 1/(piv w_i), a = -lower/piv, c = upper/piv in FP64, stored in
// T.  lz, uz, dz: the z operator; w: its column weight; f1 is zero at columns
// without an unknown (w = 0).  With periodic ends the couplings of column 0 to
// nx-2 and of nx-1 to 1 are taken out of the chain and kept as the Woodbury
// terms (W1, W2 = chain^-1 of the two couplings' unit columns).
template <typename T, bool PER>
__global__ void k_sep_factor(int nx, int nk, int m0, int nm, const double* __restrict__ z1, const double* __restrict__ lam,
                             const double* __restrict__ kx2, int pin_k, int pin_i, T* __restrict__ fac) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nm * nk) return;
  const int m = t / nk, k = t - m * nk;
  const double *lz = z1, *uz = z1 + nx, *dz = z1 + 2 * nx, *w = z1 + 3 * nx;
  const double sh = lam[k] - kx2[m0 + m];
  const bool pinned = pin_k == k && kx2[m0 + m] == 0.0;
  T* f1 = fac + (size_t)t * line_stride(nx, PER);
  T *fa = f1 + nx, *fc = fa + nx, *W1 = fc + nx, *W2 = W1 + nx, *mi = W2 + nx;
  double cprev = 0.0, v1 = 0.0, v2 = 0.0;
  for (int i = 0; i < nx; ++i) {
    const bool un = w[i] != 0.0;
    double lo = lz[i], up = uz[i], di = un ? dz[i] + sh : 1.0;
    if (pinned && i == pin_i) di *= kSepPin;
    double s1 = 0.0, s2 = 0.0;
    if (i == 0) {
      if (PER) s1 = lo;
      lo = 0.0;
    }
    if (i == nx - 1) {
      if (PER) s2 = up;
      up = 0.0;
    }
    const double ip = 1.0 / (di - lo * cprev);
    const double a = -lo * ip;
    cprev = up * ip;
    f1[i] = un ? (T)(ip / w[i]) : (T)0;
    fa[i] = (T)a;
    fc[i] = (T)cprev;
    if (PER) {
      v1 = a * v1 + s1 * ip;
      v2 = a * v2 + s2 * ip;
      W1[i] = (T)v1;
      W2[i] = (T)v2;
    }
  }
  if (PER) {
    // back substitution of the two columns
    double x1 = 0.0, x2 = 0.0, a1 = 0.0, a2 = 0.0, b1 = 0.0, b2 = 0.0;
    for (int i = nx - 1; i >= 0; --i) {
      const double c = i == nx - 1 ? 0.0 : (double)fc[i];
      x1 = (double)W1[i] - c * x1;
      x2 = (double)W2[i] - c * x2;
      W1[i] = (T)x1;
      W2[i] = (T)x2;
      if (i == nx - 2) {
        a1 = x1;
        a2 = x2;
      }
      if (i == 1) {
        b1 = x1;
        b2 = x2;
      }
    }
    const double m00 = 1.0 + a1, m01 = a2, m10 = b1, m11 = 1.0 + b2, det = m00 * m11 - m01 * m10;
    mi[0] = (T)(m11 / det);
    mi[1] = (T)(-m01 / det);
    mi[2] = (T)(-m10 / det);
    mi[3] = (T)(m00 / det);
  }
}

// The z lines, in place on t[s][k][i]: one wavefront per (mode, eigenmode) solves
// the line of both parts of the mode (solves 2m, 2m+1) with one read of the
// factors.  Point i = 64 c + lane sits in lane `lane` of stripe c; the two
// recurrences are scans of affine maps carried from stripe to stripe.  Bound by
// memory: every load of the line is issued before the first scan.
template <typename T, int CM, bool PER>
__global__ void __launch_bounds__(256) k_sep_lines(int nx, int nk, int m0, int nm, long ld, const T* __restrict__ fac,
                                                   float* __restrict__ t, const unsigned long long* __restrict__ rm,
                                                   double tol, int nsolve) {
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int m = w / nk, k = w - m * nk;
  if (m >= nm) return;
  const int s0 = 2 * (m0 + m);
  if (s0 >= nsolve) return;
  const bool two = s0 + 1 < nsolve;
  if (solved(rm, s0, tol) && (!two || solved(rm, s0 + 1, tol))) return;
  const T* f1 = fac + (size_t)w * line_stride(nx, PER);
  float* x0 = t + (size_t)s0 * ld + (size_t)k * nx;
  float* x1 = two ? x0 + ld : x0;
  T fa[CM], fc[CM], d0[CM], d1[CM];
  {
    T g[CM];
    float v0[CM], v1[CM];
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      const int i = 64 * c + lane;
      const bool in = i < nx;
      const int ii = in ? i : nx - 1;
      g[c] = f1[ii];
      fa[c] = f1[nx + ii];
      fc[c] = f1[2 * nx + ii];
      v0[c] = x0[ii];
      v1[c] = x1[ii];
      if (!in) {
        g[c] = (T)0;
        fa[c] = (T)1;
        fc[c] = (T)0;
      }
    }
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      d0[c] = g[c] * (T)v0[c];
      d1[c] = g[c] * (T)v1[c];
    }
  }
  T c0 = (T)0, c1 = (T)0;
#pragma unroll
  for (int c = 0; c < CM; ++c) {
    const Aff<T> a = wave_scan_up(Aff<T>{fa[c], d0[c]});
    const Aff<T> b = wave_scan_up(Aff<T>{fa[c], d1[c]});
    d0[c] = a.a * c0 + a.b;
    d1[c] = b.a * c1 + b.b;
    c0 = rdlane(d0[c], 63);
    c1 = rdlane(d1[c], 63);
  }
  c0 = c1 = (T)0;
#pragma unroll
  for (int c = CM - 1; c >= 0; --c) {
    const Aff<T> a = wave_scan_down(Aff<T>{-fc[c], d0[c]});
    const Aff<T> b = wave_scan_down(Aff<T>{-fc[c], d1[c]});
    d0[c] = a.a * c0 + a.b;
    d1[c] = b.a * c1 + b.b;
    c0 = rdlane(d0[c], 0);
    c1 = rdlane(d1[c], 0);
  }
  if constexpr (PER) {
    const T *W1 = f1 + 3 * nx, *W2 = W1 + nx, *mi = W2 + nx;
    const int im = nx - 2, cs = im >> 6, ls = im & 63;
    T a0 = (T)0, a1 = (T)0;
#pragma unroll
    for (int c = 0; c < CM; ++c)
      if (c == cs) {
        a0 = d0[c];
        a1 = d1[c];
      }
    const T ym0 = rdlane(a0, ls), ym1 = rdlane(a1, ls), y0 = rdlane(d0[0], 1), y1 = rdlane(d1[0], 1);
    const T g00 = mi[0] * ym0 + mi[1] * y0, g01 = mi[2] * ym0 + mi[3] * y0;
    const T g10 = mi[0] * ym1 + mi[1] * y1, g11 = mi[2] * ym1 + mi[3] * y1;
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      const int i = 64 * c + lane, ii = i < nx ? i : nx - 1;
      const T p = W1[ii], q = W2[ii];
      d0[c] -= g00 * p + g01 * q;
      d1[c] -= g10 * p + g11 * q;
    }
  }
#pragma unroll
  for (int c = 0; c < CM; ++c) {
    const int i = 64 * c + lane;
    if (i < nx) {
      x0[i] = (float)d0[c];
      if (two) x1[i] = (float)d1[c];
    }
  }
}

// max over a wavefront, then one atomic per wavefront on the bits (non-negative
// doubles order like their bits)
__device__ inline void wave_max_to(unsigned long long* to, double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  if ((threadIdx.x & 63) == 0 && v > 0.0) atomicMax(to, (unsigned long long)__double_as_longlong(v));
}

// per-solve state, and the rows of z without an unknown (the products leave
// them out): zero
// (open: the solves start without a look at their right-hand sides, so the
// first pass finds them unsolved)
__global__ void __launch_bounds__(256) k_sep_clear(unsigned long long* rm, int n, int nsmax, int open, int* cycles, int ns,
                                                   float* z, int nx, int ny, int j0, int nk) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < n) rm[t] = open && t < nsmax ? 0x7ff0000000000000ull : 0ull;
  if (t < ns) cycles[t] = 0;
  const int rows = ny - nk;  // 0..2
  if (t < ns * rows * nx) {
    const int s = t / (rows * nx), q = t - s * rows * nx, jr = q / nx;
    z[(size_t)s * nx * ny + (size_t)(jr < j0 ? 0 : ny - 1) * nx + (q - jr * nx)] = 0.f;
  }
}

// w.b of the singular kx = 0 pair (solves 0 and 1), one workgroup each
__global__ void __launch_bounds__(1024) k_sep_null(const double* __restrict__ w, const double* __restrict__ rhs,
                                                   const unsigned char* __restrict__ spec, int n,
                                                   double* __restrict__ wb) {
  __shared__ double red[16];
  const double* rt = rhs + (size_t)blockIdx.x * n;
  double a = 0.0;
  for (int p = threadIdx.x; p < n; p += 1024) a += spec[p] ? 0.0 : w[p] * -rt[p];
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < 16; ++q) t += red[q];
    wb[blockIdx.x] = t;
  }
}

struct SepStencil {
  const double* c;      // c1..c8 [8][n]
  const double* base;   // (-s9 + corr9) [n], then J [n]
  const unsigned char* spec;
  const double* kx2;    // per mode
  int nx, ny, n;
};

// A x at point p of a plane x (periodic ends: the virtual columns)
template <bool PER, typename T>
__device__ inline double stencil(double k0, double k2, double k4, double k6, double k9, const T* __restrict__ x, int p,
                                 int i, int j, int nx, int ny) {
  const int e = i < nx - 1 ? p + 1 : PER ? p - (nx - 2) : p;
  const int w = i > 0 ? p - 1 : PER ? p + (nx - 2) : p;
  const int nn = j < ny - 1 ? p + nx : p, ss = j > 0 ? p - nx : p;
  const T xe = x[e], xw = x[w], xn = x[nn], xs = x[ss], xc = x[p];
  return (k0 * (double)xe + k2 * (double)xn) + (k4 * (double)xw + k6 * (double)xs) + k9 * (double)xc;
}

// The start of a solve that does not begin with r = b as it stands (a start from
// a guess, the singular problem's compatible right-hand side): the residual
// r = b - guess A phi and its max.
template <bool PER, int RU>
__global__ void __launch_bounds__(256) k_sep_start(SepStencil S, int nsolve, const double* __restrict__ guessp,
                                                   const double* __restrict__ rhs, const double* __restrict__ phi,
                                                   const double* __restrict__ wb, int pin, int su,
                                                   double* __restrict__ r, unsigned long long* __restrict__ rm) {
  const double g = guessp ? *guessp : 0.0;
  const int p0 = blockIdx.x * (256 * RU) + threadIdx.x;
  const int s0 = blockIdx.y * su, s1 = min(s0 + su, nsolve);
  for (int s = s0; s < s1; ++s) {
    const double* rt = rhs + (size_t)s * S.n;
    const double* ph = phi + (size_t)s * S.n;
    double mx = 0.0;
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      const int p = p0 + 256 * u;
      if (p >= S.n) continue;
      const bool sp = S.spec[p];
      double v = sp ? 0.0 : -rt[p];
      if (wb && s < 2 && p == pin) v -= wb[s];
      if (g != 0.0 && !sp) {
        // the guess is zero at specified points
        const int j = p / S.nx, i = p - j * S.nx;
        const int e = i < S.nx - 1 ? p + 1 : PER ? p - (S.nx - 2) : p, w = i > 0 ? p - 1 : PER ? p + (S.nx - 2) : p;
        const int nn = j < S.ny - 1 ? p + S.nx : p, ss = j > 0 ? p - S.nx : p;
        const double xe = S.spec[e] ? 0.0 : ph[e], xw = S.spec[w] ? 0.0 : ph[w];
        const double xn = S.spec[nn] ? 0.0 : ph[nn], xs = S.spec[ss] ? 0.0 : ph[ss];
        const double k9 = S.base[p] - S.kx2[s >> 1] * S.base[S.n + p];
        v -= g * ((S.c[p] * xe + S.c[2 * (size_t)S.n + p] * xn) +
                  (S.c[4 * (size_t)S.n + p] * xw + S.c[6 * (size_t)S.n + p] * xs) + k9 * ph[p]);
      }
      r[(size_t)s * S.n + p] = v;
      mx = fmax(mx, fabs(v));
    }
    wave_max_to(rm + s, mx);
  }
}

// phi += z, r -= A z and max|r| of every solve that has not ended (first pass:
// phi = guess*phi + z; from a zero start r is b, read from the right-hand
// sides).  Bound by memory: 36 bytes per point and solve (28 in the first
// pass).
template <bool PER, int RU>
__global__ void __launch_bounds__(256) k_sep_update(SepStencil S, int nsolve, int first, int from_rhs, int it,
                                                    const double* __restrict__ guessp,
                                                    const double* __restrict__ rhs, const float* __restrict__ z,
                                                    double* __restrict__ r, double* __restrict__ phi,
                                                    const unsigned long long* __restrict__ rm,
                                                    unsigned long long* __restrict__ rm_next, double tol,
                                                    int* __restrict__ cycles, int su) {
  const int p0 = blockIdx.x * (256 * RU) + threadIdx.x;
  const int s0 = blockIdx.y * su, s1 = min(s0 + su, nsolve);
  const double g = (first && guessp) ? *guessp : 0.0;
  if (blockIdx.x == 0 && threadIdx.x < s1 - s0) {
    const int s = s0 + threadIdx.x;
    if (solved(rm, s, tol))
      atomicMax(rm_next + s, rm[s]);  // carried to the last pass
    else
      cycles[s] = it;
  }
  int i[RU], j[RU], pp[RU];
  bool in[RU], sp[RU];
  double k0[RU], k2[RU], k4[RU], k6[RU], kb[RU], kj[RU];
#pragma unroll
  for (int u = 0; u < RU; ++u) {
    const int p = p0 + 256 * u;
    in[u] = p < S.n;
    const int q = in[u] ? p : S.n - 1;
    pp[u] = q;
    j[u] = q / S.nx;
    i[u] = q - j[u] * S.nx;
    sp[u] = S.spec[q];
    k0[u] = S.c[q];
    k2[u] = S.c[2 * (size_t)S.n + q];
    k4[u] = S.c[4 * (size_t)S.n + q];
    k6[u] = S.c[6 * (size_t)S.n + q];
    kb[u] = S.base[q];
    kj[u] = S.base[S.n + q];
  }
  for (int s = s0; s < s1; ++s) {
    const size_t o = (size_t)s * S.n;
    if (solved(rm, s, tol)) {
      // a solve that met the tolerance at its start takes the scaled guess
      if (first)
        for (int u = 0; u < RU; ++u)
          if (in[u]) phi[o + pp[u]] = (g != 0.0 && !sp[u]) ? g * phi[o + pp[u]] : 0.0;
      continue;
    }
    const double kx2 = S.kx2[s >> 1];
    double mx = 0.0, rv[RU], ph[RU], az[RU], zc[RU];
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      const int p = pp[u];
      rv[u] = from_rhs ? -rhs[o + p] : r[o + p];
      ph[u] = (!first || g != 0.0) ? phi[o + p] : 0.0;
      zc[u] = (double)z[o + p];
      az[u] = stencil<PER>(k0[u], k2[u], k4[u], k6[u], kb[u] - kx2 * kj[u], z + o, p, i[u], j[u], S.nx, S.ny);
    }
#pragma unroll
    for (int u = 0; u < RU; ++u) {
      if (first) {
        if (from_rhs && sp[u]) rv[u] = 0.0;
        ph[u] = sp[u] ? 0.0 : g * ph[u];
      }
      const double rn = rv[u] - az[u];
      if (in[u]) {
        r[o + pp[u]] = rn;
        phi[o + pp[u]] = ph[u] + zc[u];
        mx = fmax(mx, fabs(rn));
      }
    }
    wave_max_to(rm_next + s, mx);
  }
}

// the singular pair: the solution with phi = 0 at the pin
__global__ void __launch_bounds__(1024) k_sep_shift(double* __restrict__ phi, int n, int pin) {
  double* p = phi + (size_t)blockIdx.x * n;
  const double v = p[pin];
  __syncthreads();
  for (int t = threadIdx.x; t < n; t += 1024) p[t] -= v;
}

// Eigenvalues and eigenvectors of the symmetric tridiagonal matrix (d, e):
// the implicit QL method with Wilkinson's shift of Martin and Wilkinson (1968;
// EISPACK's imtql2, with its recovery where a rotation vanishes), the rotations
// accumulated on the rows of zt (zt[k] is the eigenvector of d[k] on exit).
bool tridiag_eigen(std::vector<double>& d, std::vector<double> e, std::vector<double>& zt) {
  const int n = (int)d.size();
  zt.assign((size_t)n * n, 0.0);
  for (int k = 0; k < n; ++k) zt[(size_t)k * n + k] = 1.0;
  e.resize(n, 0.0);
  for (int l = 0; l < n; ++l) {
    for (int iter = 0;; ++iter) {
      int m = l;
      for (; m < n - 1; ++m)
        if (std::fabs(e[m]) <= 1.1e-16 * (std::fabs(d[m]) + std::fabs(d[m + 1]))) break;
      if (m == l) break;
      if (iter == 60) return false;
      const double h = (d[l + 1] - d[l]) / (2.0 * e[l]);
      double g = d[m] - d[l] + e[l] / (h + std::copysign(std::hypot(h, 1.0), h));
      double s = 1.0, c = 1.0, p = 0.0;
      bool cut = false;
      for (int i = m - 1; i >= l; --i) {
        const double f = s * e[i], b = c * e[i];
        const double rr = std::hypot(f, g);
        e[i + 1] = rr;
        if (rr == 0.0) {
          d[i + 1] -= p;
          e[m] = 0.0;
          cut = true;
          break;
        }
        s = f / rr;
        c = g / rr;
        const double q = d[i + 1] - p;
        const double t = (d[i] - q) * s + 2.0 * c * b;
        p = s * t;
        d[i + 1] = q + p;
        g = c * t - b;
        double* z0 = &zt[(size_t)i * n];
        double* z1 = z0 + n;
        for (int k = 0; k < n; ++k) {
          const double u = z1[k], v = z0[k];
          z1[k] = s * v + c * u;
          z0[k] = c * v - s * u;
        }
      }
      if (cut) continue;
      d[l] -= p;
      e[l] = g;
      e[m] = 0.0;
    }
  }
  return true;
}

// 16-row tiles per workgroup of a product over mtiles tiles and ncols columns:
// up to 12 (96 accumulator registers), fewer where that leaves the chip idle
int pick_mt(int mtiles, int ncols) {
  static const int opt[] = {12, 9, 8, 6, 4, 3, 2, 1};
  const int cb = (ncols + kCols - 1) / kCols;
  int best = 1;
  long cost = -1;
  for (int mt : opt) {
    const int nmb = (mtiles + mt - 1) / mt;
    // matrix instructions of the slowest compute unit (two workgroups run on
    // one side by side), plus each workgroup's reads of its columns
    const long waves = ((long)cb * nmb + 255) / 256;
    const long c = waves * (mt * 2 + 3);
    if (cost < 0 || c < cost) {
      cost = c;
      best = mt;
    }
  }
  return best;
}

// A (rows x cols, row-major) in matrix-core operand order [cols/4][tiles][64]
std::vector<float> pack_a(const std::vector<double>& a, int rows, int cols, int mtt) {
  const int nk4 = ((cols + 15) / 16) * 4;
  std::vector<float> o((size_t)nk4 * mtt * 64, 0.f);
  for (int q = 0; q < nk4; ++q)
    for (int m = 0; m < mtt; ++m)
      for (int l = 0; l < 64; ++l) {
        const int r = m * 16 + (l & 15), c = q * 4 + (l >> 4);
        if (r < rows && c < cols) o[((size_t)q * mtt + m) * 64 + l] = (float)a[(size_t)r * cols + c];
      }
  return o;
}

template <typename T>
int upload(T** to, const std::vector<T>& v) {
  EKM_CHECK(hipMalloc((void**)to, v.size() * sizeof(T)));
  EKM_CHECK(hipMemcpy(*to, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return EKM_OK;
}

}  // namespace

int sep_plan_build(SepPlan& sp, const SepProblem& q, int nsolve_max) {
  sp.on = 0;
  const HostMgLevel& L = *q.fine;
  const int nx = L.nx, ny = L.ny;
  const size_t n = (size_t)nx * ny;
  if (nx < 4 || ny < 4 || nx > 832) return EKM_OK;
  // the unknowns: rows j0..j1-1, columns i0..i1-1 (specified ends left out)
  int j0 = 0, j1 = ny, i0 = 0, i1 = nx;
  const int jm = ny / 2, im = nx / 2;
  if (q.spec[im]) j0 = 1;
  if (q.spec[im + (size_t)nx * (ny - 1)]) j1 = ny - 1;
  if (q.spec[(size_t)nx * jm]) i0 = 1;
  if (q.spec[nx - 1 + (size_t)nx * jm]) i1 = nx - 1;
  const int nk = j1 - j0;
  for (int j = 0; j < ny; ++j)
    for (int i = 0; i < nx; ++i) {
      const bool un = j >= j0 && j < j1 && i >= i0 && i < i1;
      const size_t p = i + (size_t)nx * j;
      if (un == (bool)q.spec[p]) return EKM_OK;
      if (un && !(L.jl[p] > 0.0)) return EKM_OK;
      if (un && !q.per && ((i == i0 && i == 0 && L.c[4 * n + p] != 0.0) || (i == nx - 1 && L.c[p] != 0.0))) return EKM_OK;
      if (un && ((j == 0 && L.c[6 * n + p] != 0.0) || (j == ny - 1 && L.c[2 * n + p] != 0.0))) return EKM_OK;
    }
  // J = W(i) M(j) from its middle row and column; the one-dimensional operators
  // are the medians of the scaled coefficients across the other direction
  std::vector<double> W(nx, 0.0), Mj(ny, 0.0), lz(nx, 0.0), uz(nx, 0.0), dz(nx, 0.0), ly(ny, 0.0), uy(ny, 0.0);
  for (int i = i0; i < i1; ++i) W[i] = L.jl[i + (size_t)nx * jm] / L.jl[im + (size_t)nx * jm];
  for (int j = j0; j < j1; ++j) Mj[j] = L.jl[im + (size_t)nx * j];
  std::vector<double> buf;
  auto median = [&](int lo, int hi, auto&& f) {
    buf.clear();
    for (int k = lo; k < hi; ++k) buf.push_back(f(k));
    std::nth_element(buf.begin(), buf.begin() + buf.size() / 2, buf.end());
    return buf[buf.size() / 2];
  };
  auto sc = [&](int c, int i, int j) { return L.c[c * n + i + (size_t)nx * j] / (W[i] * Mj[j]); };
  for (int i = i0; i < i1; ++i) {
    lz[i] = median(j0, j1, [&](int j) { return sc(4, i, j); });
    uz[i] = median(j0, j1, [&](int j) { return sc(0, i, j); });
    dz[i] = -(lz[i] + uz[i]);
  }
  for (int j = j0; j < j1; ++j) {
    ly[j] = median(i0, i1, [&](int i) { return sc(6, i, j); });
    uy[j] = median(i0, i1, [&](int i) { return sc(2, i, j); });
  }
  double dev = 0.0;
  for (int j = j0; j < j1; ++j)
    for (int i = i0; i < i1; ++i) {
      const size_t p = i + (size_t)nx * j;
      auto rel = [&](double v, double f) { return std::fabs(v - f) / std::max(std::fabs(f), 1e-300); };
      if (lz[i] != 0.0 || sc(4, i, j) != 0.0) dev = std::max(dev, rel(sc(4, i, j), lz[i]));
      if (uz[i] != 0.0 || sc(0, i, j) != 0.0) dev = std::max(dev, rel(sc(0, i, j), uz[i]));
      if (ly[j] != 0.0 || sc(6, i, j) != 0.0) dev = std::max(dev, rel(sc(6, i, j), ly[j]));
      if (uy[j] != 0.0 || sc(2, i, j) != 0.0) dev = std::max(dev, rel(sc(2, i, j), uy[j]));
      dev = std::max(dev, std::fabs(L.jl[p] / (W[i] * Mj[j]) - 1.0));
      const double sum = L.c[p] + L.c[2 * n + p] + L.c[4 * n + p] + L.c[6 * n + p];
      dev = std::max(dev, std::fabs((-L.s9[p] + L.corr9[p]) + sum) / sum);
      if (!(lz[i] >= 0.0 && uz[i] >= 0.0 && ly[j] >= 0.0 && uy[j] >= 0.0 && sum > 0.0)) return EKM_OK;
    }
  if (!(dev <= kSepDev)) return EKM_OK;
  // Ly = S^-1/2 T S^1/2 with T symmetric
  std::vector<double> d(nk), e(nk, 0.0), s(nk, 1.0), zt;
  for (int k = 0; k < nk; ++k) d[k] = -(ly[j0 + k] + uy[j0 + k]);
  for (int k = 0; k + 1 < nk; ++k) {
    const double up = uy[j0 + k], lo = ly[j0 + k + 1];
    if (!(up > 0.0 && lo > 0.0)) return EKM_OK;
    s[k + 1] = s[k] * up / lo;
    e[k] = std::sqrt(up * lo);
  }
  if (!tridiag_eigen(d, e, zt)) return EKM_OK;
  int kmax = 0;
  for (int k = 1; k < nk; ++k)
    if (d[k] > d[kmax]) kmax = k;
  const bool sing = q.pin >= 0;
  if (sing) d[kmax] = 0.0;  // the constants
  std::vector<double> af((size_t)nk * nk, 0.0), ab((size_t)nk * nk, 0.0);
  for (int k = 0; k < nk; ++k)
    for (int j = 0; j < nk; ++j) {
      const double v = zt[(size_t)k * nk + j], rs = std::sqrt(s[j]);
      af[(size_t)k * nk + j] = v * rs / Mj[j0 + j];
      ab[(size_t)j * nk + k] = v / rs;
    }
  sp.nx = nx;
  sp.ny = ny;
  sp.nk = nk;
  sp.j0 = j0;
  sp.nmode = q.nmode;
  sp.nsolve_max = nsolve_max;
  sp.per = q.per;
  sp.pin = q.pin;
  const int mtiles = (nk + 15) / 16;
  sp.mt = pick_mt(mtiles, nsolve_max * nx);
  const int mtt = (mtiles + sp.mt - 1) / sp.mt * sp.mt;
  const std::vector<float> pf = pack_a(af, nk, nk, mtt), pb = pack_a(ab, nk, nk, mtt);
  if (upload(&sp.af, pf) != EKM_OK || upload(&sp.ab, pb) != EKM_OK) return EKM_ERR_HIP;
  std::vector<double> base(2 * n);
  for (size_t p = 0; p < n; ++p) {
    base[p] = -L.s9[p] + L.corr9[p];
    base[n + p] = L.jl[p];
  }
  if (upload(&sp.base, base) != EKM_OK) return EKM_ERR_HIP;
  const std::vector<double> kx2(q.kx2, q.kx2 + q.nmode);
  if (upload(&sp.kx2, kx2) != EKM_OK) return EKM_ERR_HIP;
  // modes whose lines are solved in FP64
  double dmax = 0.0, lmin = 1e300;
  for (int i = i0; i < i1; ++i) dmax = std::max(dmax, std::fabs(dz[i]));
  for (int k = 0; k < nk; ++k) lmin = std::min(lmin, std::fabs(d[k]));
  sp.nmode64 = 0;
  while (sp.nmode64 < q.nmode && lmin + kx2[sp.nmode64] < kSepFp64Shift * dmax) ++sp.nmode64;
  std::vector<double> z1(4 * (size_t)nx);
  for (int i = 0; i < nx; ++i) {
    const bool un = i >= i0 && i < i1;
    z1[i] = un && i > i0 - (q.per ? 1 : 0) ? lz[i] : 0.0;
    z1[nx + i] = un && i < i1 - (q.per ? 0 : 1) ? uz[i] : 0.0;
    z1[2 * nx + i] = dz[i];
    z1[3 * nx + i] = W[i];
  }
  double *d_z1 = nullptr, *d_lam = nullptr;
  if (upload(&d_z1, z1) != EKM_OK || upload(&d_lam, d) != EKM_OK) return EKM_ERR_HIP;
  const long ls = line_stride(nx, q.per);
  const int n32 = q.nmode - sp.nmode64;
  if (n32 > 0) EKM_CHECK(hipMalloc((void**)&sp.fac, (size_t)n32 * nk * ls * sizeof(float)));
  if (sp.nmode64 > 0) EKM_CHECK(hipMalloc((void**)&sp.fac64, (size_t)sp.nmode64 * nk * ls * sizeof(double)));
  const int pk = sing ? kmax : -1, pi = sing ? q.pin % nx : -1;
  auto blocks = [](long t) { return dim3((unsigned)((t + 63) / 64)); };
  if (q.per) {
    if (n32 > 0)
      hipLaunchKernelGGL((k_sep_factor<float, true>), blocks((long)n32 * nk), dim3(64), 0, 0, nx, nk, sp.nmode64, n32, d_z1,
                         d_lam, sp.kx2, pk, pi, sp.fac);
    if (sp.nmode64 > 0)
      hipLaunchKernelGGL((k_sep_factor<double, true>), blocks((long)sp.nmode64 * nk), dim3(64), 0, 0, nx, nk, 0, sp.nmode64,
                         d_z1, d_lam, sp.kx2, pk, pi, sp.fac64);
  } else {
    if (n32 > 0)
      hipLaunchKernelGGL((k_sep_factor<float, false>), blocks((long)n32 * nk), dim3(64), 0, 0, nx, nk, sp.nmode64, n32, d_z1,
                         d_lam, sp.kx2, pk, pi, sp.fac);
    if (sp.nmode64 > 0)
      hipLaunchKernelGGL((k_sep_factor<double, false>), blocks((long)sp.nmode64 * nk), dim3(64), 0, 0, nx, nk, 0, sp.nmode64,
                         d_z1, d_lam, sp.kx2, pk, pi, sp.fac64);
  }
  EKM_CHECK(hipGetLastError());
  EKM_CHECK(hipDeviceSynchronize());
  (void)hipFree(d_z1);
  (void)hipFree(d_lam);
  EKM_CHECK(hipMalloc((void**)&sp.wb, 2 * sizeof(double)));
  EKM_CHECK(hipMalloc((void**)&sp.rmax, (size_t)(kSepIter + 1) * nsolve_max * sizeof(unsigned long long)));
  sp.on = 1;
  return EKM_OK;
}

void sep_plan_free(SepPlan& sp) {
  void* p[] = {sp.af, sp.ab, sp.fac, sp.fac64, sp.base, sp.kx2, sp.wb, sp.rmax};
  for (void* q : p)
    if (q) (void)hipFree(q);
  sp = SepPlan();
}

namespace {

template <typename TI>
int launch_gemm(int mt, const float* A, int M, int nx, int nsolve, long ld, const TI* X, float alpha, float* Y,
                const unsigned long long* rm, double tol, hipStream_t st) {
  const int mtiles = (M + 15) / 16, nmb = (mtiles + mt - 1) / mt, mtt = nmb * mt;
  const int ncols = nsolve * nx, cb = (ncols + kCols - 1) / kCols;
  const dim3 grid((unsigned)((cb + 7) / 8 * 8 * nmb));
#define CASE(N)                                                                                                       \
  case N:                                                                                                             \
    hipLaunchKernelGGL((k_sep_gemm<N, TI>), grid, dim3(256), 0, st, A, mtt, mtiles, M, nx, ncols, ld, X, alpha, Y, rm, tol, \
                       nmb);                                                                                          \
    break
  switch (mt) {
    CASE(1);
    CASE(2);
    CASE(3);
    CASE(4);
    CASE(6);
    CASE(8);
    CASE(9);
    CASE(12);
    default: return EKM_ERR_ARG;
  }
#undef CASE
  EKM_CHECK(hipGetLastError());
  return EKM_OK;
}

template <typename T, bool PER>
int launch_lines(int nx, int nk, int m0, int nm, const T* fac, float* t, long ld, const unsigned long long* rm, double tol,
                 int nsolve, hipStream_t st) {
  const dim3 grid((unsigned)(((long)nm * nk + 3) / 4));
#define CASE(N)                                                                                                      \
  hipLaunchKernelGGL((k_sep_lines<T, N, PER>), grid, dim3(256), 0, st, nx, nk, m0, nm, ld, fac, t, rm, tol, nsolve)
  const int cm = (nx + 63) / 64;
  if (cm <= 1) CASE(1);
  else if (cm <= 2) CASE(2);
  else if (cm <= 3) CASE(3);
  else if (cm <= 5) CASE(5);
  else if (cm <= 7) CASE(7);
  else if (cm <= 9) CASE(9);
  else CASE(13);
#undef CASE
  EKM_CHECK(hipGetLastError());
  return EKM_OK;
}

// A thread's loads of all its points are in flight together, and its points'
// coefficients serve all solves of its workgroup: as many of both as leave the
// chip 4 workgroups per compute unit (1024), below which it stands partly idle.
// Together with the first pass that takes a zero start's residual from the
// right-hand sides, a step takes this much of its time with 2 points and 8 solves
// for every size (both builds in turn on one box): 256x385x769 with both subgrid
// models 0.956, 512x257x513 0.969, 256x193x257 0.965, 64x65x65 from graphs 0.947.
UpdSplit pick_upd(int n, int nsolve) {
  for (int rows = 4; rows > 1; rows >>= 1)
    for (int solves = 8; solves > 1; solves >>= 1)
      if ((long)((n + 256 * rows - 1) / (256 * rows)) * ((nsolve + solves - 1) / solves) >= 1024) return {rows, solves};
  return {1, 2};
}

template <bool PER>
int solve_typed(const SepPlan& sp, const SepBuffers& b, int nsolve, const double* guess, hipStream_t st) {
  const int nx = sp.nx, ny = sp.ny, nk = sp.nk, nmode = (nsolve + 1) / 2;
  const int n = nx * ny, K = sep_iters(b.maxit), nm = sp.nsolve_max;
  const int n64 = sp.nmode64 < nmode ? sp.nmode64 : nmode;
  const SepStencil S{b.cf64, sp.base, b.spec, sp.kx2, nx, ny, n};
  float *t1 = b.t, *t2 = b.t + (size_t)nsolve * n;
  unsigned long long* rm = sp.rmax;
  const bool sing = b.wnull != nullptr;
  // r = b as it stands is read from the right-hand sides by the first pass
  const int store = guess != nullptr || sing;
  const int ncl = std::max(std::max((K + 1) * nm, nsolve), nsolve * (ny - nk) * nx);
  hipLaunchKernelGGL(k_sep_clear, dim3((unsigned)((ncl + 255) / 256)), dim3(256), 0, st, rm, (K + 1) * nm, nm, !store,
                     b.cycles, nsolve, t2, nx, ny, sp.j0, nk);
  if (sing) hipLaunchKernelGGL(k_sep_null, dim3(2), dim3(1024), 0, st, b.wnull, b.rhs, b.spec, n, sp.wb);
  const UpdSplit us = pick_upd(n, nsolve);
  const unsigned gy = (unsigned)((nsolve + us.solves - 1) / us.solves);
  EKM_CHECK(hipGetLastError());
  const dim3 gu((unsigned)((n + 256 * us.rows - 1) / (256 * us.rows)), gy);
#define START(RU)                                                                                                 \
  hipLaunchKernelGGL((k_sep_start<PER, RU>), gu, dim3(256), 0, st, S, nsolve, guess, b.rhs, b.phi,                \
                     sing ? sp.wb : nullptr, sp.pin, us.solves, b.r, rm)
  if (store) {
    if (us.rows == 4) START(4);
    else if (us.rows == 2) START(2);
    else START(1);
  }
#undef START
  EKM_CHECK(hipGetLastError());
  for (int it = 1; it <= K; ++it) {
    const unsigned long long* rp = rm + (size_t)(it - 1) * nm;
    const bool first = it == 1;
    const int from_rhs = first && !store;
    // rows j0..j0+nk-1 hold the unknowns
    const long jo = (long)sp.j0 * nx;
    int e = launch_gemm<double>(sp.mt, sp.af, nk, nx, nsolve, n, (from_rhs ? b.rhs : (const double*)b.r) + jo,
                                from_rhs ? -1.f : 1.f, t1, rp, b.tol, st);
    if (e != EKM_OK) return e;
    if (n64 > 0) e = launch_lines<double, PER>(nx, nk, 0, n64, sp.fac64, t1, n, rp, b.tol, nsolve, st);
    if (e == EKM_OK && nmode > n64)
      e = launch_lines<float, PER>(nx, nk, sp.nmode64, nmode - n64, sp.fac, t1, n, rp, b.tol, nsolve, st);
    if (e != EKM_OK) return e;
    e = launch_gemm<float>(sp.mt, sp.ab, nk, nx, nsolve, n, t1, 1.f, t2 + jo, rp, b.tol, st);
    if (e != EKM_OK) return e;
#define UPD(RU)                                                                                                        \
  hipLaunchKernelGGL((k_sep_update<PER, RU>), gu, dim3(256), 0, st, S, nsolve, (int)first, from_rhs, it, guess, b.rhs, t2, \
                     b.r, b.phi, rp, rm + (size_t)it * nm, b.tol, b.cycles, us.solves)
    if (us.rows == 4) UPD(4);
    else if (us.rows == 2) UPD(2);
    else UPD(1);
#undef UPD
    EKM_CHECK(hipGetLastError());
  }
  if (sing) hipLaunchKernelGGL(k_sep_shift, dim3(2), dim3(1024), 0, st, b.phi, n, sp.pin);
  EKM_CHECK(hipGetLastError());
  return EKM_OK;
}

}  // namespace

int sep_solve(const SepPlan& sp, const SepBuffers& b, int nsolve, const double* guess, hipStream_t st) {
  return sp.per ? solve_typed<true>(sp, b, nsolve, guess, st) : solve_typed<false>(sp, b, nsolve, guess, st);
}
