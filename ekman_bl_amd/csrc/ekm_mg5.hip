// ekm_mg5.hip -- the MUDPACK replica on grids without cross terms (5-point
// rows on every level): the same iterates as ekm_mg.hip, bit for bit, in a
// form whose chains of dependent steps are several times shorter.
//
// MUDPACK's four colours are the points with i + j = 2, 3, 0, 1 (mod 4), each
// swept as four row phases because a 9-point row couples points of one colour
// through its corners.  A 5-point row does not: its four neighbours have the
// two adjacent colours, so the four row phases of a colour are independent
// and a sweep is 4 steps instead of 16, with the same values.  The products
// with the zero corner coefficients are left out (adding a zero changes no
// value), and on the levels held in LDS the division by c9 is the correctly
// rounded quotient from the reciprocal (Markstein's correction steps: with
// y = 1/c9 rounded and q within one ulp, q + (x - q c9) y rounds correctly).
// That holds for finite operands whose quotient and products neither overflow
// nor fall below the normal range; a solve that has overflowed may hold NaN
// where the division gives an infinity (the sweeps around it turn both to NaN).
//
// A solve is bound by the latency of those steps (a W cycle visits level l
// 2^(ngrid-l) times), so every array is kept in a colour layout, where the
// points of a step and each of their neighbours are consecutive words: levels
// whose colours hold at most 64 points are swept by wave 0 with a visit's
// coefficients in registers; the next ones by the whole block from LDS (first
// all arrays, then the correction alone, as it fits), the finest from global
// memory with the first points of the next step requested before the barrier.
// The transfers evaluate MUDPACK's expressions with selected operands instead
// of by cases, and the prolongation's y pass adds where it interpolates.
// Measured per launch: 64x65x65 (44 solves) about 6 -> 1.8 ms, 256x193x257
// (172 solves) 33 -> 12.5 ms; a sweep of a one-wavefront level 0.9 us.
#include <algorithm>
#include <cstring>
#include <vector>

#include "ekm_host.h"
#include "ekm_internal.h"
#include "ekm_mg5.h"

namespace {

constexpr int kMaxLev5 = 16;
enum Op5 : int { OP5_RELAX = 0, OP5_RESTRICT = 1, OP5_CORRECT = 2, OP5_FMGPROL = 3 };
// where a level's arrays live: 0 global; 1 the correction in LDS; 2 all in LDS;
// 3 all in LDS and at most 64 points per colour
enum Store5 : int { ST_GLOBAL = 0, ST_PHI = 1, ST_LDS = 2, ST_WAVE = 3 };

struct Lev5 {
  int nx, ny, rs, cs, e4;   // points, row and colour strides, elements of an array
  int st;
  int phi, rhs, c9;         // offsets in LDS or in the solve's workspace (c9 of an LDS level: after c0, c2, c4, c6)
  int tab;                  // ST_WAVE levels: [4][64] points of the colours 2, 3, 0, 1 (i | j << 16, -1: none)
  int cf;                   // LDS levels: c0, c2, c4, c6, c9, 1/c9 from here, e4 apart
  const double* c;          // c0, c2, c4, c6, s9, corr9, J [7][e4] (zero where there is no point)
};

struct Mg5 {
  int ngrid, nxa, nxb, nyc, nyd, maxcy, nfx, nfy;
  double tolmax;
  int ws;                   // doubles per solve
  int resf_g, resf_l;       // scratch of a restriction (residual) or a prolongation (x-interpolated coarse rows)
  int red;                  // LDS reduction scratch
  int tab, tab_n;           // point tables: LDS offset (doubles) and count (ints)
  int nops_fmg, nops_w;
  Lev5 lev[kMaxLev5 + 1];
  const int* tabg;          // point tables (global copy)
  const int* ops;           // full-multigrid start, then one W cycle: (count << 16) | (op << 8) | level
};

extern __shared__ double lds5[];

__host__ __device__ inline int pos5(const Lev5& L, int i, int j) { return ((i + j) & 3) * L.cs + j * L.rs + (i >> 2); }

// an array in LDS, in global memory, or in either (pointers to either memory
// take flat loads, which wait on both)
typedef __attribute__((address_space(1))) double gdouble;
enum Mem5 : int { M_GLOBAL = 0, M_LDS = 1, M_ANY = 2 };
template <int M>
struct Arr {
  double* g;
  int o;
  __device__ double get(int k) const {
    if constexpr (M == M_LDS) return lds5[o + k];
    else if constexpr (M == M_GLOBAL) return ((const gdouble*)g)[k];
    else return g[k];
  }
  __device__ void put(int k, double v) const {
    if constexpr (M == M_LDS)
      lds5[o + k] = v;
    else if constexpr (M == M_GLOBAL)
      ((gdouble*)g)[k] = v;
    else
      g[k] = v;
  }
};
template <int M>
__device__ inline Arr<M> arr5(bool lds, double* W, int off) {
  return Arr<M>{M == M_LDS ? nullptr : ((M == M_ANY && lds) ? lds5 : W) + off, off};
}

// The value is needed here: keeps the compiler from moving its load into a later
// branch, where the loads of several points would wait for each other.
__device__ inline void keep(double& x) { asm volatile("" : "+v"(x)); }

struct Fd5 {
  float rcp;
  int d;
};
__device__ inline Fd5 fd5(int d) { return Fd5{1.0f / (float)d, d}; }
// t = q*d + r for 0 <= t < 2^22 through a float reciprocal and one correction
__device__ inline void dm5(int t, const Fd5& f, int& q, int& r) {
  q = (int)((float)t * f.rcp);
  r = t - q * f.d;
  if (r < 0) {
    --q;
    r += f.d;
  } else if (r >= f.d) {
    ++q;
    r -= f.d;
  }
}

// slot t of a level's colour layout (4 * np of them, np = ny * rs): its point,
// false where it holds none
__device__ inline bool slot5(const Lev5& L, int t, int np, const Fd5& fp, const Fd5& f, int& i, int& j) {
  int s, w, jj, a;
  dm5(t, fp, s, w);
  dm5(w, f, jj, a);
  j = jj + 1;
  i = 4 * a + ((s - j) & 3);
  return i >= 1 && i <= L.nx;
}

// Executor: the whole block, or wave 0 alone (levels of ST_WAVE)
template <bool WAVE>
__device__ inline void sync5() {
  if constexpr (WAVE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  } else {
    __syncthreads();
  }
}

// (rhs - (c1 phi_E + c3 phi_N + c5 phi_W + c7 phi_S)), MUDPACK's order
__device__ inline double gs_num(double c0, double c2, double c4, double c6, double rhs, double e, double n, double w,
                                double s) {
  return rhs - (c0 * e + c2 * n + c4 * w + c6 * s);
}
// x / c, correctly rounded, from rc = 1/c correctly rounded
__device__ inline double div_rc(double x, double c, double rc) {
  const double q = x * rc;
  const double q1 = __builtin_fma(__builtin_fma(-c, q, x), rc, q);
  return __builtin_fma(__builtin_fma(-c, q1, x), rc, q1);
}

// virtual points of periodic ends, after each colour
template <bool WAVE, int PL>
__device__ inline void periodic5(const Mg5& g, const Lev5& L, const Arr<PL>& phi, int tid, int nt) {
  const int nx = L.nx, ny = L.ny, mx = g.nxa == 0 ? ny : 0, m = mx + (g.nyc == 0 ? nx : 0);
  for (int t = tid; t < m; t += nt) {
    if (t < mx) {
      const int j = t + 1;
      phi.put(pos5(L, 0, j), phi.get(pos5(L, nx - 1, j)));
      phi.put(pos5(L, nx + 1, j), phi.get(pos5(L, 2, j)));
    } else {
      const int i = t - mx + 1;
      phi.put(pos5(L, i, 0), phi.get(pos5(L, i, ny - 1)));
      phi.put(pos5(L, i, ny + 1), phi.get(pos5(L, i, 2)));
    }
  }
  sync5<WAVE>();
}

// Sweeps of a level with at most 64 points per colour by wave 0, one point of
// the colour per lane; coefficients and right-hand side are read once for all
// sweeps of the visit.
__device__ __forceinline__ void relax_wave5(const Mg5& g, const Lev5& L, int sweeps) {
  const int lane = threadIdx.x;
  const int* tab = reinterpret_cast<const int*>(lds5 + g.tab) + L.tab + lane;
  double k0[4], k2[4], k4[4], k6[4], k9[4], kr[4], rh[4];
  int pc[4], pe[4], pn[4], pw[4], ps[4];
  bool in[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int en = tab[64 * q];
    in[q] = en >= 0;
    const int ii = in[q] ? en & 0xffff : 1, jc = in[q] ? en >> 16 : 1;
    pc[q] = pos5(L, ii, jc);
    pe[q] = L.phi + pos5(L, ii + 1, jc);
    pn[q] = L.phi + pos5(L, ii, jc + 1);
    pw[q] = L.phi + pos5(L, ii - 1, jc);
    ps[q] = L.phi + pos5(L, ii, jc - 1);
    const double* c = lds5 + L.cf + pc[q];
    k0[q] = c[0];
    k2[q] = c[L.e4];
    k4[q] = c[2 * L.e4];
    k6[q] = c[3 * L.e4];
    k9[q] = c[4 * L.e4];
    kr[q] = c[5 * L.e4];
    rh[q] = lds5[L.rhs + pc[q]];
  }
  const bool per = g.nxa == 0 || g.nyc == 0;
  for (int sw = 0; sw < sweeps; ++sw) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (in[q]) {
        const double x = gs_num(k0[q], k2[q], k4[q], k6[q], rh[q], lds5[pe[q]], lds5[pn[q]], lds5[pw[q]], lds5[ps[q]]);
        lds5[L.phi + pc[q]] = div_rc(x, k9[q], kr[q]);
      }
      sync5<true>();
      if (per) periodic5<true, M_LDS>(g, L, arr5<M_LDS>(true, nullptr, L.phi), lane, 64);
    }
  }
}

struct Pt5 {
  double k0, k2, k4, k6, k9, rh, kr;
  int i, j, p;
  bool in;
};
template <int ST>
__device__ inline Pt5 load_pt5(const Lev5& L, double* W, int t, int np, int s, const Fd5& f) {
  Pt5 r;
  int jj, a;
  dm5(t < np ? t : 0, f, jj, a);
  r.j = jj + 1;
  r.i = 4 * a + ((s - r.j) & 3);
  r.in = t < np && r.i >= 1 && r.i <= L.nx;
  if (!r.in) r.i = r.j = 1;
  r.p = pos5(L, r.i, r.j);
  if constexpr (ST >= ST_LDS) {
    const double* c = lds5 + L.cf + r.p;
    r.k0 = c[0];
    r.k2 = c[L.e4];
    r.k4 = c[2 * L.e4];
    r.k6 = c[3 * L.e4];
    r.k9 = c[4 * L.e4];
    r.kr = c[5 * L.e4];
    r.rh = lds5[L.rhs + r.p];
  } else {
    const gdouble* c = (const gdouble*)L.c + r.p;
    const gdouble* w = (const gdouble*)W + r.p;
    r.k0 = c[0];
    r.k2 = c[L.e4];
    r.k4 = c[2 * (size_t)L.e4];
    r.k6 = c[3 * (size_t)L.e4];
    r.k9 = w[L.c9];
    r.rh = w[L.rhs];
  }
  return r;
}

// points per thread and round of the whole-block passes: their loads are issued
// together.  A round of a global level is one trip to memory (about 2.5 us), an
// LDS level's colour is one round.  (The code of all passes must stay within the
// 64 KB instruction cache: at 80 KB every pass, the LDS levels' too, took 1.5
// times as long, and four points per round of the global levels, with their
// code, gained nothing.)
template <int ST>
constexpr int unroll5 = ST >= ST_LDS ? 1 : 2;

// Sweeps of a level by the whole block
template <int ST>
__device__ __forceinline__ void relax_block5(const Mg5& g, const Lev5& L, double* W, int sweeps) {
  constexpr int U = unroll5<ST>;
  const auto phi = arr5<(ST >= ST_PHI ? M_LDS : M_GLOBAL)>(false, W, L.phi);
  const int tid = threadIdx.x, nt = blockDim.x;
  const int np = L.ny * L.rs;
  const Fd5 f = fd5(L.rs);
  const bool per = g.nxa == 0 || g.nyc == 0;
  Pt5 a[U];
#pragma unroll
  for (int u = 0; u < U; ++u) a[u] = load_pt5<ST>(L, W, tid + u * nt, np, 2, f);
  __syncthreads();
  for (int ph = 0; ph < 4 * sweeps; ++ph) {
    const int s = (2 + ph) & 3;
    for (int t = tid;;) {
      double e[U][4];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        e[u][0] = phi.get(pos5(L, a[u].i + 1, a[u].j));
        e[u][1] = phi.get(pos5(L, a[u].i, a[u].j + 1));
        e[u][2] = phi.get(pos5(L, a[u].i - 1, a[u].j));
        e[u][3] = phi.get(pos5(L, a[u].i, a[u].j - 1));
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) keep(e[u][q]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double v = gs_num(a[u].k0, a[u].k2, a[u].k4, a[u].k6, a[u].rh, e[u][0], e[u][1], e[u][2], e[u][3]);
        const double x = ST >= ST_LDS ? div_rc(v, a[u].k9, a[u].kr) : v / a[u].k9;
        if (a[u].in) phi.put(a[u].p, x);
      }
      t += U * nt;
      if (t >= np) break;
#pragma unroll
      for (int u = 0; u < U; ++u) a[u] = load_pt5<ST>(L, W, t + u * nt, np, s, f);
    }
    // the next step's first points do not depend on this one
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = load_pt5<ST>(L, W, tid + u * nt, np, (s + 1) & 3, f);
    __syncthreads();
    if (per) periodic5<false, (ST >= ST_PHI ? M_LDS : M_GLOBAL)>(g, L, phi, tid, nt);
  }
}

// resmd2cr + res2 (src/mud2cr.f:1618-1665, src/mudcom.f:120-258): level F -> C
template <int SF>
__device__ __forceinline__ void restrict5(const Mg5& g, const Lev5& F, const Lev5& C, double* W) {
  constexpr bool WAVE = SF == ST_WAVE, IN = SF >= ST_LDS;
  const int tid = WAVE ? (int)(threadIdx.x & 63) : (int)threadIdx.x, nt = WAVE ? 64 : (int)blockDim.x;
  if constexpr (!WAVE) __syncthreads();
  if (WAVE && threadIdx.x >= 64) return;
  const int nx = F.nx, ny = F.ny, ncx = C.nx, ncy = C.ny;
  const auto phi = arr5<(SF >= ST_PHI ? M_LDS : M_GLOBAL)>(true, W, F.phi);
  const auto resf = arr5<(IN ? M_LDS : M_GLOBAL)>(IN, W, IN ? g.resf_l : g.resf_g);
  const auto phic = arr5<(IN ? M_LDS : M_ANY)>(C.st >= ST_PHI, W, C.phi);
  const auto rhsc = arr5<(IN ? M_LDS : M_ANY)>(C.st >= ST_LDS, W, C.rhs);
  for (int t = tid; t < C.e4; t += nt) phic.put(t, 0.0);
  // every point of the colour layout, colour by colour
  const int np = ny * F.rs;
  const Fd5 f = fd5(F.rs), fp = fd5(np);
  constexpr int U = unroll5<SF>;
  for (int t0 = tid; t0 < 4 * np; t0 += U * nt) {
    double v[U], e[U][5];
    Pt5 a[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = t0 + u * nt;
      int s, w;
      dm5(t < 4 * np ? t : 0, fp, s, w);
      a[u] = load_pt5<SF>(F, W, w, np, s, f);
      a[u].in = a[u].in && t < 4 * np;
      e[u][0] = phi.get(pos5(F, a[u].i + 1, a[u].j));
      e[u][1] = phi.get(pos5(F, a[u].i, a[u].j + 1));
      e[u][2] = phi.get(pos5(F, a[u].i - 1, a[u].j));
      e[u][3] = phi.get(pos5(F, a[u].i, a[u].j - 1));
      e[u][4] = phi.get(a[u].p);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = a[u].rh - (a[u].k0 * e[u][0] + a[u].k2 * e[u][1] + a[u].k4 * e[u][2] + a[u].k6 * e[u][3] + a[u].k9 * e[u][4]);
#pragma unroll
    for (int u = 0; u < U; ++u) keep(v[u]);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (a[u].in) resf.put(a[u].p, v[u]);
  }
  sync5<WAVE>();
  const int ix = (ncx == nx) ? 0 : 1, jy = (ncy == ny) ? 0 : 1;
  // coarse points colour by colour too: 64 of them read each of the nine
  // residuals from one run of words (lanes that alternate between the colours'
  // planes would take one memory transaction each)
  const int npc = ncy * C.rs;
  const Fd5 fc = fd5(C.rs), fpc = fd5(npc);
  for (int t = tid; t < 4 * npc; t += nt) {
    int ic, jc;
    if (!slot5(C, t, npc, fpc, fc, ic, jc)) continue;
    const int i = ic + ix * (ic - 1), j = jc + jy * (jc - 1);
    int im1 = i - 1, ip1 = i + 1, jm1 = j - 1, jp1 = j + 1;
    if (jc == 1 || jc == ncy) {
      jm1 = j - 1 > 2 ? j - 1 : 2;
      jp1 = j + 1 < ny - 1 ? j + 1 : ny - 1;
      if (j == 1 && g.nyc == 0) jm1 = ny - 1;
      if (j == ny && g.nyc == 0) jp1 = 2;
    }
    if (ic == 1 || ic == ncx) {
      im1 = i - 1 > 2 ? i - 1 : 2;
      ip1 = i + 1 < nx - 1 ? i + 1 : nx - 1;
      if (i == 1 && g.nxa == 0) im1 = nx - 1;
      if (i == nx && g.nxa == 0) ip1 = 2;
    }
#define RF(a, b) resf.get(pos5(F, a, b))
    double v = (RF(im1, jm1) + RF(ip1, jm1) + RF(im1, jp1) + RF(ip1, jp1) +
                2. * (RF(im1, j) + RF(ip1, j) + RF(i, jm1) + RF(i, jp1)) + 4. * RF(i, j)) * .0625;
#undef RF
    if ((g.nxa == 1 && ic == 1) || (g.nxb == 1 && ic == ncx) || (g.nyc == 1 && jc == 1) || (g.nyd == 1 && jc == ncy))
      v = 0.0;
    rhsc.put(pos5(C, ic, jc), v);
  }
  sync5<WAVE>();
}

// Interpolation of an even point of a line of m between its odd points
// (prolon1, src/mudcom.f:420-500): the four operands' indices and which of
// MUDPACK's expressions applies, so that every lane runs the same instructions.
struct Tap5 {
  int a, b, c, d;
  int kind;  // 1: (-a + 9 (b + c) - d)/16; 2: (5 a + 15 b - 5 c + d)/16; 3: (a + b)/2
};
__device__ inline Tap5 tap5(int i, int m, bool cubic, bool per) {
  if (!cubic) return Tap5{i - 1, i + 1, i + 1, i + 1, 3};
  if (i == 2) return per ? Tap5{m - 2, 1, 3, 5, 1} : Tap5{1, 3, 5, 7, 2};
  if (i == m - 1) return per ? Tap5{m - 4, m - 2, m, 3, 1} : Tap5{m, m - 2, m - 4, m - 6, 2};
  return Tap5{i - 3, i - 1, i + 1, i + 3, 1};
}
__device__ inline double interp5(int kind, double a, double b, double c, double d) {
  const double v1 = (-a + 9. * (b + c) - d) * .0625, v2 = (5. * a + 15. * b - 5. * c + d) * .0625;
  return kind == 1 ? v1 : kind == 2 ? v2 : 0.5 * (a + b);
}

// cor2 (src/mudcom.f:502-553) when `add`: phi_F += P phi_C; otherwise the full
// multigrid start's phi_F = P phi_C (src/mud2cr.f:281-290), which sets the
// virtual columns of the coarse rows only.  P (prolon2, src/mudcom.f:261-420):
// the coarse rows are interpolated along x into the scratch X (rows of four
// runs, by column mod 4), then along y where they are added.  Both passes go
// through the points in a level's colour layout.
template <int SF>
__device__ __forceinline__ void correct5(const Mg5& g, const Lev5& C, const Lev5& F, double* W, bool add) {
  constexpr bool WAVE = SF == ST_WAVE, IN = SF >= ST_LDS;
  constexpr int U = unroll5<SF>;
  const int tid = WAVE ? (int)(threadIdx.x & 63) : (int)threadIdx.x, nt = WAVE ? 64 : (int)blockDim.x;
  if constexpr (!WAVE) __syncthreads();
  if (WAVE && threadIdx.x >= 64) return;
  const auto phic = arr5<(IN ? M_LDS : M_ANY)>(C.st >= ST_PHI, W, C.phi);
  const auto phi = arr5<(SF >= ST_PHI ? M_LDS : M_GLOBAL)>(true, W, F.phi);
  const auto X = arr5<(IN ? M_LDS : M_GLOBAL)>(IN, W, IN ? g.resf_l : g.resf_g);
  const int nx = F.nx, ny = F.ny, ncx = C.nx, ncy = C.ny, rs = F.rs;
  const int ist = g.nxa == 1 ? 2 : 1, ifn = g.nxb == 1 ? nx - 1 : nx;
  const int jst = g.nyc == 1 ? 2 : 1, jfn = g.nyd == 1 ? ny - 1 : ny;
  // specified end points are not interpolated from (their value is zero)
  const int io0 = g.nxa == 1 ? 3 : 1, io1 = g.nxb == 1 ? nx - 2 : nx;
  const int jo0 = g.nyc == 1 ? 3 : 1, jo1 = g.nyd == 1 ? ny - 2 : ny;
  const bool xsub = ncx < nx, ysub = ncy < ny;
  auto xpos = [&](int i, int jc) { return 4 * rs * (jc - 1) + (i & 3) * rs + (i >> 2); };
  {
    const int np = ncy * C.rs;
    const Fd5 f = fd5(C.rs), fp = fd5(np);
    for (int t = tid; t < 4 * np; t += nt) {
      int ic, jc;
      if (!slot5(C, t, np, fp, f, ic, jc)) continue;
      if (!xsub) {
        X.put(xpos(ic, jc), phic.get(pos5(C, ic, jc)));
        continue;
      }
      auto odd = [&](int k) {
        const double x = phic.get(pos5(C, (k + 1) >> 1, jc));
        return (k >= io0 && k <= io1) ? x : 0.0;
      };
      const int i = 2 * ic;
      X.put(xpos(i - 1, jc), odd(i - 1));
      if (ic < ncx) {
        const Tap5 p = tap5(i, nx, ncx >= 4, g.nxa == 0);
        X.put(xpos(i, jc), interp5(p.kind, odd(p.a), odd(p.b), odd(p.c), odd(p.d)));
      }
    }
  }
  sync5<WAVE>();
  {
    const int np = ny * rs;
    const Fd5 f = fd5(rs), fp = fd5(np);
    for (int t0 = tid; t0 < 4 * np; t0 += U * nt) {
      double o[U][5];
      int q[U], kind[U];
      bool in[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = t0 + u * nt;
        int i, j;
        in[u] = slot5(F, t < 4 * np ? t : 0, np, fp, f, i, j) && t < 4 * np && i >= ist && i <= ifn && j >= jst && j <= jfn;
        if (!in[u]) {
          i = ist;
          j = jst;
        }
        q[u] = pos5(F, i, j);
        o[u][4] = phi.get(q[u]);
        const int base = (i & 3) * rs + (i >> 2);
        auto row = [&](int k) {
          const double y = X.get(4 * rs * ((k - 1) >> 1) + base);
          return (k >= jo0 && k <= jo1) ? y : 0.0;
        };
        if (!ysub) {
          kind[u] = 0;
          o[u][0] = o[u][1] = o[u][2] = o[u][3] = X.get(4 * rs * (j - 1) + base);
        } else {
          // an odd row is the coarse row itself: all four operands are it
          const bool od = j & 1;
          const Tap5 p = tap5(od ? 4 : j, ny, ncy >= 4, g.nyc == 0);
          kind[u] = od ? 0 : p.kind;
          o[u][0] = row(od ? j : p.a);
          o[u][1] = row(od ? j : p.b);
          o[u][2] = row(od ? j : p.c);
          o[u][3] = row(od ? j : p.d);
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int k = 0; k < 5; ++k) keep(o[u][k]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (in[u]) {
          const double v = kind[u] == 0 ? o[u][0] : interp5(kind[u], o[u][0], o[u][1], o[u][2], o[u][3]);
          phi.put(q[u], add ? o[u][4] + v : v);
        }
    }
  }
  sync5<WAVE>();
  const int ni = ifn - ist + 1;
  if (g.nyc == 0) {
    for (int t = tid; t < ni; t += nt) {
      const int i = ist + t;
      phi.put(pos5(F, i, 0), phi.get(pos5(F, i, ny - 1)));
      phi.put(pos5(F, i, ny + 1), phi.get(pos5(F, i, 2)));
    }
    sync5<WAVE>();
  }
  if (g.nxa == 0) {
    const bool coarse_rows = !add && ysub;
    const int r0 = coarse_rows ? jo0 : jst, r1 = coarse_rows ? jo1 : jfn, st = coarse_rows ? 2 : 1;
    for (int j = r0 + st * tid; j <= r1; j += st * nt) {
      phi.put(pos5(F, 0, j), phi.get(pos5(F, nx - 1, j)));
      phi.put(pos5(F, nx + 1, j), phi.get(pos5(F, 2, j)));
    }
    sync5<WAVE>();
  }
}

// (inlined: called, its arguments and with them every level's sizes would be
// per-lane values, and the addressing per-lane multiplications)
__device__ __forceinline__ void run_program5(const Mg5& g, double* W, const int* ops, int n) {
  for (int k = 0; k < n; ++k) {
    const int step = __builtin_amdgcn_readfirstlane(ops[k]);
    const int op = (step >> 8) & 0xff, l = step & 0xff, cnt = step >> 16;
    const Lev5& L = g.lev[l];
    if (op == OP5_RELAX) {
      if (L.st == ST_WAVE) {
        if (threadIdx.x < 64) relax_wave5(g, L, cnt);
      } else if (L.st == ST_LDS) {
        relax_block5<ST_LDS>(g, L, W, cnt);
      } else if (L.st == ST_PHI) {
        relax_block5<ST_PHI>(g, L, W, cnt);
      } else {
        relax_block5<ST_GLOBAL>(g, L, W, cnt);
      }
    } else if (op == OP5_RESTRICT) {
      if (L.st == ST_WAVE)
        restrict5<ST_WAVE>(g, L, g.lev[l - 1], W);
      else if (L.st == ST_LDS)
        restrict5<ST_LDS>(g, L, g.lev[l - 1], W);
      else if (L.st == ST_PHI)
        restrict5<ST_PHI>(g, L, g.lev[l - 1], W);
      else
        restrict5<ST_GLOBAL>(g, L, g.lev[l - 1], W);
    } else {
      const Lev5& F = g.lev[l + 1];
      if (F.st == ST_WAVE)
        correct5<ST_WAVE>(g, L, F, W, op == OP5_CORRECT);
      else if (F.st == ST_LDS)
        correct5<ST_LDS>(g, L, F, W, op == OP5_CORRECT);
      else if (F.st == ST_PHI)
        correct5<ST_PHI>(g, L, F, W, op == OP5_CORRECT);
      else
        correct5<ST_GLOBAL>(g, L, F, W, op == OP5_CORRECT);
    }
  }
}

template <int NTMAX>
__global__ void __launch_bounds__(NTMAX) k_mg5_solve(const Mg5* __restrict__ gp, double* __restrict__ ws,
                                                    const double* __restrict__ rhs_tmp, double* __restrict__ phi_out,
                                                    const double* __restrict__ kx2, int* __restrict__ cycles, size_t plane,
                                                    int iguess) {
  const Mg5& g = *gp;
  const int s = blockIdx.x;
  double* W = ws + (size_t)s * g.ws;
  const double k2 = kx2[s];
  const int nfx = g.nfx, nfy = g.nfy, ng = g.ngrid;
  const double* rt = rhs_tmp + (size_t)s * plane;
  double* pout = phi_out + (size_t)s * plane;
  const int TID = threadIdx.x, NT = blockDim.x;
  auto phi_at = [&](const Lev5& L, int p) -> double& { return L.st >= ST_PHI ? lds5[L.phi + p] : W[L.phi + p]; };
  auto rhs_at = [&](const Lev5& L, int p) -> double& { return L.st >= ST_LDS ? lds5[L.rhs + p] : W[L.rhs + p]; };
  // per-solve c9 = ((ce - s9) + corr9), ce = -kx2 J (1 where there is no
  // point); LDS levels also take their coefficients and 1/c9
  for (int l = 1; l <= ng; ++l) {
    const Lev5& L = g.lev[l];
    const size_t e = L.e4;
    for (int t = TID; t < L.e4; t += NT) {
      const double s9 = L.c[4 * e + t], c9 = ((-(k2 * L.c[6 * e + t])) - s9) + L.c[5 * e + t];
      phi_at(L, t) = 0.0;
      rhs_at(L, t) = 0.0;
      if (L.st >= ST_LDS) {
        double* c = lds5 + L.cf + t;
        for (int q = 0; q < 4; ++q) c[q * L.e4] = L.c[q * e + t];
        c[4 * L.e4] = c9;
        c[5 * L.e4] = 1.0 / c9;
      } else {
        W[L.c9 + t] = c9;
      }
    }
  }
  {
    int* tab = reinterpret_cast<int*>(lds5 + g.tab);
    for (int t = TID; t < g.tab_n; t += NT) tab[t] = g.tabg[t];
  }
  __syncthreads();
  // swk2 + phi_bc: phi = initial guess (0 unless iguess), rhs = -RHS_TMP
  {
    const Lev5& L = g.lev[ng];
    for (int t = TID; t < nfx * nfy; t += NT) {
      const int j = 1 + t / nfx, i = 1 + t - (j - 1) * nfx, p = pos5(L, i, j);
      if (iguess) phi_at(L, p) = pout[t];
      rhs_at(L, p) = -rt[t];
    }
  }
  __syncthreads();
  // adjmd2cr: specified boundaries take phi
  auto adjust = [&](int l) {
    const Lev5& L = g.lev[l];
    for (int t = TID; t < L.nx * L.ny; t += NT) {
      const int j = 1 + t / L.nx, i = 1 + t - (j - 1) * L.nx;
      if ((g.nxa == 1 && i == 1) || (g.nxb == 1 && i == L.nx) || (g.nyc == 1 && j == 1) || (g.nyd == 1 && j == L.ny))
        rhs_at(L, pos5(L, i, j)) = phi_at(L, pos5(L, i, j));
    }
    __syncthreads();
  };
  if (!iguess) {
    // trsfc2 down to every level (injection of phi, which is zero, and rhs)
    for (int l = ng - 1; l >= 1; --l) {
      const Lev5 &F = g.lev[l + 1], &C = g.lev[l];
      for (int t = TID; t < C.nx * C.ny; t += NT) {
        const int jc = 1 + t / C.nx, ic = 1 + t - (jc - 1) * C.nx;
        const int i = (C.nx < F.nx) ? ic + ic - 1 : ic, j = (C.ny < F.ny) ? jc + jc - 1 : jc;
        rhs_at(C, pos5(C, ic, jc)) = rhs_at(F, pos5(F, i, j));
      }
      __syncthreads();
    }
    for (int l = 1; l <= ng; ++l) adjust(l);
  } else {
    adjust(ng);
  }
  // program 0: the full multigrid start (skipped with an initial guess);
  // programs 1..maxcy: W cycles from the finest level with the relmax test
  // (mud2cr1 :238-337)
  double* red = lds5 + g.red;
  const Lev5& L = g.lev[ng];
  const int np = L.ny * L.rs;
  const Fd5 fp = fd5(np), fr = fd5(L.rs);
  int itero = 0;
  bool done = false;
  for (int iter = iguess ? 1 : 0; iter <= g.maxcy && !done; ++iter) {
    __syncthreads();
    run_program5(g, W, iter == 0 ? g.ops : g.ops + g.nops_fmg, iter == 0 ? g.nops_fmg : g.nops_w);
    __syncthreads();
    if (iter == 0) {
      // the caller's phi is the relmax reference of the first cycle: zero
      for (int t = TID; t < nfx * nfy; t += NT) pout[t] = 0.0;
      continue;
    }
    itero = iter;
    if (g.tolmax > 0.0) {
      double rel = 0.0, pm = 0.0;
      for (int t = TID; t < 4 * np; t += NT) {
        int i, j;
        if (!slot5(L, t, np, fp, fr, i, j)) continue;
        const int q = (i - 1) + nfx * (j - 1);
        const double w = phi_at(L, pos5(L, i, j));
        pm = fmax(pm, fabs(w));
        rel = fmax(rel, fabs(w - pout[q]));
        pout[q] = w;
      }
      for (int o = 32; o > 0; o >>= 1) {
        pm = fmax(pm, __shfl_xor(pm, o, 64));
        rel = fmax(rel, __shfl_xor(rel, o, 64));
      }
      if ((TID & 63) == 0) {
        red[TID >> 6] = rel;
        red[16 + (TID >> 6)] = pm;
      }
      __syncthreads();
      double relmax = 0.0, phmax = 0.0;
      for (int w = 0; w < (NT >> 6); ++w) {
        relmax = fmax(relmax, red[w]);
        phmax = fmax(phmax, red[16 + w]);
      }
      __syncthreads();
      if (phmax > 0.0) relmax = relmax / phmax;
      if (relmax <= g.tolmax) done = true;
    }
  }
  __syncthreads();
  if (!done) {
    for (int t = TID; t < 4 * np; t += NT) {
      int i, j;
      if (slot5(L, t, np, fp, fr, i, j)) pout[(i - 1) + nfx * (j - 1)] = phi_at(L, pos5(L, i, j));
    }
  }
  if (TID == 0) cycles[s] = itero;
}

}  // namespace

bool mg5_applies(const std::vector<HostMgLevel>& hl, int ngrid) {
  for (int k = 1; k <= ngrid; ++k) {
    const HostMgLevel& H = hl[k];
    const size_t n = (size_t)H.nx * H.ny;
    if (H.nx < 3 || H.ny < 3) return false;
    for (int c = 1; c < 8; c += 2)
      for (size_t q = 0; q < n; ++q)
        if (H.c[c * n + q] != 0.0) return false;
  }
  return ngrid <= kMaxLev5;
}

int mg5_plan_build(Mg5Plan& mp, const MgPlan& mg, const Dims& d, const std::vector<HostMgLevel>& hl,
                   const std::vector<int>& ops, size_t lds_budget_doubles) {
  Mg5 g;
  std::memset(&g, 0, sizeof(g));
  const int ng = mg.ngrid;
  g.ngrid = ng;
  g.nxa = mg.nxa;
  g.nxb = mg.nxb;
  g.nyc = mg.nyc;
  g.nyd = mg.nyd;
  g.maxcy = mg.maxcy;
  g.tolmax = mg.tolmax;
  g.nfx = d.NZ2;
  g.nfy = d.NY2;
  size_t lo = 0, go = 0, coef = 0, resf_l = 0, resf_g = 0;
  int top = ST_WAVE;  // storage never rises from a level to the next finer one
  const size_t red = 32;
  std::vector<int> tab;
  size_t tabs = 0;  // doubles of the point tables
  for (int k = 1; k <= ng; ++k) {
    Lev5& L = g.lev[k];
    L.nx = hl[k].nx;
    L.ny = hl[k].ny;
    L.rs = (L.nx + 5) >> 2;
    L.cs = (L.ny + 2) * L.rs;
    L.e4 = 4 * L.cs;
    const size_t e = (size_t)L.e4;
    if (top == ST_WAVE) {
      int t[4][64], most = 0;
      for (int q = 0; q < 4; ++q) {
        int m = 0;
        for (int j = 1; j <= L.ny; ++j)
          for (int i = 1; i <= L.nx; ++i)
            if (((i + j) & 3) == ((2 + q) & 3)) {
              if (m < 64) t[q][m] = i | (j << 16);
              ++m;
            }
        for (int u = m; u < 64; ++u) t[q][u] = -1;
        most = std::max(most, m);
      }
      if (most <= 64) {
        L.tab = (int)tab.size();
        tab.insert(tab.end(), &t[0][0], &t[0][0] + 256);
        tabs += 128;
      } else {
        top = ST_LDS;
      }
    }
    // all eight arrays and the restriction's residual, or the correction alone
    if (top >= ST_LDS && lo + 9 * e + red + tabs > lds_budget_doubles) top = ST_PHI;
    if (top == ST_PHI && lo + resf_l + e + red + tabs > lds_budget_doubles) top = ST_GLOBAL;
    L.st = top;
    if (top >= ST_PHI) {
      L.phi = (int)lo;
      lo += e;
    } else {
      L.phi = (int)go;
      go += e;
    }
    if (top >= ST_LDS) {
      L.rhs = (int)lo;
      L.cf = (int)(lo + e);
      L.c9 = (int)(lo + 5 * e);
      lo += 7 * e;
      resf_l = std::max(resf_l, e);
    } else {
      L.rhs = (int)go;
      L.c9 = (int)(go + e);
      go += 2 * e;
      resf_g = std::max(resf_g, e);
    }
    coef += 7 * e;
  }
  g.resf_l = (int)lo;
  lo += resf_l;
  g.red = (int)lo;
  lo += red;
  g.tab = (int)lo;
  g.tab_n = (int)tab.size();
  lo += tab.size() / 2;
  if (lo > lds_budget_doubles) return EKM_ERR_UNSUPPORTED;
  g.resf_g = (int)go;
  go += resf_g;
  go = (go + 31) & ~(size_t)31;
  g.ws = (int)go;
  mp.lds = lo * sizeof(double);
  mp.ws = go;
  // the programs with consecutive relaxations of a level joined
  std::vector<int> o2;
  auto join = [&](int a, int b) {
    const int at = (int)o2.size();
    for (int k = a; k < b; ++k) {
      if (((ops[k] >> 8) & 0xff) == OP5_RELAX && (int)o2.size() > at && (o2.back() & 0xffff) == ops[k])
        o2.back() += 1 << 16;
      else
        o2.push_back((1 << 16) | ops[k]);
    }
    return (int)o2.size() - at;
  };
  g.nops_fmg = join(0, mg.nops_fmg);
  g.nops_w = join(mg.nops_fmg, mg.nops_fmg + mg.nops_w);
  std::vector<double> host(coef, 0.0);
  const size_t desc = (sizeof(Mg5) + 255) & ~(size_t)255, opb = ((o2.size() + tab.size()) * sizeof(int) + 255) & ~(size_t)255;
  EKM_CHECK(hipMalloc((void**)&mp.mem, desc + opb + coef * sizeof(double)));
  double* dc = (double*)(mp.mem + desc + opb);
  size_t off = 0;
  for (int k = 1; k <= ng; ++k) {
    Lev5& L = g.lev[k];
    const HostMgLevel& H = hl[k];
    const size_t n = (size_t)H.nx * H.ny, e = (size_t)L.e4;
    // slots without a point: c9 = ((-0) - (-1)) + 0 = 1
    for (size_t t = 0; t < e; ++t) host[off + 4 * e + t] = -1.0;
    for (int j = 1; j <= L.ny; ++j)
      for (int i = 1; i <= L.nx; ++i) {
        const size_t q = (size_t)(i - 1) + (size_t)L.nx * (j - 1), p = (size_t)pos5(L, i, j);
        for (int c = 0; c < 4; ++c) host[off + c * e + p] = H.c[2 * c * n + q];
        host[off + 4 * e + p] = H.s9[q];
        host[off + 5 * e + p] = H.corr9[q];
        host[off + 6 * e + p] = H.jl[q];
      }
    L.c = dc + off;
    off += 7 * e;
  }
  g.ops = (const int*)(mp.mem + desc);
  g.tabg = g.ops + o2.size();
  o2.insert(o2.end(), tab.begin(), tab.end());
  EKM_CHECK(hipMemcpy(mp.mem, &g, sizeof(g), hipMemcpyHostToDevice));
  EKM_CHECK(hipMemcpy(mp.mem + desc, o2.data(), o2.size() * sizeof(int), hipMemcpyHostToDevice));
  EKM_CHECK(hipMemcpy(dc, host.data(), coef * sizeof(double), hipMemcpyHostToDevice));
  if (mp.lds > 65536)
    for (const void* k : {(const void*)k_mg5_solve<512>, (const void*)k_mg5_solve<1024>})
      EKM_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mp.lds));
  mp.on = 1;
  return EKM_OK;
}

int mg5_solve(const MgPlan& mg, const Dims& d, int nsolve, int iguess, hipStream_t st) {
  // up to 512 threads a lane may use 256 registers (LDS allows one block per CU)
  if (mg.block <= 512)
    hipLaunchKernelGGL(k_mg5_solve<512>, dim3(nsolve), dim3(mg.block), mg.five.lds, st, (const Mg5*)mg.five.mem, mg.ws,
                       (const double*)mg.rhs, mg.phi, (const double*)mg.kx2, mg.cycles, d.plane, iguess);
  else
    hipLaunchKernelGGL(k_mg5_solve<1024>, dim3(nsolve), dim3(mg.block), mg.five.lds, st, (const Mg5*)mg.five.mem, mg.ws,
                       (const double*)mg.rhs, mg.phi, (const double*)mg.kx2, mg.cycles, d.plane, iguess);
  EKM_CHECK(hipGetLastError());
  return EKM_OK;
}
