// Closing part of the turbulence stage of met_num (met_num.f90:697-930) on
// gfx950: the line-implicit phase of the two transport equations
// (impli2_eqt_3d), the limiters of at_cutke (met_cut, met_cutsa) and the
// eddy viscosity of the SA and k-omega models (met_samut, met_kocmut).
#include "common.hpp"

#include <algorithm>
#include <utility>
#include <vector>

using namespace codens;

#define REAL3(b)  \
  int c[3];       \
  if (!line_cell((b), xcd_linear(), c)) return;

// Workspace of the implicit phase: the half normal velocities uf and the
// coefficients ce of the faces of the three directions, the increments dw6,
// dw7, the right-hand sides r6, r7 of the current sweep's lines (overwritten by
// the eliminated ones), and of the lines of each direction the coefficient lc,
// the elimination coefficients al and the denominators den.  Entries of the i
// lines are line-major, all others at the block-local index m.
struct ImpliWs {
  double *uf, *ce, *dw6, *dw7, *r6, *r7, *lc, *al, *den;
  double *cd;  // the cells' diagonal, read before dw6 is written
};

constexpr int IMPLI_PLANES = 19;

// the planes of nnn of a block's workspace starting at ws
__host__ __device__ inline ImpliWs impli_ws(double *ws, long nnn) {
  return ImpliWs{ws,           ws + 3 * nnn,  ws + 6 * nnn,  ws + 7 * nnn,  ws + 8 * nnn,
                 ws + 9 * nnn, ws + 10 * nnn, ws + 13 * nnn, ws + 16 * nnn, ws + 6 * nnn};
}

// impli2_eqt_3d.f90:113-208: coefficients of every face i1..i2 (resp. j, k)
// of the real transverse range; the launch covers the cells up to i2, j2, k2.
// rv = (mu + mut/cmt)/rho of the two cells (zero of a ghost, as in the
// reference's cleared array) is formed here, its divisions and the velocities'
// sharing one reciprocal per cell.  All loads first and no idle lanes: its 22
// planes move at 4.7 TB/s, 32 us on 130 x 96 x 66; with tiles of 64 x 4, the
// loads between the divisions and behind the neighbours' branches it took 42
// us, and a pass of its own for rv and one that cleared the work arrays 29 more.
__host__ __device__ __forceinline__ Blk upto_high(Blk b) {
  b.i2++;
  b.j2++;
  b.k2++;
  return b;
}
__device__ __forceinline__ void faces_body(const Blk &b, unsigned wg, const double *__restrict__ v, long ldv,
                                           const double *__restrict__ mu, const double *__restrict__ mut, double cmt,
                                           const double *__restrict__ sn, const double *__restrict__ vol,
                                           const ImpliWs &w) {
  int c[3];
  if (!line_cell(upto_high(b), wg, c)) return;
  const int high = (c[0] == b.i2) + (c[1] == b.j2) + (c[2] == b.k2);
  if (high > 1) return;
  const long n = b.idx(c[0], c[1], c[2]), m = n - b.npc, n1 = b.idx(b.i1, b.j1, b.k1);
  // the cell and its low neighbours: rho, momentum, mu, mut, vol (a ghost has
  // no mu and mut: those of the first cell are loaded and not used)
  double z[4][7], s[3][3];
#pragma unroll
  for (int x = 0; x < 4; x++) {
    const long nx = x ? n - b.inc(x - 1) : n;
#pragma unroll
    for (int e = 0; e < 4; e++) z[x][e] = v[e * ldv + nx];
    const int d = x - 1;
    const long nr = (x ? c[d] > b.lo(d) && (!high || c[d] == b.hi(d)) : !high) ? nx : n1;
    z[x][4] = mu[nr];
    z[x][5] = mut[nr];
    z[x][6] = vol[nx];
  }
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int e = 0; e < 3; e++) s[d][e] = snv(sn, b.nnn, m, d, e);
  loads_issued();
  const double yc = rcp64(cmt);
  auto cell = [&](const double z[7], bool real, double q[4]) {
    const double y = rcp64(z[0]);
#pragma unroll
    for (int e = 0; e < 3; e++) q[e] = div_rcp(z[1 + e], z[0], y);
    const double rv = div_rcp(z[4] + div_rcp(z[5], cmt, yc), z[0], y);
    q[3] = real ? rv : 0.;
  };
  double q[4];
  cell(z[0], !high, q);
#pragma unroll
  for (int d = 0; d < 3; d++) {
    bool ok = true;
#pragma unroll
    for (int x = 0; x < 3; x++) ok = ok && c[x] <= b.hi(x) - (x == d ? 0 : 1);
    const double s1 = s[d][0], s2 = s[d][1], s3 = s[d][2];
    double cnds = s1 * s1 + s2 * s2 + s3 * s3;
    double l[4];
    cell(z[d + 1], c[d] > b.lo(d), l);
    double uu = 0.5 * (q[0] + l[0]), vv = 0.5 * (q[1] + l[1]), ww = 0.5 * (q[2] + l[2]);
    double uf = 0.5 * (uu * s1 + vv * s2 + ww * s3);
    const double ce = fabs(uf) + (q[3] + l[3]) * cnds / (z[0][6] + z[d + 1][6]);
    if (ok) {
      w.uf[d * b.nnn + m] = uf;
      w.ce[d * b.nnn + m] = ce;
    }
  }
}

__global__ void __launch_bounds__(256) k_impli2_faces(Blk b, const double *__restrict__ v, long ldv,
                                                         const double *__restrict__ mu,
                                                         const double *__restrict__ mut, double cmt,
                                                         const double *__restrict__ sn,
                                                         const double *__restrict__ vol, ImpliWs w) {
  faces_body(b, xcd_linear(), v, ldv, mu, mut, cmt, sn, vol, w);
}

// One sweep along direction d (impli2_eqt_3d.f90:238-275, 292-329, 346-383)
// solves a a-b-c system per grid line for both equations.  The coefficients do
// not change between sweeps, so the part of the elimination that is theirs
// (al, den) is done once for all directions (k_impli2_elim), next to each
// other in one launch as each is a serial chain per line.  A sweep is then
//
// k_impli2_rhs, over all real cells: the right-hand sides, whose transverse
// terms read the previous sweep's increments only (those of ghosts are zero;
// before the first sweep all are, and k_impli2_diag writes the right-hand
// sides, -u).
//
// k_impli2_line, one lane per line and equation: the elimination of the
// right-hand side from the high end of the line (recursion values zero beyond
// the last real cell, as the reference's zeroed arrays give) and the
// substitution from the low end, which writes the increments, or at the last
// sweep adds them to v (impli2_eqt_3d.f90:406-416).
//
// Lines of j and k are neighbours in i, so their entries lie at the cells' own
// index.  The lines of i are kept line-major, entry (i - i1) * nl + line with
// the line index (j - j1) + (k - k1) * nj, so that the recursions read
// consecutive lines at consecutive addresses; the kernels over cells transpose
// tiles of 16 x 16 cells through LDS for them, so that both sides move
// 128-byte runs.
//
// On 130 x 96 x 66 the elimination of the coefficients takes 25 us (its 18
// planes move at 4.8 TB/s), a sweep's right-hand sides 13 us (5 TB/s) and its
// recursions 19 to 25 us (0.15 to 0.3 us per step of a line, two equations of
// 32 lines per wave, as few lines as there are then spread over more SIMDs);
// with the coefficients formed and eliminated again in every sweep, one lane
// for both equations and the loads a batch of eight steps ahead the two took
// 20 and 40 us.  The whole phase 454 -> 280 us.
constexpr int RT = 16;

// writes val[e] of cell c = (i, j, k) of this thread's tile to the line-major
// arrays out[e] (i lines)
template <int N>
__device__ __forceinline__ void put_i_lines(const Blk &b, dim3 xb, const double val[N], double *const out[N]) {
  __shared__ double sh[N][RT][RT + 1];
  const int tx = threadIdx.x % RT, ty = threadIdx.x / RT;
#pragma unroll
  for (int e = 0; e < N; e++) sh[e][ty][tx] = val[e];
  __syncthreads();
  const long nj = b.j2 - b.j1, nl = nj * (b.k2 - b.k1);
  const int i = b.i1 + xb.x * RT + ty, j = b.j1 + xb.y * RT + tx;
  if (i < b.i2 && j < b.j2) {
    const long L = (long)(i - b.i1) * nl + (j - b.j1) + (long)xb.z * nj;
#pragma unroll
    for (int e = 0; e < N; e++) out[e][L] = sh[e][tx][ty];
  }
}

// impli2_eqt_3d.f90:113-122, 210-220: the cells' diagonal, the coefficients a,
// b, c of the i lines (a and b where k_impli2_elim leaves al and den) and the
// right-hand sides of the first sweep
__device__ __forceinline__ void diag_body(const Blk &b, dim3 xb, const double *__restrict__ dt,
                                          const double *__restrict__ vol, const double *__restrict__ cfke,
                                          const double *__restrict__ u, long ldv, const ImpliWs &w) {
  const int i = b.i1 + xb.x * RT + threadIdx.x % RT, j = b.j1 + xb.y * RT + threadIdx.x / RT;
  double val[5] = {0., 0., 0., 0., 0.};
  if (i < b.i2 && j < b.j2) {
    const long n = b.idx(i, j, b.k1 + xb.z), m = n - b.npc, nnn = b.nnn;
    const double *__restrict__ ce = w.ce, *__restrict__ uf = w.uf;
    const double c0 = ce[m], c1 = ce[m + 1], u0 = uf[m], u1 = uf[m + 1];
    double cd = vol[n] / dt[n] + cfke[n] * vol[n];
    cd = cd + c0 + c1 + ce[nnn + m] + ce[nnn + m + b.nid] + ce[2 * nnn + m] + ce[2 * nnn + m + b.nijd];
    w.cd[m] = cd;
    val[0] = c0 + u0;
    val[1] = cd + u1 - u0;
    val[2] = -c1 + u1;
    val[3] = -u[5 * ldv + n];
    val[4] = -u[6 * ldv + n];
  }
  double *const out[5] = {w.al, w.den, w.lc, w.r6, w.r7};
  put_i_lines<5>(b, xb, val, out);
}

__global__ void __launch_bounds__(RT *RT) k_impli2_diag(Blk b, const double *__restrict__ dt,
                                                        const double *__restrict__ vol,
                                                        const double *__restrict__ cfke,
                                                        const double *__restrict__ u, long ldv, ImpliWs w) {
  diag_body(b, xcd_block(), dt, vol, cfke, u, ldv, w);
}

__device__ __forceinline__ void rhs_body(const Blk &b, dim3 xb, int d, const double *__restrict__ u, long ldv,
                                         const ImpliWs &w) {
  const int p = d == 0 ? 1 : 0, q = d == 2 ? 1 : 2;
  int c[3];
  c[0] = b.i1 + xb.x * RT + threadIdx.x % RT;
  c[1] = b.j1 + xb.y * RT + threadIdx.x / RT;
  c[2] = b.k1 + xb.z;
  const bool in = c[0] < b.i2 && c[1] < b.j2;
  double val[2] = {0., 0.};
  if (in) {
    const long ip = b.inc(p), iq = b.inc(q), nnn = b.nnn;
    const long n = b.idx(c[0], c[1], c[2]), m = n - b.npc;
    const double *__restrict__ uP = w.uf + p * nnn, *__restrict__ uQ = w.uf + q * nnn;
    const double *__restrict__ cP = w.ce + p * nnn, *__restrict__ cQ = w.ce + q * nnn;
    const bool lp = c[p] > b.lo(p), hp = c[p] + 1 < b.hi(p), lq = c[q] > b.lo(q), hq = c[q] + 1 < b.hi(q);
    double td = -uP[m + ip] + uP[m] - uQ[m + iq] + uQ[m];
    double tpp = cP[m + ip] - uP[m + ip], tmp_ = cP[m] + uP[m];
    double tpq = cQ[m + iq] - uQ[m + iq], tmq = cQ[m] + uQ[m];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const double *__restrict__ dw = e == 0 ? w.dw6 : w.dw7;
      const double wl = lp ? dw[m - ip] : 0., wh = hp ? dw[m + ip] : 0.;
      const double ql = lq ? dw[m - iq] : 0., qh = hq ? dw[m + iq] : 0.;
      val[e] = -u[(5 + e) * ldv + n] + td * dw[m] + tmp_ * wl + tpp * wh + tmq * ql + tpq * qh;
    }
    if (d != 0) {
      w.r6[m] = val[0];
      w.r7[m] = val[1];
    }
  }
  if (d == 0) {
    double *const out[2] = {w.r6, w.r7};
    put_i_lines<2>(b, xb, val, out);
  }
}

__global__ void __launch_bounds__(RT *RT) k_impli2_rhs(Blk b, int d, const double *__restrict__ u, long ldv,
                                                        ImpliWs w) {
  rhs_body(b, xcd_block(), d, u, ldv, w);
}

// Line t of direction d: its length, the cell's index of its first entry and
// the step from one to the next, and the same for the arrays of the lines.
struct Line {
  int nd;
  long m0, inc, at, step;
  bool ok;
};
__device__ __forceinline__ Line line_of(const Blk &b, int d, long t) {
  const int p = d == 0 ? 1 : 0, q = d == 2 ? 1 : 2;
  const long np_ = b.hi(p) - b.lo(p), nl = np_ * (b.hi(q) - b.lo(q));
  Line l;
  l.ok = t < nl;
  int c[3];
  c[p] = b.lo(p) + (int)(t % np_);
  c[q] = b.lo(q) + (int)(t / np_);
  c[d] = b.lo(d);
  l.nd = b.hi(d) - b.lo(d);
  l.m0 = b.idx(c[0], c[1], c[2]) - b.npc;
  l.inc = b.inc(d);
  l.at = d == 0 ? t : l.m0;
  l.step = d == 0 ? nl : l.inc;
  return l;
}

// The recursions run at the latency of their loads unless those are far ahead:
// each keeps the operands of its next LU steps in registers and loads a step's
// operands where it has used those of the step LU before.  LU steps' loads
// and stores are near the 63 that a wave can have in flight.
constexpr int LU = 15;

// The coefficients' elimination from the high end of a line.
template <bool I>
__device__ __forceinline__ void elim_body(const Blk &b, int d, long t, const ImpliWs &w) {
  const Line l = line_of(b, d, t);
  if (!l.ok) return;
  const long nnn = b.nnn;
  double *const al = w.al + d * nnn + l.at, *const den = w.den + d * nnn + l.at, *const lc = w.lc + d * nnn + l.at;
  const double *const uD = w.uf + d * nnn + l.m0, *const cD = w.ce + d * nnn + l.m0, *const cd = w.cd + l.m0;
  double al1 = 0., uh = 0., ch = 0.;  // al, uD and cD of the next cell up the line
  if (!I) {
    uh = uD[l.nd * l.inc];
    ch = cD[l.nd * l.inc];
  }
  double x[LU][3];
  auto load = [&](double z[3], int a) {
    const long i = max(a, 0);
    if (I) {
      z[0] = al[i * l.step]; z[1] = den[i * l.step]; z[2] = lc[i * l.step];
    } else {
      z[0] = uD[i * l.inc]; z[1] = cD[i * l.inc]; z[2] = cd[i * l.inc];
    }
  };
  auto run = [&](const double z[3], int a) {
    const long i = a * l.step;
    double A = z[0], B = z[1], C = z[2];
    if (!I) {
      A = z[1] + z[0];
      B = z[2] + uh - z[0];
      C = -ch + uh;
      uh = z[0];
      ch = z[1];
      lc[i] = C;
    }
    const double dn = B + C * al1;
    al1 = div_rcp(A, dn, rcp64(dn));
    al[i] = al1;
    den[i] = dn;
  };
#pragma unroll
  for (int s = 0; s < LU; s++) load(x[s], l.nd - 1 - s);
  int a = l.nd - 1;
  for (; a >= LU - 1; a -= LU) {
#pragma unroll
    for (int s = 0; s < LU; s++) {
      run(x[s], a - s);
      load(x[s], a - s - LU);
    }
  }
#pragma unroll
  for (int s = 0; s < LU - 1; s++)
    if (a - s >= 0) run(x[s], a - s);
}

__host__ __device__ inline long n_lines(const Blk &b, int d) {
  const int p = d == 0 ? 1 : 0, q = d == 2 ? 1 : 2;
  return (long)(b.hi(p) - b.lo(p)) * (b.hi(q) - b.lo(q));
}

__global__ void __launch_bounds__(64) k_impli2_elim(Blk b, ImpliWs w) {
  const int d = blockIdx.y;
  if (d == 0) elim_body<true>(b, 0, blockIdx.x * 64L + threadIdx.x, w);
  else elim_body<false>(b, d, blockIdx.x * 64L + threadIdx.x, w);
}

// The two recursions of a line for one equation: lanes 0..31 of a wave are 32
// lines of the first, lanes 32..63 of the second.
constexpr int LINES = 32;  // lines per wave
template <bool LAST>
__device__ __forceinline__ void line_body(const Blk &b, int d, long t0, double *v, long ldv, const ImpliWs &w) {
  const int eq = threadIdx.x / LINES;
  const Line l = line_of(b, d, t0 + threadIdx.x % LINES);
  if (!l.ok) return;
  const long nnn = b.nnn;
  double *const R = (eq ? w.r7 : w.r6) + l.at;
  const double *const al = w.al + d * nnn + l.at, *const den = w.den + d * nnn + l.at;
  const double *const lc = w.lc + d * nnn + l.at;
  {
    double x[LU][3], b1 = 0.;
    auto load = [&](double z[3], int a) {
      const long j = max(a, 0) * l.step;
      z[0] = R[j]; z[1] = den[j]; z[2] = lc[j];
    };
    auto run = [&](const double z[3], int a) {
      b1 = div_rcp(z[0] - z[2] * b1, z[1], rcp64(z[1]));
      R[a * l.step] = b1;
    };
#pragma unroll
    for (int s = 0; s < LU; s++) load(x[s], l.nd - 1 - s);
    int a = l.nd - 1;
    for (; a >= LU - 1; a -= LU) {
#pragma unroll
      for (int s = 0; s < LU; s++) {
        run(x[s], a - s);
        load(x[s], a - s - LU);
      }
    }
#pragma unroll
    for (int s = 0; s < LU - 1; s++)
      if (a - s >= 0) run(x[s], a - s);
  }
  // substitution from the low end (the same lane wrote R above, so its own
  // loads see those values)
  double *const out = LAST ? v + (5 + eq) * ldv + b.npc + l.m0 : (eq ? w.dw7 : w.dw6) + l.m0;
  double x[LU][3], wl = 0.;  // wl: increment of the cell below, zero of the ghost
  auto load = [&](double z[3], int a) {
    const long i = min(a, l.nd - 1);
    z[0] = al[i * l.step]; z[1] = R[i * l.step];
    if (LAST) z[2] = out[i * l.inc];
  };
  auto run = [&](const double z[3], int a) {
    wl = z[0] * wl + z[1];
    out[a * l.inc] = LAST ? z[2] + wl : wl;
  };
#pragma unroll
  for (int s = 0; s < LU; s++) load(x[s], s);
  int a = 0;
  for (; a + LU <= l.nd; a += LU) {
#pragma unroll
    for (int s = 0; s < LU; s++) {
      run(x[s], a + s);
      load(x[s], a + s + LU);
    }
  }
#pragma unroll
  for (int s = 0; s < LU - 1; s++)
    if (a + s < l.nd) run(x[s], a + s);
}

template <bool LAST>
__global__ void __launch_bounds__(64) k_impli2_line(Blk b, int d, double *v, long ldv, ImpliWs w) {
  line_body<LAST>(b, d, blockIdx.x * (long)LINES, v, ldv, w);
}

extern "C" int codens_impli2_eqt_3d(const codens_block *cb, const double *u, int64_t ldv, const double *dt,
                                    double *v, const double *mu, const double *mut, const double *cfke,
                                    const double *sn, const double *vol, double cmt, void *stream) {
  int rc = codens_check_block(cb, "codens_impli2_eqt_3d");
  if (rc) return rc;
  if (!u || !dt || !v || !mu || !mut || !cfke || !sn || !vol || !(cmt > 0.)) {
    codens_set_error("codens_impli2_eqt_3d: invalid argument");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  hipStream_t st = (hipStream_t)stream;
  double *ws = (double *)codens_workspace(sizeof(double) * IMPLI_PLANES * b.nnn, 3);
  if (!ws) {
    codens_set_error("codens_impli2_eqt_3d: workspace allocation failed");
    return CODENS_EHIP;
  }
  ImpliWs w = impli_ws(ws, b.nnn);
  CodensTimed _tm("impli2_eqt_3d", st);
  hipLaunchKernelGGL(k_impli2_faces, cell_line(upto_high(b)), dim3(256), 0, st, b, v, (long)ldv, mu, mut, cmt, sn, vol, w);
  dim3 gr((b.i2 - b.i1 + RT - 1) / RT, (b.j2 - b.j1 + RT - 1) / RT, b.k2 - b.k1);
  hipLaunchKernelGGL(k_impli2_diag, gr, dim3(RT * RT), 0, st, b, dt, vol, cfke, u, (long)ldv, w);
  const long most = std::max(n_lines(b, 0), std::max(n_lines(b, 1), n_lines(b, 2)));
  hipLaunchKernelGGL(k_impli2_elim, dim3((unsigned)((most + 63) / 64), 3), dim3(64), 0, st, b, w);
  for (int s = 0; s < 6; s++) {
    const int d = s / 2;
    if (s > 0) hipLaunchKernelGGL(k_impli2_rhs, gr, dim3(RT * RT), 0, st, b, d, u, (long)ldv, w);
    hipLaunchKernelGGL(s == 5 ? k_impli2_line<true> : k_impli2_line<false>,
                       dim3((unsigned)((n_lines(b, d) + LINES - 1) / LINES)), dim3(64), 0, st, b, d, v, (long)ldv, w);
  }
  return codens_check_launch("codens_impli2_eqt_3d");
}

// ---------------------------------------------------------------------------
// impli2_eqt_3d for all blocks of a layout: each pass of the phase (faces,
// diagonal, coefficients' elimination, and per sweep the right-hand sides and
// the line recursions) is one flattened launch over every block, with a device
// table of the blocks' extents and first workgroups per pass.  Block l's
// workspace starts at IMPLI_PLANES npc.  The line recursion is a serial chain
// per line, so a launch takes about the time of its longest line: one launch
// over the lines of all blocks replaces one per block.
enum { TB_FACE, TB_RHS, TB_ELIM0, TB_ELIM1, TB_ELIM2, TB_LINE0, TB_LINE1, TB_LINE2, TB_N };

struct TurbEnt {
  Blk b;
  unsigned start[TB_N];         // first workgroup of this block, per pass
  unsigned gx[TB_N], gy[TB_N];  // this block's grid, per pass
};

__global__ void __launch_bounds__(256) k_impli2_faces_batch(const TurbEnt *__restrict__ tab, int nb,
                                                               const double *__restrict__ v, long ldv,
                                                               const double *__restrict__ mu,
                                                               const double *__restrict__ mut, double cmt,
                                                               const double *__restrict__ sn_all,
                                                               const double *__restrict__ vol, double *ws) {
  const unsigned wg = xcd_grouped(64);
  const TurbEnt &E = tab[tab_find(tab, nb, TB_FACE, wg)];
  const Blk b = uniform_blk(E.b);
  faces_body(b, wg - E.start[TB_FACE], v, ldv, mu, mut, cmt, sn_all + 9 * b.npc, vol,
             impli_ws(ws + IMPLI_PLANES * b.npc, b.nnn));
}

__global__ void __launch_bounds__(RT *RT) k_impli2_diag_batch(const TurbEnt *__restrict__ tab, int nb,
                                                              const double *__restrict__ dt,
                                                              const double *__restrict__ vol,
                                                              const double *__restrict__ cfke,
                                                              const double *__restrict__ u, long ldv, double *ws) {
  const unsigned wg = xcd_grouped(64);
  const TurbEnt &E = tab[tab_find(tab, nb, TB_RHS, wg)];
  const Blk b = uniform_blk(E.b);
  diag_body(b, tab_tile(E, TB_RHS, wg), dt, vol, cfke, u, ldv, impli_ws(ws + IMPLI_PLANES * b.npc, b.nnn));
}

__global__ void __launch_bounds__(64) k_impli2_elim_batch(const TurbEnt *__restrict__ tab, int nb, double *ws) {
  const int d = blockIdx.y;
  const unsigned wg = blockIdx.x;
  const TurbEnt &L = tab[nb - 1];
  if (wg >= L.start[TB_ELIM0 + d] + L.gx[TB_ELIM0 + d]) return;  // the grid is that of the direction with most
  const TurbEnt &E = tab[tab_find(tab, nb, TB_ELIM0 + d, wg)];
  const Blk b = uniform_blk(E.b);
  const long t = (wg - E.start[TB_ELIM0 + d]) * 64L + threadIdx.x;
  const ImpliWs w = impli_ws(ws + IMPLI_PLANES * b.npc, b.nnn);
  if (d == 0) elim_body<true>(b, 0, t, w);
  else elim_body<false>(b, d, t, w);
}

__global__ void __launch_bounds__(RT *RT) k_impli2_rhs_batch(const TurbEnt *__restrict__ tab, int nb, int d,
                                                             const double *__restrict__ u, long ldv, double *ws) {
  const unsigned wg = xcd_grouped(64);
  const TurbEnt &E = tab[tab_find(tab, nb, TB_RHS, wg)];
  const Blk b = uniform_blk(E.b);
  rhs_body(b, tab_tile(E, TB_RHS, wg), d, u, ldv, impli_ws(ws + IMPLI_PLANES * b.npc, b.nnn));
}

template <bool LAST>
__global__ void __launch_bounds__(64) k_impli2_line_batch(const TurbEnt *__restrict__ tab, int nb, int d, double *v,
                                                          long ldv, double *ws) {
  const TurbEnt &E = tab[tab_find(tab, nb, TB_LINE0 + d, blockIdx.x)];
  const Blk b = uniform_blk(E.b);
  line_body<LAST>(b, d, (blockIdx.x - E.start[TB_LINE0 + d]) * (long)LINES, v, ldv,
                  impli_ws(ws + IMPLI_PLANES * b.npc, b.nnn));
}

extern "C" int codens_impli2_eqt_3d_batch(int32_t nblk, const codens_block *blocks, const double *u, int64_t ldv,
                                          const double *dt, double *v, const double *mu, const double *mut,
                                          const double *cfke, const double *sn_all, const double *vol, double cmt,
                                          void *stream) {
  const char *what = "codens_impli2_eqt_3d_batch";
  if (nblk <= 0 || !blocks || !u || !dt || !v || !mu || !mut || !cfke || !sn_all || !vol || !(cmt > 0.)) {
    codens_set_error("%s: null or invalid argument", what);
    return CODENS_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  std::vector<TurbEnt> ent(nblk);
  std::vector<int32_t> key;
  std::vector<std::pair<long, long>> span(nblk);
  unsigned tot[TB_N] = {0};
  for (int l = 0; l < nblk; l++) {
    int rc = codens_check_block(&blocks[l], what);
    if (rc) return rc;
    const int32_t *wd = (const int32_t *)&blocks[l];
    key.insert(key.end(), wd, wd + sizeof(codens_block) / sizeof(int32_t));
    Blk b = make_blk(&blocks[l]);
    span[l] = {b.npc, b.npc + b.nnn};
    TurbEnt &E = ent[l];
    E.b = b;
    const unsigned ni = b.i2 - b.i1, nj = b.j2 - b.j1, nk = b.k2 - b.k1;
    auto waves = [&](int d, int per) { return (unsigned)((n_lines(b, d) + per - 1) / per); };
    unsigned g[TB_N][3] = {{cell_line(upto_high(b)).x, 1, 1},
                           {(ni + RT - 1) / RT, (nj + RT - 1) / RT, nk},
                           {waves(0, 64), 1, 1},
                           {waves(1, 64), 1, 1},
                           {waves(2, 64), 1, 1},
                           {waves(0, LINES), 1, 1},
                           {waves(1, LINES), 1, 1},
                           {waves(2, LINES), 1, 1}};
    for (int p = 0; p < TB_N; p++) {
      E.start[p] = tot[p];
      E.gx[p] = g[p][0];
      E.gy[p] = g[p][1];
      tot[p] += g[p][0] * g[p][1] * g[p][2];
    }
  }
  std::sort(span.begin(), span.end());
  for (int l = 0; l < nblk; l++) {
    if ((l == 0 && span[0].first != 0) || (l > 0 && span[l].first < span[l - 1].second) || span[l].second > ldv) {
      codens_set_error("%s: the blocks must start at entry 0, not overlap, and lie within ldv", what);
      return CODENS_EINVAL;
    }
  }
  const long tot_n = span[nblk - 1].second;
  TurbEnt *tab = (TurbEnt *)codens_device_table(2, key, ent.data(), sizeof(TurbEnt) * nblk, st, what);
  if (!tab) return CODENS_EHIP;
  double *ws = (double *)codens_workspace(sizeof(double) * IMPLI_PLANES * tot_n, 3);
  if (!ws) {
    codens_set_error("%s: workspace allocation failed", what);
    return CODENS_EHIP;
  }
  const TurbEnt *ct = tab;
  const int nb = nblk;
  CodensTimed _tm("impli2_eqt_3d", st);
  hipLaunchKernelGGL(k_impli2_faces_batch, dim3(tot[TB_FACE]), dim3(256), 0, st, ct, nb, (const double *)v,
                     (long)ldv, mu, mut, cmt, sn_all, vol, ws);
  hipLaunchKernelGGL(k_impli2_diag_batch, dim3(tot[TB_RHS]), dim3(RT * RT), 0, st, ct, nb, dt, vol, cfke, u,
                     (long)ldv, ws);
  hipLaunchKernelGGL(k_impli2_elim_batch, dim3(std::max(tot[TB_ELIM0], std::max(tot[TB_ELIM1], tot[TB_ELIM2])), 3),
                     dim3(64), 0, st, ct, nb, ws);
  for (int s = 0; s < 6; s++) {
    const int d = s / 2;
    if (s > 0) hipLaunchKernelGGL(k_impli2_rhs_batch, dim3(tot[TB_RHS]), dim3(RT * RT), 0, st, ct, nb, d, u, (long)ldv, ws);
    hipLaunchKernelGGL(s == 5 ? k_impli2_line_batch<true> : k_impli2_line_batch<false>, dim3(tot[TB_LINE0 + d]),
                       dim3(64), 0, st, ct, nb, d, v, (long)ldv, ws);
  }
  return codens_check_launch(what);
}

// met_samut.f90:46-58
__global__ void __launch_bounds__(TX *TY) k_met_samut(Blk b, double cv13, const double *__restrict__ v, long ldv,
                                                      const double *__restrict__ mu, double *__restrict__ mut) {
  REAL3(b)
  long n = b.idx(c[0], c[1], c[2]);
  double x = v[5 * ldv + n] / mu[n];
  double x3 = x * x * x;
  double fv1 = x3 / (x3 + cv13);
  mut[n] = v[5 * ldv + n] * fv1;
}

// met_kocmut.f90:53-90
__global__ void __launch_bounds__(TX *TY) k_met_kocmut(Blk b, int kwsst, double betas, const double *__restrict__ v,
                                                       long ldv, const double *__restrict__ mu,
                                                       double *__restrict__ mut, const double *__restrict__ dist,
                                                       const double *__restrict__ g9) {
  REAL3(b)
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc, nnn = b.nnn;
  if (kwsst == 0) {
    mut[n] = v[n] * v[5 * ldv + n] / v[6 * ldv + n];
    return;
  }
  double a1 = sqrt(betas);
  double omeg = v[6 * ldv + n] / v[n];
  double coef1 = sqrt(v[5 * ldv + n] / v[n]) / (betas * omeg * dist[n]);
  double coef2 = 500. * mu[n] / (v[6 * ldv + n] * (dist[n] * dist[n]));
  double x = g9[7 * nnn + m] - g9[5 * nnn + m], y = g9[2 * nnn + m] - g9[6 * nnn + m];
  double z = g9[3 * nnn + m] - g9[nnn + m];
  double rota = sqrt(x * x + y * y + z * z);
  double zeta = coef1 > coef2 ? coef1 : coef2;
  double z2 = 2. * (zeta * zeta);
  double exp2x = exp(z2 < 25. ? z2 : 25.);
  double f2 = (exp2x - 1.) / (exp2x + 1);
  double lim = rota * f2 / a1;
  mut[n] = v[5 * ldv + n] / (omeg > lim ? omeg : lim);
}

// met_cutsa.f90:40-49 (which = 2) and met_cut.f90:41-53 (which = 1)
__global__ void __launch_bounds__(TX *TY) k_met_cut(Blk b, int which, double epsk, double epse, double *v, long ldv) {
  REAL3(b)
  long n = b.idx(c[0], c[1], c[2]);
  double *s6 = v + 5 * ldv, *s7 = v + 6 * ldv;
  if (which == 2) {
    if (s6[n] < 0.) s6[n] = epsk;
    s7[n] = 0.;
  } else {
    double t6 = copysign(1.0, s6[n] - epsk), t7 = copysign(1.0, s7[n] - epse);
    double ts = copysign(1.0, t6 + t7 - 1.5);
    s6[n] = 0.5 * ((1. + ts) * s6[n] + (1. - ts) * epsk);
    s7[n] = 0.5 * ((1. + ts) * s7[n] + (1. - ts) * epse);
  }
}

extern "C" int codens_teq_gradv(const codens_block *cb, const double *sn, const double *vol, double *v, int64_t ldv,
                                double *g9, void *stream);

extern "C" int codens_met_samut(const codens_block *cb, const double *tc, const double *v, int64_t ldv,
                                const double *mu, double *mut, void *stream) {
  int rc = codens_check_block(cb, "codens_met_samut");
  if (rc) return rc;
  if (!tc || !v || !mu || !mut) {
    codens_set_error("codens_met_samut: null argument");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  double cv1 = tc[7];
  hipLaunchKernelGGL(k_met_samut, cell_line(b), dim3(TX, TY), 0, (hipStream_t)stream, b, cv1 * cv1 * cv1, v,
                     (long)ldv, mu, mut);
  return codens_check_launch("codens_met_samut");
}

extern "C" int codens_met_kocmut(const codens_block *cb, const double *tc, int32_t kwsst, const double *sn,
                                 const double *vol, double *v, int64_t ldv, const double *mu, double *mut,
                                 const double *dist, double *g9, void *stream) {
  int rc = codens_check_block(cb, "codens_met_kocmut");
  if (rc) return rc;
  if (!tc || !v || !mu || !mut || (kwsst == 1 && (!sn || !vol || !dist || !g9)) || (kwsst != 0 && kwsst != 1)) {
    codens_set_error("codens_met_kocmut: invalid argument");
    return CODENS_EINVAL;
  }
  if (kwsst == 1) {  // the reference computes the velocity gradients here (met_kocmut.f90:55-61)
    rc = codens_teq_gradv(cb, sn, vol, v, ldv, g9, stream);
    if (rc) return rc;
  }
  Blk b = make_blk(cb);
  hipLaunchKernelGGL(k_met_kocmut, cell_line(b), dim3(TX, TY), 0, (hipStream_t)stream, b, (int)kwsst, tc[10], v,
                     (long)ldv, mu, mut, dist, g9);
  return codens_check_launch("codens_met_kocmut");
}

extern "C" int codens_met_cut(const codens_block *cb, int32_t which, double epsk, double epse, double *v,
                              int64_t ldv, void *stream) {
  int rc = codens_check_block(cb, "codens_met_cut");
  if (rc) return rc;
  if (!v || (which != 1 && which != 2)) {
    codens_set_error("codens_met_cut: invalid argument (which = 1 met_cut, 2 met_cutsa)");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  hipLaunchKernelGGL(k_met_cut, cell_line(b), dim3(TX, TY), 0, (hipStream_t)stream, b, (int)which, epsk, epse, v,
                     (long)ldv);
  return codens_check_launch("codens_met_cut");
}

// met_smkor.f90:47-70: Wilcox k-omega sources with cross diffusion and the
// strain-rate limiter; fd = gradients of k and omega, g9 = velocity gradients
// and tprod block-local.
__global__ void __launch_bounds__(TX *TY) k_met_smkor(Blk b, double beta, double betas, double sigmw, double sigmd,
                                                      const double *__restrict__ v, long ldv,
                                                      const double *__restrict__ fd,
                                                      const double *__restrict__ g9,
                                                      const double *__restrict__ tprod, double *__restrict__ cfke,
                                                      double *__restrict__ ts6, double *__restrict__ ts7) {
  REAL3(b)
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc, nnn = b.nnn;
  double xw = beta / betas - sigmw * (0.41 * 0.41) / sqrt(betas);
  double rcmu = 1. / sqrt(0.09);
  double gkgo = fd[3 * ldv + n] * fd[n] + fd[4 * ldv + n] * fd[ldv + n] + fd[5 * ldv + n] * fd[2 * ldv + n];
  double omeg = v[6 * ldv + n] / v[n];
  double cd = sigmd * v[n] * (gkgo > 0. ? gkgo : 0.) / omeg;
  double dxx = g9[m], dyy = g9[4 * nnn + m], dzz = g9[8 * nnn + m];
  double a = g9[7 * nnn + m] + g9[5 * nnn + m], bb = g9[2 * nnn + m] + g9[6 * nnn + m];
  double cc = g9[3 * nnn + m] + g9[nnn + m];
  double ss = sqrt(4. * (dxx * dxx + dyy * dyy + dzz * dzz) / 3. + a * a + bb * bb + cc * cc) / omeg;
  double r = rcmu / ss;
  double alpha = 1. < r ? 1. : r;
  ts6[n] = tprod[m] - betas * v[5 * ldv + n] * omeg;
  ts7[n] = xw * tprod[m] * v[6 * ldv + n] / v[5 * ldv + n] / alpha - beta * v[6 * ldv + n] * omeg + cd;
  cfke[n] = 0.18 * omeg;
}

// met_smch.f90:88-108: Chien low-Reynolds k-epsilon sources
__global__ void __launch_bounds__(TX *TY) k_met_smch(Blk b, double cke1, double cke2, double utaumin,
                                                     const double *__restrict__ v, long ldv,
                                                     const double *__restrict__ mu,
                                                     const double *__restrict__ dist,
                                                     const int32_t *__restrict__ mnpar,
                                                     const double *__restrict__ utau,
                                                     const double *__restrict__ tprod, double *__restrict__ ts6,
                                                     double *__restrict__ ts7) {
  REAL3(b)
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc;
  int mp = mnpar[n];
  double yplus = 1000.;
  if (mp >= 1) {
    double ut = fabs(utau[mp - 1]);
    yplus = (ut > utaumin ? ut : utaumin) * dist[n] * v[n] / mu[n];
  }
  double rodst = v[n] * (dist[n] * dist[n]);
  double k = v[5 * ldv + n], e = v[6 * ldv + n];
  ts6[n] = tprod[m] - e - 2. * mu[n] * k / rodst;
  double epssk = e / k;
  double rtur = k / (mu[n] * epssk);
  double f2 = 1. - .22222222 * exp(-rtur * rtur / 36.);
  ts7[n] = cke1 * epssk * tprod[m] - cke2 * f2 * epssk * e - 2. * mu[n] * (e / rodst) * exp(-yplus / 2.);
}

extern "C" int codens_met_smkor(const codens_block *cb, const double *tc, double sigmd, const double *v,
                                int64_t ldv, const double *fd, const double *g9, const double *tprod, double *cfke,
                                double *ts6, double *ts7, void *stream) {
  int rc = codens_check_block(cb, "codens_met_smkor");
  if (rc) return rc;
  if (!tc || !v || !fd || !g9 || !tprod || !cfke || !ts6 || !ts7) {
    codens_set_error("codens_met_smkor: null argument");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  hipLaunchKernelGGL(k_met_smkor, cell_line(b), dim3(TX, TY), 0, (hipStream_t)stream, b, tc[11], tc[10], tc[13],
                     sigmd, v, (long)ldv, fd, g9, tprod, cfke, ts6, ts7);
  return codens_check_launch("codens_met_smkor");
}

extern "C" int codens_met_smch(const codens_block *cb, double cke1, double cke2, double utaumin, const double *v,
                               int64_t ldv, const double *mu, const double *dist, const int32_t *mnpar,
                               const double *utau, const double *tprod, double *ts6, double *ts7, void *stream) {
  int rc = codens_check_block(cb, "codens_met_smch");
  if (rc) return rc;
  if (!v || !mu || !dist || !mnpar || !utau || !tprod || !ts6 || !ts7) {
    codens_set_error("codens_met_smch: null argument");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  hipLaunchKernelGGL(k_met_smch, cell_line(b), dim3(TX, TY), 0, (hipStream_t)stream, b, cke1, cke2, utaumin, v,
                     (long)ldv, mu, dist, mnpar, utau, tprod, ts6, ts7);
  return codens_check_launch("codens_met_smch");
}
