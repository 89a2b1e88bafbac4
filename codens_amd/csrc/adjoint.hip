// Discrete tangent-linear (JVP) and adjoint (VJP) of the block residual of
// sch_roe on gfx950, for laminar Navier-Stokes with unlimited kappa-MUSCL
// (ilim = 0), adiabatic walls (clpara) and characteristic far fields (clnrd):
//
//   u(v; sn, vol) = sch_roe(v, ps, tq(v), sn)   after
//   zpres and zvismo on the real cells, the wall and far-field ghosts, and
//   zvisqc (Green-Gauss gradients, stresses, ghost stresses = adjacent cell),
//
// with the far-field normals and the free-stream state held fixed.  The
// minmod form (ilim = 1) is not covered: its chained slope ratios
// (sch_roe.f90:146-194) make each face's limiter a continued fraction over
// the whole grid line, and the reference build itself amplifies 1e-15
// changes of the state to 5e-3 within 10 stages there.
//
// Every piece of the residual is written once, templated on the scalar:
// double gives the values, Dual (value, tangent) gives exact directional
// derivatives.  The JVP runs the chain on Dual planes.  The VJP forms the
// values and walks the chain backwards with hand-written reverse sweeps of
// the face fluxes, the stresses, the gradients and the thermodynamics (the
// ghost rules: one Dual pass per input).  Its passes gather: a face's
// adjoints are stored at the face and summed by the cells that use them, so
// that only the ghosts, a surface, scatter with FP64 atomic adds.
//
// Arithmetic restates oracle_flux.c / oracle_visc.c (sch_roe.f90:322-578,
// zpres.f90:66-79, zvismo.f90:90-104, clpara.f90:44-58, clnrd.f90:60-134,
// zgrad2.f90:148-485, zfluto.f90:104-121) in the same operation order, so
// the double instantiation reproduces the residual to rounding.
#include "common.hpp"

#pragma clang fp contract(off)

using namespace codens;

namespace {

// ---------------------------------------------------------------------------
// dual numbers
struct Dual {
  double v, d;
};
__device__ inline Dual mk(double v, double d = 0.) { return Dual{v, d}; }
__device__ inline Dual operator+(Dual a, Dual b) { return {a.v + b.v, a.d + b.d}; }
__device__ inline Dual operator-(Dual a, Dual b) { return {a.v - b.v, a.d - b.d}; }
__device__ inline Dual operator*(Dual a, Dual b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
__device__ inline Dual operator/(Dual a, Dual b) {
  double q = a.v / b.v;
  return {q, (a.d - q * b.d) / b.v};
}
__device__ inline Dual operator-(Dual a) { return {-a.v, -a.d}; }
__device__ inline Dual operator+(Dual a, double b) { return {a.v + b, a.d}; }
__device__ inline Dual operator+(double a, Dual b) { return {a + b.v, b.d}; }
__device__ inline Dual operator-(Dual a, double b) { return {a.v - b, a.d}; }
__device__ inline Dual operator-(double a, Dual b) { return {a - b.v, -b.d}; }
__device__ inline Dual operator*(Dual a, double b) { return {a.v * b, a.d * b}; }
__device__ inline Dual operator*(double a, Dual b) { return {a * b.v, a * b.d}; }
__device__ inline Dual operator/(Dual a, double b) { return {a.v / b, a.d / b}; }
__device__ inline Dual operator/(double a, Dual b) {
  double q = a / b.v;
  return {q, -q * b.d / b.v};
}
__device__ inline Dual sqrt(Dual a) {
  double s = ::sqrt(a.v);
  return {s, 0.5 * a.d / s};
}
__device__ inline Dual fabs(Dual a) { return a.v < 0. ? -a : a; }
__device__ inline double sqrt(double a) { return ::sqrt(a); }
__device__ inline double fabs(double a) { return ::fabs(a); }
__device__ inline double val(double a) { return a; }
__device__ inline double val(Dual a) { return a.v; }
__device__ inline double tan_(Dual a) { return a.d; }
template <typename T>
__device__ inline T zro();
template <>
__device__ inline double zro<double>() { return 0.; }
template <>
__device__ inline Dual zro<Dual>() { return Dual{0., 0.}; }

// a plane pair (values, tangents); T = double reads the values only
template <typename T>
struct Pl;
template <>
struct Pl<double> {
  const double *v;
  __device__ double operator[](long i) const { return v[i]; }
};
template <>
struct Pl<Dual> {
  const double *v, *d;
  __device__ Dual operator[](long i) const { return Dual{v[i], d[i]}; }
};
template <typename T>
struct Wp;
template <>
struct Wp<double> {
  double *v;
  __device__ void set(long i, double x) const { v[i] = x; }
};
template <>
struct Wp<Dual> {
  double *v, *d;
  __device__ void set(long i, Dual x) const {
    v[i] = x.v;
    d[i] = x.d;
  }
};

struct APhys {
  double gam, gam1, pinfl, pr, cp, usrey, asuth;
  int iflu;
};

// zpres.f90:66-79 then zvismo.f90:90-104 (mut = 0)
template <typename T>
__device__ inline void thermo(const APhys &ph, const T w[5], T &p, T &tt, T &mu) {
  T rhoe = w[4] - 0.5 * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]) / w[0];
  p = ph.gam1 * (rhoe - ph.pinfl);
  tt = ph.gam * p / w[0];
  if (ph.iflu == 1)
    mu = ph.usrey * tt * sqrt(tt) * (1. + ph.asuth) / (tt + ph.asuth);
  else
    mu = tt * 0. + ph.usrey;
}

// Ghost state of a boundary face as a function of the adjacent real cell:
// conservative state wg (read by the boundary flux), primitive state qg
// (rho, u, v, w, p: read by the MUSCL reconstruction) and temperature tg
// (read by the gradients).
template <typename T>
__device__ inline void ghost_prims(const T wg[5], T pg, T qg[5]) {
  qg[0] = wg[0];
  qg[1] = wg[1] / wg[0];
  qg[2] = wg[2] / wg[0];
  qg[3] = wg[3] / wg[0];
  qg[4] = pg;
}

// clpara.f90:44-58
template <typename T>
__device__ inline void wall_ghost(const APhys &ph, const T vi[5], T wg[5], T qg[5], T &tg) {
  T rhoe1 = vi[4] - 0.5 * (vi[1] * vi[1] + vi[2] * vi[2] + vi[3] * vi[3]) / vi[0];
  T p, mu;
  thermo(ph, vi, p, tg, mu);
  wg[0] = vi[0];
  wg[1] = vi[1] * 0.;
  wg[2] = vi[1] * 0.;
  wg[3] = vi[1] * 0.;
  wg[4] = rhoe1;
  ghost_prims(wg, p, qg);
}

// rbve.f90 copy then clnrd.f90:60-134 against the state w0 (inward unit
// normal n)
template <typename T>
__device__ inline void far_ghost(const APhys &ph, const double *w0, double nx, double ny, double nz, const T vi[5],
                                 T wg[5], T qg[5], T &tg) {
  const double gam = ph.gam, gam1 = ph.gam1, pinfl = ph.pinfl;
  T ro0 = vi[0];
  T ps0 = gam1 * (vi[4] - 0.5 * (vi[1] * vi[1] + vi[2] * vi[2] + vi[3] * vi[3]) / vi[0] - pinfl);
  T roc0 = sqrt(gam * ps0 * ro0);
  T roqn0 = vi[1] * nx + vi[2] * ny + vi[3] * nz;
  double epsm = .5 + copysign(.5, val(roc0 - roqn0));
  double eps0 = .5 + copysign(.5, -val(roqn0));
  double epsp = .5 + copysign(.5, val(-roc0 - roqn0));
  double rod = w0[0];
  double qxd = w0[1] / rod, qyd = w0[2] / rod, qzd = w0[3] / rod;
  double pd = gam1 * (w0[4] - .5 * rod * (qxd * qxd + qyd * qyd + qzd * qzd) - pinfl);
  double qnd = qxd * nx + qyd * ny + qzd * nz;
  double qtxd = qxd - qnd * nx, qtyd = qyd - qnd * ny, qtzd = qzd - qnd * nz;
  T ros = vi[0];
  T qxs = vi[1] / ros, qys = vi[2] / ros, qzs = vi[3] / ros;
  T p_s = gam1 * (vi[4] - .5 * ros * (qxs * qxs + qys * qys + qzs * qzs) - pinfl);
  T qns = qxs * nx + qys * ny + qzs * nz;
  T qtxs = qxs - qns * nx, qtys = qys - qns * ny, qtzs = qzs - qns * nz;
  T qtx = eps0 * qtxs + (1. - eps0) * qtxd;
  T qty = eps0 * qtys + (1. - eps0) * qtyd;
  T qtz = eps0 * qtzs + (1. - eps0) * qtzd;
  T am = epsm * (p_s - roc0 * qns) + (1. - epsm) * (pd - roc0 * qnd);
  T ap = epsp * (p_s + roc0 * qns) + (1. - epsp) * (pd + roc0 * qnd);
  T qn = 0.5 * (ap - am) / roc0;
  T p = 0.5 * (ap + am);
  T bs = (p - p_s) * (ro0 * ro0) / (roc0 * roc0) + ros;
  T b0 = (p - pd) * (ro0 * ro0) / (roc0 * roc0) + rod;
  T ro = eps0 * bs + (1. - eps0) * b0;
  wg[0] = ro;
  wg[1] = ro * (qtx + qn * nx);
  wg[2] = ro * (qty + qn * ny);
  wg[3] = ro * (qtz + qn * nz);
  wg[4] = p / gam1 + pinfl + 0.5 * (wg[1] * wg[1] + wg[2] * wg[2] + wg[3] * wg[3]) / ro;
  tg = gam * p / ro;
  ghost_prims(wg, p, qg);
}

// zfluto.f90:104-121 with mut = 0; g: the 12 scaled gradients
template <typename T>
__device__ inline void stresses(const APhys &ph, const T g[12], T mu, T tq[9]) {
  const double ds3 = 2. / 3.;
  T xx = g[0], xy = g[1], xz = g[2], yx = g[3], yy = g[4], yz = g[5], zx = g[6], zy = g[7], zz = g[8];
  T mt = mu + 0.;
  tq[0] = ds3 * mt * (2 * xx - yy - zz);
  tq[3] = ds3 * mt * (2 * yy - xx - zz);
  tq[5] = ds3 * mt * (2 * zz - xx - yy);
  tq[1] = mt * (xy + yx);
  tq[2] = mt * (xz + zx);
  tq[4] = mt * (yz + zy);
  T kq = ph.cp * (mu / ph.pr + 0.);
  tq[6] = kq * g[9];
  tq[7] = kq * g[10];
  tq[8] = kq * g[11];
}

// zgrad2.f90:463-485: scale 0.5 / vol, guarded for vol <= 0
template <typename T>
__device__ inline T grad_scale(T vol) {
  if (!signbit(val(vol))) return .5 / (vol + DBL_MIN);  // vols = vol
  return vol * 0. + .5 / (0.00001 + DBL_MIN);            // vols = eps
}

// Roe flux of one face (2x the numerical flux . S), sch_roe.f90:327-473
template <typename T>
__device__ void roe_face_t(const APhys &ph, const T s[3], const T L[5], const T R[5], const T tl[9], const T tr[9],
                           T f[5]) {
  const double gam = ph.gam, gam1 = ph.gam1, pinfl = ph.pinfl;
  T rhol = L[0], ul = L[1], vl = L[2], wl = L[3], pl = L[4];
  T rhor = R[0], ur = R[1], vr = R[2], wr = R[3], prr = R[4];
  const double igam1 = 1. / gam1;
  T s0 = s[0], s1 = s[1], s2 = s[2];
  T cnds = sqrt(s0 * s0 + s1 * s1 + s2 * s2), icn = 1. / cnds;
  T nx = s0 * icn, ny = s1 * icn, nz = s2 * icn;
  T irl = 1. / rhol, irr = 1. / rhor;
  T al2 = gam * pl * irl, ar2 = gam * prr * irr;
  T q2l = ul * ul + vl * vl + wl * wl, q2r = ur * ur + vr * vr + wr * wr;
  T hl = al2 * igam1 + 0.5 * q2l, hr = ar2 * igam1 + 0.5 * q2r;
  T el = (pl * igam1 + pinfl) * irl + 0.5 * q2l;
  T er = (prr * igam1 + pinfl) * irr + 0.5 * q2r;
  T gd = sqrt(rhor * irl), gd1 = 1. / (1. + gd), gd2 = gd * gd1;
  T rhom = sqrt(rhol * rhor), rhomi = 1. / rhom;
  T um = gd1 * ul + gd2 * ur, vm = gd1 * vl + gd2 * vr, wm = gd1 * wl + gd2 * wr;
  T hm = gd1 * hl + gd2 * hr;
  T vitm2 = 0.5 * (um * um + vm * vm + wm * wm);
  T am = sqrt(gam1 * (hm - vitm2)), ami = 1. / am;
  T am2i = ami * ami;
  T vn = um * nx + vm * ny + wm * nz;
  T rhoiam = rhom * ami, rhoami = ami * rhomi;
  T l1 = fabs(vn * cnds), l4 = fabs(vn * cnds + am * cnds), l5 = fabs(vn * cnds - am * cnds);
  T dw0 = rhor - rhol;
  T dw1 = rhor * ur - rhol * ul;
  T dw2 = rhor * vr - rhol * vl;
  T dw3 = rhor * wr - rhol * wl;
  T dw4 = rhor * er - rhol * el;
  T g = gam1 * vitm2 * am2i;
  T qdw = gam1 * (um * dw1 + vm * dw2 + wm * dw3 - dw4);
  T a0 = (1. - g) * nx * dw0 - (vm * nz - wm * ny) * rhomi * dw0 + nx * am2i * qdw + (nz * dw2 - ny * dw3) * rhomi;
  T a1 = (1. - g) * ny * dw0 - (wm * nx - um * nz) * rhomi * dw0 + ny * am2i * qdw + (nx * dw3 - nz * dw1) * rhomi;
  T a2 = (1. - g) * nz * dw0 - (um * ny - vm * nx) * rhomi * dw0 + nz * am2i * qdw + (ny * dw1 - nx * dw2) * rhomi;
  T mdw = (nx * dw1 + ny * dw2 + nz * dw3) * rhomi;
  T cdw = gam1 * rhoami * (vitm2 * dw0 - um * dw1 - vm * dw2 - wm * dw3 + dw4);
  T a3 = cdw - vn * rhomi * dw0 + mdw;
  T a4 = cdw + vn * rhomi * dw0 - mdw;
  a0 = a0 * l1; a1 = a1 * l1; a2 = a2 * l1; a3 = a3 * l4; a4 = a4 * l5;
  T h = 0.5 * rhoiam;
  T di0 = nx * a0 + ny * a1 + nz * a2 + h * (a3 + a4);
  T di1 = um * nx * a0 + (um * ny - rhom * nz) * a1 + (um * nz + rhom * ny) * a2 +
          h * ((um + nx * am) * a3 + (um - nx * am) * a4);
  T di2 = (vm * nx + rhom * nz) * a0 + vm * ny * a1 + (vm * nz - rhom * nx) * a2 +
          h * ((vm + ny * am) * a3 + (vm - ny * am) * a4);
  T di3 = (wm * nx - rhom * ny) * a0 + (wm * ny + rhom * nx) * a1 + wm * nz * a2 +
          h * ((wm + nz * am) * a3 + (wm - nz * am) * a4);
  T di4 = (vitm2 * nx + rhom * (vm * nz - wm * ny)) * a0 + (vitm2 * ny + rhom * (wm * nx - um * nz)) * a1 +
          (vitm2 * nz + rhom * (um * ny - vm * nx)) * a2 + h * ((hm + am * vn) * a3 + (hm - am * vn) * a4);
  T dfxx = rhor * (ur * ur) + prr - pinfl - tr[0] + rhol * (ul * ul) + pl - pinfl - tl[0];
  T dfxy = rhor * ur * vr - tr[1] + rhol * ul * vl - tl[1];
  T dfxz = rhor * ur * wr - tr[2] + rhol * ul * wl - tl[2];
  T dfyy = rhor * (vr * vr) + prr - pinfl - tr[3] + rhol * (vl * vl) + pl - pinfl - tl[3];
  T dfyz = rhor * vr * wr - tr[4] + rhol * vl * wl - tl[4];
  T dfzz = rhor * (wr * wr) + prr - pinfl - tr[5] + rhol * (wl * wl) + pl - pinfl - tl[5];
  T Er = rhor * er + prr - pinfl, El = rhol * el + pl - pinfl;
  T dfex = Er * ur + El * ul - (tr[0] * ur + tr[1] * vr + tr[2] * wr) - (tl[0] * ul + tl[1] * vl + tl[2] * wl) -
           tr[6] - tl[6];
  T dfey = Er * vr + El * vl - (tr[1] * ur + tr[3] * vr + tr[4] * wr) - (tl[1] * ul + tl[3] * vl + tl[4] * wl) -
           tr[7] - tl[7];
  T dfez = Er * wr + El * wl - (tr[2] * ur + tr[4] * vr + tr[5] * wr) - (tl[2] * ul + tl[4] * vl + tl[5] * wl) -
           tr[8] - tl[8];
  f[0] = (rhor * ur + rhol * ul) * s0 + (rhor * vr + rhol * vl) * s1 + (rhor * wr + rhol * wl) * s2 - di0;
  f[1] = dfxx * s0 + dfxy * s1 + dfxz * s2 - di1;
  f[2] = dfxy * s0 + dfyy * s1 + dfyz * s2 - di2;
  f[3] = dfxz * s0 + dfyz * s1 + dfzz * s2 - di3;
  f[4] = dfex * s0 + dfey * s1 + dfez * s2 - di4;
}

// Physical flux of a ghost state on a boundary face, Navier-Stokes form
// (sch_roe.f90:497-578; oracle_flux.c phys_flux with rho_div = w[0])
template <typename T>
__device__ void phys_flux_t(const APhys &ph, const T w[5], T p, const T t[9], const T s[3], T f[5]) {
  const double pinfl = ph.pinfl;
  T fxx = w[1] * (w[1] / w[0]) + p - pinfl - t[0];
  T fxy = w[2] * (w[1] / w[0]) - t[1];
  T fxz = w[3] * (w[1] / w[0]) - t[2];
  T fyy = w[2] * (w[2] / w[0]) + p - pinfl - t[3];
  T fyz = w[3] * (w[2] / w[0]) - t[4];
  T fzz = w[3] * (w[3] / w[0]) + p - pinfl - t[5];
  T fex = ((w[4] + p - pinfl - t[0]) * w[1] - t[1] * w[2] - t[2] * w[3]) / w[0] - t[6];
  T fey = ((w[4] + p - pinfl - t[3]) * w[2] - t[1] * w[1] - t[4] * w[3]) / w[0] - t[7];
  T fez = ((w[4] + p - pinfl - t[5]) * w[3] - t[2] * w[1] - t[4] * w[2]) / w[0] - t[8];
  f[0] = w[1] * s[0] + w[2] * s[1] + w[3] * s[2];
  f[1] = fxx * s[0] + fxy * s[1] + fxz * s[2];
  f[2] = fxy * s[0] + fyy * s[1] + fyz * s[2];
  f[3] = fxz * s[0] + fyz * s[1] + fzz * s[2];
  f[4] = fex * s[0] + fey * s[1] + fez * s[2];
}

// ---------------------------------------------------------------------------
// Workspace planes (block-local index m, nnn entries each; JVP tangents in a
// second set).  Q: primitive state of every real and ghost cell; TT: T;
// MU: mu of the real cells; W: conservative ghost state; TQ: stresses and
// heat flux (9); H: face fluxes (3 directions x 5, JVP only).
constexpr int P_Q = 0, P_TT = 5, P_MU = 6, P_W = 7, P_TQ = 12, P_H = 21, NPLANE = 36, NVPLANE = 21;

struct AdjArgs {
  Blk b;
  APhys ph;
  double muscl, xk;
  long ldv;
  const double *v, *vd;      // state (5 x ldv) and its tangent
  const double *sn, *snd;    // block metrics (9 x nnn) and tangent
  const double *vol, *vold;  // ldv
  const double *w0;          // far-field state (5)
  double *ws, *wd;           // planes and tangent planes
};

template <typename T>
__device__ inline Pl<T> plane(const AdjArgs &a, int p);
template <>
__device__ inline Pl<double> plane<double>(const AdjArgs &a, int p) {
  return {a.ws + (long)p * a.b.nnn};
}
template <>
__device__ inline Pl<Dual> plane<Dual>(const AdjArgs &a, int p) {
  return {a.ws + (long)p * a.b.nnn, a.wd + (long)p * a.b.nnn};
}
template <typename T>
__device__ inline Wp<T> wplane(const AdjArgs &a, int p);
template <>
__device__ inline Wp<double> wplane<double>(const AdjArgs &a, int p) {
  return {a.ws + (long)p * a.b.nnn};
}
template <>
__device__ inline Wp<Dual> wplane<Dual>(const AdjArgs &a, int p) {
  return {a.ws + (long)p * a.b.nnn, a.wd + (long)p * a.b.nnn};
}
template <typename T>
__device__ inline T ldx(const double *v, const double *d, long i);
template <>
__device__ inline double ldx<double>(const double *v, const double *, long i) {
  return v[i];
}
template <>
__device__ inline Dual ldx<Dual>(const double *v, const double *d, long i) {
  return Dual{v[i], d[i]};
}

template <typename T>
__device__ inline void load_v(const AdjArgs &a, long n, T w[5]) {
#pragma unroll
  for (int e = 0; e < 5; e++) w[e] = ldx<T>(a.v, a.vd, e * a.ldv + n);
}
template <typename T>
__device__ inline T load_sn(const AdjArgs &a, long m, int d, int c) {
  long o = ((long)c * 3 + d) * a.b.nnn + m;
  return ldx<T>(a.sn, a.snd, o);
}


// face of direction d (along index a1..a2, real transverse range), i fastest
__device__ inline bool face_of(const Blk &b, int d, unsigned t, int c[3]) {
  const unsigned n0 = b.i2 - b.i1 + (d == 0), n1 = b.j2 - b.j1 + (d == 1), n2 = b.k2 - b.k1 + (d == 2);
  if (t >= n0 * n1 * n2) return false;
  c[0] = b.i1 + (int)(t % n0);
  c[1] = b.j1 + (int)((t / n0) % n1);
  c[2] = b.k1 + (int)(t / (n0 * n1));
  return true;
}
__device__ inline int along(const int c[3], int d) { return c[d]; }

// ---------------------------------------------------------------------------
// forward pieces (T = double: values; T = Dual: values and tangents)

template <typename T>
__global__ void __launch_bounds__(256) k_adj_thermo(AdjArgs a) {
  int c[3];
  if (!line_cell(a.b, xcd_linear(), c)) return;
  long n = a.b.idx(c[0], c[1], c[2]), m = n - a.b.npc;
  T w[5], p, tt, mu;
  load_v(a, n, w);
  thermo(a.ph, w, p, tt, mu);
  T q[5] = {w[0], w[1] / w[0], w[2] / w[0], w[3] / w[0], p};
#pragma unroll
  for (int e = 0; e < 5; e++) wplane<T>(a, P_Q + e).set(m, q[e]);
  wplane<T>(a, P_TT).set(m, tt);
  wplane<T>(a, P_MU).set(m, mu);
}

template <typename T, int FAR>
__global__ void __launch_bounds__(256) k_adj_ghost(AdjArgs a, long nf, const int64_t *__restrict__ g,
                                                   const int64_t *__restrict__ in, const double *__restrict__ nrm) {
  long f = blockIdx.x * 256L + threadIdx.x;
  if (f >= nf) return;
  long mg = g[f] - a.b.npc;
  T vi[5], wg[5], qg[5], tg;
  load_v(a, in[f], vi);
  if (FAR)
    far_ghost(a.ph, a.w0, nrm[f], nrm[nf + f], nrm[2 * nf + f], vi, wg, qg, tg);
  else
    wall_ghost(a.ph, vi, wg, qg, tg);
#pragma unroll
  for (int e = 0; e < 5; e++) {
    wplane<T>(a, P_W + e).set(mg, wg[e]);
    wplane<T>(a, P_Q + e).set(mg, qg[e]);
  }
  wplane<T>(a, P_TT).set(mg, tg);
}

// value of gradient quantity q (u, v, w, T) at block-local m
template <typename T>
__device__ inline T gq(const AdjArgs &a, int q, long m) {
  return q < 3 ? plane<T>(a, P_Q + 1 + q)[m] : plane<T>(a, P_TT)[m];
}
__device__ inline const double *gqp(const AdjArgs &a, int q) { return a.ws + (q < 3 ? P_Q + 1 + q : P_TT) * a.b.nnn; }

// Green-Gauss sums of one real cell in zgrad2's accumulation order
// (directions k, j, i; per direction the low face, then the high one),
// scaled, and the stresses from them (128x64x32 cells: 19 us with the faces'
// loads behind branches, 15 with a direction's together).
template <typename T>
__global__ void __launch_bounds__(256) k_adj_grad(AdjArgs a) {
  int c[3];
  if (!line_cell(a.b, xcd_linear(), c)) return;
  const Blk &b = a.b;
  long m = b.idx(c[0], c[1], c[2]) - b.npc;
  T G[12], here[4];
#pragma unroll
  for (int x = 0; x < 12; x++) G[x] = zro<T>();
#pragma unroll
  for (int q = 0; q < 4; q++) here[q] = gq<T>(a, q, m);
#pragma unroll
  for (int d = 2; d >= 0; d--) {
    const long inc = b.inc(d);
    const bool lo_in = c[d] > b.lo(d), hi_in = c[d] < b.hi(d) - 1;
    T slo[3], shi[3], lo[4], hi[4];
#pragma unroll
    for (int cc = 0; cc < 3; cc++) {
      slo[cc] = load_sn<T>(a, m, d, cc);
      shi[cc] = load_sn<T>(a, m + inc, d, cc);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      lo[q] = gq<T>(a, q, m - inc);
      hi[q] = gq<T>(a, q, m + inc);
    }
    loads_issued();
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const T fl = (lo_in ? here[q] : lo[q]) + lo[q], fh = hi[q] + (hi_in ? here[q] : hi[q]);
#pragma unroll
      for (int cc = 0; cc < 3; cc++) G[3 * q + cc] = G[3 * q + cc] - fl * slo[cc] + fh * shi[cc];
    }
  }
  const T c0 = grad_scale(ldx<T>(a.vol, a.vold, m + b.npc));
  T tq[9];
#pragma unroll
  for (int x = 0; x < 12; x++) G[x] = G[x] * c0;
  stresses(a.ph, G, plane<T>(a, P_MU)[m], tq);
#pragma unroll
  for (int x = 0; x < 9; x++) wplane<T>(a, P_TQ + x).set(m, tq[x]);
}

// rbte.f90: ghost stresses = adjacent real cell
template <typename T>
__global__ void __launch_bounds__(256) k_adj_tq_ghost(AdjArgs a, long nf, const int64_t *__restrict__ g,
                                                      const int64_t *__restrict__ in) {
  long f = blockIdx.x * 256L + threadIdx.x;
  if (f >= nf) return;
  long mg = g[f] - a.b.npc, mi = in[f] - a.b.npc;
#pragma unroll
  for (int x = 0; x < 9; x++) wplane<T>(a, P_TQ + x).set(mg, plane<T>(a, P_TQ + x)[mi]);
}

// MUSCL coefficients of q(a-2), q(a-1), q(a), q(a+1) in the left and right
// states of the face between a-1 and a (sch_roe_euler.f90:143-171)
template <typename T>
__device__ inline void muscl_lr(double muscl, double xk, const T q0, const T q1, const T q2, const T q3, T &L,
                                T &R) {
  L = q1 + 0.25 * muscl * ((1. - xk) * (q1 - q0) + (1. + xk) * (q2 - q1));
  R = q2 - 0.25 * muscl * ((1. + xk) * (q2 - q1) + (1. - xk) * (q3 - q2));
}

// face flux H (0.5 x Roe flux on interior faces, the ghost's physical flux
// on boundary faces) of direction d at face index m
template <typename T>
__device__ inline void face_h(const AdjArgs &a, int d, const int c[3], T H[5]) {
  const Blk &b = a.b;
  long inc = b.inc(d), m = b.idx(c[0], c[1], c[2]) - b.npc;
  int al = c[d], a1 = b.lo(d), a2 = b.hi(d);
  T s[3];
#pragma unroll
  for (int cc = 0; cc < 3; cc++) s[cc] = load_sn<T>(a, m, d, cc);
  if (al > a1 && al < a2) {
    T L[5], R[5], tl[9], tr[9], f[5];
#pragma unroll
    for (int e = 0; e < 5; e++) {
      Pl<T> q = plane<T>(a, P_Q + e);
      muscl_lr(a.muscl, a.xk, q[m - 2 * inc], q[m - inc], q[m], q[m + inc], L[e], R[e]);
    }
#pragma unroll
    for (int x = 0; x < 9; x++) {
      tl[x] = plane<T>(a, P_TQ + x)[m - inc];
      tr[x] = plane<T>(a, P_TQ + x)[m];
    }
    roe_face_t(a.ph, s, L, R, tl, tr, f);
#pragma unroll
    for (int e = 0; e < 5; e++) H[e] = f[e] * 0.5;
  } else {
    long mg = al == a1 ? m - inc : m;
    T w[5], t[9];
#pragma unroll
    for (int e = 0; e < 5; e++) w[e] = plane<T>(a, P_W + e)[mg];
#pragma unroll
    for (int x = 0; x < 9; x++) t[x] = plane<T>(a, P_TQ + x)[mg];
    phys_flux_t(a.ph, w, plane<T>(a, P_Q + 4)[mg], t, s, H);
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_adj_faces(AdjArgs a, int d) {
  int c[3];
  if (!face_of(a.b, d, blockIdx.x * 256L + threadIdx.x, c)) return;
  long m = a.b.idx(c[0], c[1], c[2]) - a.b.npc;
  T H[5];
  face_h(a, d, c, H);
#pragma unroll
  for (int e = 0; e < 5; e++) wplane<T>(a, P_H + 5 * d + e).set(m, H[e]);
}

// u = sum over directions of H(high face) - H(low face) on the real cells
template <typename T>
__global__ void __launch_bounds__(256) k_adj_gather(AdjArgs a, double *u, double *ud) {
  int c[3];
  if (!line_cell(a.b, xcd_linear(), c)) return;
  const Blk &b = a.b;
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc;
#pragma unroll
  for (int e = 0; e < 5; e++) {
    Pl<T> h0 = plane<T>(a, P_H + e), h1 = plane<T>(a, P_H + 5 + e), h2 = plane<T>(a, P_H + 10 + e);
    T r = h0[m + 1] - h0[m];
    r = r + (h1[m + b.nid] - h1[m]);
    r = r + (h2[m + b.nijd] - h2[m]);
    u[e * a.ldv + n] = val(r);
    if constexpr (sizeof(T) == sizeof(Dual)) ud[e * a.ldv + n] = tan_(r);
  }
}

// ---------------------------------------------------------------------------
// adjoint pieces.  Adjoint planes (block-local, nnn each): F the left and
// right MUSCL states of every face (3 directions x (5 + 5), zero on boundary
// faces), W the conservative ghost state and its pressure (5 + 1), V the
// gradient quantities u, v, w, T of the ghosts (4), G the raw gradient sums
// (the nine distinct ones: the adjoint of the velocity gradient is
// symmetric), LM log mu (which stays finite where mu is zero).
constexpr int B_F = 0, B_W = 30, B_V = 36, B_G = 40, B_LM = 49, NBPLANE = 50;

struct AdjBar {
  double *bw;                 // adjoint planes
  const double *ub;           // adjoint of u (5 x ldv)
  double *vb, *snb, *volb;    // results: v (5 x ldv), sn (9 x nnn), vol (ldv)
};

__device__ inline double *bpl(const AdjArgs &a, const AdjBar &B, int p) { return B.bw + (long)p * a.b.nnn; }

// The transposed products below are reverse sweeps written out by hand: the
// values of the flux are formed once and its operations walked backwards,
// about four flux evaluations, where a Dual pass per input took 31 (or 18)
// evaluations of more than twice the work each.
//
// tau (xx xy xz yy yz zz of t) times S
__device__ inline void tau_s(const double t[9], const double s[3], double r[3]) {
  r[0] = t[0] * s[0] + t[1] * s[1] + t[2] * s[2];
  r[1] = t[1] * s[0] + t[3] * s[1] + t[4] * s[2];
  r[2] = t[2] * s[0] + t[4] * s[1] + t[5] * s[2];
}

__device__ inline double dot3(const double a[3], const double b[3]) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }

// The viscous part -(tau S) . (w, u) - q . S of a flux against the adjoint
// (w, f4) of its momentum and energy: sb += its adjoint of S.
__device__ inline void visc_sb(const double w[3], double f4, const double u[3], const double t[9], double sb[3]) {
  const double y[3] = {-(w[0] + f4 * u[0]), -(w[1] + f4 * u[1]), -(w[2] + f4 * u[2])};
  double ty[3];
  tau_s(t, y, ty);
#pragma unroll
  for (int x = 0; x < 3; x++) sb[x] += ty[x] - f4 * t[6 + x];
}

// Adjoint of roe_face_t: fb of f (5) to Lb, Rb (5 each) and sb (3).  The dissipation P |Lambda| Q dW is taken in its wave form:
// with the Roe averages u, h, c, the mean density r, the jumps dr, dp, du
// and dn = du . n,
//   a0 = |un| (dr - dp/c^2),  a1, a2 = |un +- c| (dp +- r c dn) / (2 c^2),
//   D = ( a0 + a1 + a2,
//         (a0 + a1 + a2) u + |un| r (du - n dn) + (a1 - a2) c n,
//         a0 u^2/2 + |un| r (u . du - un dn) + (a1 + a2) h + (a1 - a2) c un ),
// the same function of L, R and S, since dp = gam1 (u^2/2 drho - u . dm +
// dE) holds for the Roe averages of any two states.
__device__ __forceinline__ void roe_face_vjp(const APhys &ph, const double s[3], const double L[5], const double R[5],
                                             const double tl[9], const double tr[9], const double fb[5], double Lb[5],
                                             double Rb[5], double sb[3]) {
#pragma clang fp contract(fast)
  const double gam1 = ph.gam1, gg = ph.gam / ph.gam1;
  const double *w = fb + 1;  // adjoint of the momentum flux
  const double f4 = fb[4];
  const double A = ::sqrt(dot3(s, s)), iA = 1. / A;
  const double n[3] = {s[0] * iA, s[1] * iA, s[2] * iA};
  const double irl = 1. / L[0], irr = 1. / R[0];
  const double *uL = L + 1, *uR = R + 1;
  const double hL = gg * L[4] * irl + 0.5 * dot3(uL, uL), hR = gg * R[4] * irr + 0.5 * dot3(uR, uR);
  const double gd = ::sqrt(R[0] * irl), g1 = 1. / (1. + gd), g2 = gd * g1, r = L[0] * gd;
  double u[3], du[3];
#pragma unroll
  for (int x = 0; x < 3; x++) {
    u[x] = g1 * uL[x] + g2 * uR[x];
    du[x] = uR[x] - uL[x];
  }
  const double h = g1 * hL + g2 * hR, k = 0.5 * dot3(u, u), c = ::sqrt(gam1 * (h - k)), ic = 1. / c, ic2 = ic * ic;
  const double vn = dot3(u, n), dn = dot3(du, n), dr = R[0] - L[0], dp = R[4] - L[4];
  const double e0 = vn < 0. ? -1. : 1., e1 = vn + c < 0. ? -1. : 1., e2 = vn - c < 0. ? -1. : 1.;
  const double l0 = e0 * vn, l1 = e1 * (vn + c), l2 = e2 * (vn - c);
  const double p0 = dr - dp * ic2, p1 = 0.5 * ic2 * (dp + r * c * dn), p2 = 0.5 * ic2 * (dp - r * c * dn);
  const double a0 = l0 * p0, a1 = l1 * p1, a2 = l2 * p2, sh = l0 * r, a12 = a1 - a2, udu = dot3(u, du);
  // D and its adjoint -A fb
  const double D0 = a0 + a1 + a2;
  double fD = fb[0] * D0 + f4 * (a0 * k + sh * (udu - vn * dn) + (a1 + a2) * h + a12 * c * vn);
#pragma unroll
  for (int x = 0; x < 3; x++) fD += w[x] * (D0 * u[x] + sh * (du[x] - n[x] * dn) + a12 * c * n[x]);
  const double d4 = -A * f4;
  double dv[3] = {-A * w[0], -A * w[1], -A * w[2]};
  const double dvn = dot3(dv, n), t0 = -A * fb[0] + dot3(dv, u);
  const double a12b = c * (dvn + d4 * vn), a0b = t0 + d4 * k, a1b = t0 + d4 * h + a12b, a2b = t0 + d4 * h - a12b;
  const double shb = dot3(dv, du) - dvn * dn + d4 * (udu - vn * dn);
  double cb = a12 * (dvn + d4 * vn), vnb = d4 * (a12 * c - sh * dn), dnb = -sh * (dvn + d4 * vn);
  double hb = d4 * (a1 + a2), kb = d4 * a0;
  double ub[3], dub[3], nb[3];
#pragma unroll
  for (int x = 0; x < 3; x++) {
    ub[x] = D0 * dv[x] + d4 * sh * du[x];
    dub[x] = sh * (dv[x] + d4 * u[x]);
    nb[x] = (a12 * c - sh * dn) * dv[x];
  }
  // wave strengths
  const double p0b = a0b * l0, p1b = a1b * l1, p2b = a2b * l2;
  const double l0b = a0b * p0 + shb * r, l1b = a1b * p1, l2b = a2b * p2;
  double rb = shb * l0;
  const double dpb = ic2 * (0.5 * (p1b + p2b) - p0b), zb = 0.5 * ic2 * (p1b - p2b);
  double c2b = ic2 * (p0b * dp * ic2 - p1b * p1 - p2b * p2);
  rb += zb * c * dn;
  cb += zb * r * dn;
  dnb += zb * r * c;
  vnb += e0 * l0b + e1 * l1b + e2 * l2b;
  cb += e1 * l1b - e2 * l2b;
  c2b += 0.5 * ic * cb;
  hb += gam1 * c2b;
  kb -= gam1 * c2b;
#pragma unroll
  for (int x = 0; x < 3; x++) {
    ub[x] += kb * u[x] + vnb * n[x];
    nb[x] += vnb * u[x] + dnb * du[x];
    dub[x] += dnb * n[x];
  }
  // averages
  const double gdb = (dot3(ub, du) + hb * (hR - hL)) * g1 * g1;
  Lb[0] = -p0b + 0.5 * rb * r * irl - 0.5 * gdb * gd * irl;
  Rb[0] = p0b + 0.5 * rb * r * irr + 0.5 * gdb * gd * irr;
  Lb[4] = -dpb;
  Rb[4] = dpb;
  // physical fluxes F(L) + F(R): m = rho u . S, (m, m u + p S, m h)
  const double nbn = dot3(nb, n);
#pragma unroll
  for (int x = 0; x < 3; x++) sb[x] = (nb[x] - n[x] * nbn) * iA - fD * n[x];
#pragma unroll
  for (int side = 0; side < 2; side++) {
    const double *q = side ? R : L, *uq = side ? uR : uL, *t = side ? tr : tl;
    double *qb = side ? Rb : Lb;
    const double ir = side ? irr : irl, hq = side ? hR : hL, gq_ = side ? g2 : g1, sg = side ? 1. : -1.;
    const double un = dot3(uq, s), m = q[0] * un;
    const double mb = fb[0] + dot3(w, uq) + f4 * hq, hqb = f4 * m + gq_ * hb;
    double ts[3];
    tau_s(t, s, ts);
    qb[0] += mb * un - hqb * gg * q[4] * ir * ir;
    qb[4] += dot3(w, s) + hqb * gg * ir;
    const double unb = mb * q[0];
#pragma unroll
    for (int x = 0; x < 3; x++) {
      qb[1 + x] = sg * dub[x] + gq_ * ub[x] + m * w[x] - f4 * ts[x] + unb * s[x] + hqb * uq[x];
      sb[x] += unb * uq[x] + (q[4] - ph.pinfl) * w[x];
    }
    visc_sb(w, f4, uq, t, sb);
  }
}

// Adjoint of phys_flux_t: with u = m / rho and U = u . S the flux is
// (rho U, m U + (p - pinfl) S - tau S, (E + p - pinfl) U - u . tau S - q . S)
__device__ __forceinline__ void phys_flux_vjp(const APhys &ph, const double v[5], double p, const double t[9],
                                              const double s[3], const double fb[5], double vb[5], double &pb,
                                              double sb[3]) {
#pragma clang fp contract(fast)
  const double *w = fb + 1;
  const double f4 = fb[4], ir = 1. / v[0];
  const double u[3] = {v[1] * ir, v[2] * ir, v[3] * ir};
  const double U = dot3(u, s), Ub = fb[0] * v[0] + dot3(w, v + 1) + f4 * (v[4] + p - ph.pinfl);
  double ts[3], ub[3];
  tau_s(t, s, ts);
  pb = dot3(w, s) + f4 * U;
  vb[4] = f4 * U;
#pragma unroll
  for (int x = 0; x < 3; x++) {
    ub[x] = Ub * s[x] - f4 * ts[x];
    vb[1 + x] = U * w[x] + ub[x] * ir;
    sb[x] = Ub * u[x] + (p - ph.pinfl) * w[x];
  }
  vb[0] = fb[0] * U - dot3(ub, u) * ir;
  visc_sb(w, f4, u, t, sb);
}

// MUSCL: L = cl0 q0 + cl1 q1 + cl2 q2, R = cr1 q1 + cr2 q2 + cr3 q3
struct MusclW {
  double l0, l1, l2, r1, r2, r3;
};
__device__ inline MusclW muscl_w(const AdjArgs &a) {
  const double c4 = 0.25 * a.muscl, m = c4 * (1. - a.xk), p = c4 * (1. + a.xk);
  return {-m, 1. + (m - p), p, p, 1. - (p - m), -m};
}

// Transposed Jacobian of every face's flux, the three directions in one
// launch (nb0, nb1: workgroups of the first two): adjoints of the MUSCL
// states, of the ghost state on boundary faces, and the metric's.  One
// writer per entry.  The stresses' adjoints are gathered by k_adjb_tq.
// Bound by the planes it moves (39 written, 66 read): 128x64x32 cells took
// 49 us with loads behind branches, a boundary face's one after another (each
// wave of direction i has some), 44 with all of a face's in one group.
__global__ void __launch_bounds__(128) k_adjb_faces(AdjArgs a, AdjBar B, unsigned nb0, unsigned nb1) {
  const unsigned wg = xcd_linear();
  const int d = wg < nb0 ? 0 : (wg < nb0 + nb1 ? 1 : 2);
  const long blk = wg - (d == 0 ? 0 : (d == 1 ? nb0 : nb0 + nb1));
  int c[3];
  if (!face_of(a.b, d, blk * 128L + threadIdx.x, c)) return;
  const Blk &b = a.b;
  const long inc = b.inc(d), m = b.idx(c[0], c[1], c[2]) - b.npc, nnn = b.nnn, ldv = a.ldv;
  const int al = c[d], a1 = b.lo(d), a2 = b.hi(d);
  const double *ub = B.ub + b.npc;
  const unsigned mb = 8u * (unsigned)m, ib = 8u * (unsigned)inc;  // byte offsets in a plane
  double s[3], sb[3];
#pragma unroll
  for (int cc = 0; cc < 3; cc++) s[cc] = ldp(a.sn + ((long)cc * 3 + d) * nnn, mb);
  double Lb[5] = {0., 0., 0., 0., 0.}, Rb[5] = {0., 0., 0., 0., 0.};
  if (al > a1 && al < a2) {
    // u(m) has -H(m), u(m-inc) has +H(m); H = 0.5 f
    double fb[5], L[5], R[5], tl[9], tr[9], u[2][5], q[4][5];
#pragma unroll
    for (int e = 0; e < 5; e++) {
      u[0][e] = ldp(ub + e * ldv, mb - ib);
      u[1][e] = ldp(ub + e * ldv, mb);
#pragma unroll
      for (int x = 0; x < 4; x++) q[x][e] = ldp(a.ws + (P_Q + e) * nnn, mb + (unsigned)(x - 2) * ib);
    }
#pragma unroll
    for (int x = 0; x < 9; x++) {
      tl[x] = ldp(a.ws + (P_TQ + x) * nnn, mb - ib);
      tr[x] = ldp(a.ws + (P_TQ + x) * nnn, mb);
    }
    loads_issued();
#pragma unroll
    for (int e = 0; e < 5; e++) {
      fb[e] = 0.5 * (u[0][e] - u[1][e]);
      muscl_lr(a.muscl, a.xk, q[0][e], q[1][e], q[2][e], q[3][e], L[e], R[e]);
    }
    roe_face_vjp(a.ph, s, L, R, tl, tr, fb, Lb, Rb, sb);
  } else {
    const bool lo = al == a1;
    const unsigned mg = lo ? mb - ib : mb, mh = lo ? mb : mb - ib;
    double hb[5], w[5], t[9], wb[5], pb, p = ldp(a.ws + (P_Q + 4) * nnn, mg);
#pragma unroll
    for (int e = 0; e < 5; e++) hb[e] = ldp(ub + e * ldv, mh);
#pragma unroll
    for (int e = 0; e < 5; e++) w[e] = ldp(a.ws + (P_W + e) * nnn, mg);
#pragma unroll
    for (int x = 0; x < 9; x++) t[x] = ldp(a.ws + (P_TQ + x) * nnn, mg);
    loads_issued();
#pragma unroll
    for (int e = 0; e < 5; e++) hb[e] = lo ? -hb[e] : hb[e];
    phys_flux_vjp(a.ph, w, p, t, s, hb, wb, pb, sb);
#pragma unroll
    for (int e = 0; e < 5; e++) *gp(bpl(a, B, B_W + e), mg) = wb[e];
    *gp(bpl(a, B, B_W + 5), mg) = pb;
  }
#pragma unroll
  for (int e = 0; e < 5; e++) {
    *gp(bpl(a, B, B_F + 10 * d + e), mb) = Lb[e];
    *gp(bpl(a, B, B_F + 10 * d + 5 + e), mb) = Rb[e];
  }
#pragma unroll
  for (int cc = 0; cc < 3; cc++) *gp(B.snb + ((long)cc * 3 + d) * nnn, mb) = sb[cc];
}

// A face's flux has -(tau S) . (w, u) - q . S against its adjoint w (four
// components, momentum and energy), with u the velocity of one side: the part
// of tb, the adjoint of that side's stresses and heat flux.
__device__ __forceinline__ void tq_face(const double w[4], const double u[3], const double s[3], bool there,
                                        double tb[9]) {
#pragma clang fp contract(fast)
  double y[3], f4 = there ? w[3] : 0.;  // y: the adjoint of tau S
#pragma unroll
  for (int x = 0; x < 3; x++) y[x] = there ? -(w[x] + w[3] * u[x]) : 0.;
  tb[0] += y[0] * s[0];
  tb[1] += y[0] * s[1] + y[1] * s[0];
  tb[2] += y[0] * s[2] + y[2] * s[0];
  tb[3] += y[1] * s[1];
  tb[4] += y[1] * s[2] + y[2] * s[1];
  tb[5] += y[2] * s[2];
#pragma unroll
  for (int x = 0; x < 3; x++) tb[6 + x] -= f4 * s[x];
}

// tq is linear in mu and in the scale c0 of the gradients: from the adjoint tb
// of cell m's those of the raw gradient sums (g), of log mu and of vol
struct TqBar {
  double g[9], lm, vol;
};
__device__ __forceinline__ TqBar tq_cell(const AdjArgs &a, unsigned mb, long m, const double tb[9]) {
#pragma clang fp contract(fast)
  const long nnn = a.b.nnn;
  const double mu = a.ws[P_MU * nnn + m], vol = a.vol[m + a.b.npc], c0 = grad_scale(vol);
  double tt = 0.;
#pragma unroll
  for (int x = 0; x < 9; x++) tt += tb[x] * ldp(a.ws + (P_TQ + x) * nnn, mb);
  const double mc = mu * c0, m3 = 2. / 3. * mc, kq = a.ph.cp * (mu / a.ph.pr) * c0;
  return TqBar{{m3 * (2. * tb[0] - tb[3] - tb[5]), mc * tb[1], mc * tb[2], m3 * (2. * tb[3] - tb[0] - tb[5]),
                mc * tb[4], m3 * (2. * tb[5] - tb[0] - tb[3]), kq * tb[6], kq * tb[7], kq * tb[8]},
               tt,
               signbit(vol) ? 0. : -tt / (vol + DBL_MIN)};
}

// Stresses of a real cell: their adjoints gathered from the cell's interior
// faces, then those of what they are made of (26 us with its conditional loads
// one by one, 18 with a direction's together; 128x64x32 cells).
__global__ void __launch_bounds__(256) k_adjb_tq(AdjArgs a, AdjBar B) {
#pragma clang fp contract(fast)
  int c[3];
  if (!line_cell(a.b, xcd_linear(), c)) return;
  const Blk &b = a.b;
  const long m = b.idx(c[0], c[1], c[2]) - b.npc, nnn = b.nnn, ldv = a.ldv;
  const unsigned mb = 8u * (unsigned)m;  // the cell's byte offset in a plane
  const double *Q = a.ws + (P_Q + 1) * nnn;
  const double c4m = 0.25 * a.muscl * (1. - a.xk), c4p = 0.25 * a.muscl * (1. + a.xk);
  double ub0[4], u0[3], tb[9];
#pragma unroll
  for (int e = 0; e < 4; e++) ub0[e] = ldp(B.ub + (e + 1) * ldv + b.npc, mb);
#pragma unroll
  for (int x = 0; x < 3; x++) u0[x] = ldp(Q + x * nnn, mb);
#pragma unroll
  for (int x = 0; x < 9; x++) tb[x] = 0.;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const long inc = b.inc(d);
    const unsigned ib = 8u * (unsigned)inc;
    const bool bnd[2] = {c[d] == b.lo(d), c[d] == b.hi(d) - 1};
    // of the neighbours below and above: velocities, adjoints of u (a boundary's
    // are not read), and the faces' normals
    double um[2][3], un[2][4], s[2][3];
#pragma unroll
    for (int side = 0; side < 2; side++) {
      const unsigned mo = side ? mb + ib : mb - ib;
#pragma unroll
      for (int x = 0; x < 3; x++) um[side][x] = ldp(Q + x * nnn, mo);
#pragma unroll
      for (int e = 0; e < 4; e++) un[side][e] = ldp(B.ub + (e + 1) * ldv + b.npc, bnd[side] ? mb : mo);
#pragma unroll
      for (int x = 0; x < 3; x++) s[side][x] = ldp(a.sn + ((long)x * 3 + d) * nnn, side ? mo : mb);
    }
    loads_issued();
#pragma unroll
    for (int side = 0; side < 2; side++) {
      double w[4], u[3];
#pragma unroll
      for (int e = 0; e < 4; e++) w[e] = (side ? 0.5 : -0.5) * (ub0[e] - un[side][e]);
      // the MUSCL state of the cell's side: extrapolated toward the face
#pragma unroll
      for (int x = 0; x < 3; x++) u[x] = u0[x] + c4m * (u0[x] - um[1 - side][x]) + c4p * (um[side][x] - u0[x]);
      tq_face(w, u, s[side], !bnd[side], tb);
    }
  }
  const TqBar r = tq_cell(a, mb, m, tb);
  bpl(a, B, B_LM)[m] = r.lm;
  B.volb[m + b.npc] = r.vol;
#pragma unroll
  for (int x = 0; x < 9; x++) *gp(bpl(a, B, B_G + x), mb) = r.g[x];
}

// Whether storage entry m of a block (block-local) is the ghost of a boundary
// face; then the direction it lies in and whether below the block.  An edge's,
// a corner's or a deeper ghost is read by no face.
__device__ __forceinline__ bool face_ghost(const Blk &b, long m, int &d, bool &lo) {
  const int c[3] = {b.id1 + (int)(m % b.nid), b.jd1 + (int)((m / b.nid) % (b.nijd / b.nid)),
                    b.kd1 + (int)(m / b.nijd)};
  int layers = 0;
  d = 0;
#pragma unroll
  for (int x = 0; x < 3; x++) {
    const int out = max(b.lo(x) - c[x], c[x] - b.hi(x) + 1);
    if (out > 0) {
      d = x;
      layers += out;
    }
  }
  lo = c[d] < b.lo(d);
  return layers == 1;
}

// Ghost stresses transposed: a boundary face's go to the cell that the list
// copies them from, 11 atomic adds a ghost (10 us for the 28,672 of 128x64x32;
// gathered by the adjacent cell they cost nothing, but the lists may name others).
__global__ void __launch_bounds__(128) k_adjb_tq_ghost(AdjArgs a, AdjBar B, long nwall, const int64_t *__restrict__ wg,
                                                       const int64_t *__restrict__ wi, long nfar,
                                                       const int64_t *__restrict__ fg,
                                                       const int64_t *__restrict__ fi) {
#pragma clang fp contract(fast)
  const long t = blockIdx.x * 128L + threadIdx.x;
  if (t >= nwall + nfar) return;
  const Blk &b = a.b;
  const long nnn = b.nnn, mg = (t < nwall ? wg[t] : fg[t - nwall]) - b.npc;
  const long mi = (t < nwall ? wi[t] : fi[t - nwall]) - b.npc;
  int d;
  bool lo;
  if (!face_ghost(b, mg, d, lo)) return;
  const long inc = b.inc(d), mr = lo ? mg + inc : mg - inc, mf = lo ? mr : mg;  // its face's cell, its face
  double w[4], u[3], s[3], tb[9];
#pragma unroll
  for (int e = 0; e < 4; e++) w[e] = (lo ? -1. : 1.) * B.ub[(e + 1) * a.ldv + b.npc + mr];
  const double ir = 1. / a.ws[P_W * nnn + mg];
#pragma unroll
  for (int x = 0; x < 3; x++) {
    u[x] = a.ws[(P_W + 1 + x) * nnn + mg] * ir;
    s[x] = a.sn[((long)x * 3 + d) * nnn + mf];
  }
#pragma unroll
  for (int x = 0; x < 9; x++) tb[x] = 0.;
  tq_face(w, u, s, true, tb);
  const TqBar r = tq_cell(a, 8u * (unsigned)mi, mi, tb);
  atomicAdd(bpl(a, B, B_LM) + mi, r.lm);
  atomicAdd(B.volb + b.npc + mi, r.vol);
#pragma unroll
  for (int x = 0; x < 9; x++) atomicAdd(bpl(a, B, B_G + x) + mi, r.g[x]);
}

// plane (from B_G) of the adjoint of d(quantity q)/d(x_cc)
__device__ inline constexpr int g_plane(int q, int cc) {
  return q == 3 ? 6 + cc : (q + cc == 0 ? 0 : (q == cc ? (q == 1 ? 3 : 5) : q + cc + (q + cc == 3 ? 1 : 0)));
}
static_assert(g_plane(0, 1) == 1 && g_plane(2, 0) == 2 && g_plane(1, 1) == 3 && g_plane(1, 2) == 4 && g_plane(2, 2) == 5,
              "xx xy xz yy yz zz");

// Real cells, the last pass over them: the Green-Gauss sums of the cell's six
// faces transposed (onto its own u, v, w, T; onto a boundary face's ghost;
// onto the metrics of its low faces and of the block's high faces), the MUSCL
// states' adjoints of the faces that reach the cell, and the thermodynamics
// onto the conservative state.  Bound by its 82 planes: 128x64x32 cells took
// 51 us with a branch around each conditional load, 45 (4.1 TB/s) with two
// groups of unconditional loads per direction, the face states' sums formed
// before the second (48 with all of them at once: 330 registers, one wave).
__global__ void __launch_bounds__(256) k_adjb_cells(AdjArgs a, AdjBar B) {
#pragma clang fp contract(fast)
  int c[3];
  if (!line_cell(a.b, xcd_linear(), c)) return;
  const Blk &b = a.b;
  const long n = b.idx(c[0], c[1], c[2]), m = n - b.npc, nnn = b.nnn;
  const unsigned mb = 8u * (unsigned)m;  // the cell's byte offset in a plane
  const MusclW mw = muscl_w(a);
  double g0[9], q0[4], vb[4] = {0., 0., 0., 0.}, qb[5] = {0., 0., 0., 0., 0.};
#pragma unroll
  for (int x = 0; x < 9; x++) g0[x] = ldp(bpl(a, B, B_G + x), mb);
#pragma unroll
  for (int q = 0; q < 4; q++) q0[q] = ldp(gqp(a, q), mb);
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const long inc = b.inc(d);
    const int al = c[d], a1 = b.lo(d), a2 = b.hi(d);
    const unsigned ib = 8u * (unsigned)inc;
    const bool bnd[2] = {al == a1, al == a2 - 1};
    // the cell is q1 of its high face, q2 of its low face, q0 of the face
    // after the high one and q3 of the face before the low one
    double L[3][5], R[3][5];
    const bool far = al + 2 < a2, near = al - 1 > a1;
#pragma unroll
    for (int e = 0; e < 5; e++) {
      const double *Lb = bpl(a, B, B_F + 10 * d + e), *Rb = Lb + 5 * nnn;
      L[0][e] = ldp(Lb, mb);
      L[1][e] = ldp(Lb, mb + ib);
      L[2][e] = ldp(Lb, mb + (far ? 2 * ib : 0));
      R[0][e] = ldp(Rb, mb);
      R[1][e] = ldp(Rb, mb + ib);
      R[2][e] = ldp(Rb, mb - (near ? ib : 0));
    }
    loads_issued();
#pragma unroll
    for (int e = 0; e < 5; e++) {
      double r = mw.l2 * L[0][e] + mw.r2 * R[0][e] + mw.l1 * L[1][e] + mw.r1 * R[1][e];
      r += far ? mw.l0 * L[2][e] : 0.;
      r += near ? mw.r3 * R[2][e] : 0.;
      qb[e] += r;
      asm volatile("" : "+v"(qb[e]));  // formed here, its loads' registers free for the next ones
    }
    const unsigned mh = mb + (bnd[1] ? ib : 0);
    double s[2][3], gn[2][9], qn[2][4], sb0[3], sb1[3];
#pragma unroll
    for (int side = 0; side < 2; side++) {
      const unsigned mo = side ? mb + ib : mb - ib, mi = bnd[side] ? mb : mo;
#pragma unroll
      for (int x = 0; x < 3; x++) s[side][x] = ldp(a.sn + ((long)x * 3 + d) * nnn, side ? mo : mb);
#pragma unroll
      for (int x = 0; x < 9; x++) gn[side][x] = ldp(bpl(a, B, B_G + x), mi);
#pragma unroll
      for (int q = 0; q < 4; q++) qn[side][q] = ldp(gqp(a, q), mo);
    }
#pragma unroll
    for (int x = 0; x < 3; x++) {
      sb0[x] = ldp(B.snb + ((long)x * 3 + d) * nnn, mb);
      sb1[x] = ldp(B.snb + ((long)x * 3 + d) * nnn, mh);
    }
    loads_issued();
#pragma unroll
    for (int side = 0; side < 2; side++) {
      const unsigned mo = side ? mb + ib : mb - ib;
      double t[9], sb[3] = {0., 0., 0.};
      // adjoint of the face sums: low cell's less high cell's
#pragma unroll
      for (int x = 0; x < 9; x++) {
        const double g = bnd[side] ? 0. : gn[side][x];
        t[x] = side ? g0[x] - g : g - g0[x];
      }
      double f[4];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        f[q] = 0.;
#pragma unroll
        for (int x = 0; x < 3; x++) f[q] += t[g_plane(q, x)] * s[side][x];
        vb[q] += bnd[side] ? 0. : f[q];
        const double fv = bnd[side] ? 2. * qn[side][q] : q0[q] + qn[side][q];
#pragma unroll
        for (int x = 0; x < 3; x++) sb[x] += t[g_plane(q, x)] * fv;
      }
      if (bnd[side]) {
#pragma unroll
        for (int q = 0; q < 4; q++) *gp(bpl(a, B, B_V + q), mo) = 2. * f[q];
      }
      // a face's by the cell above it, the block's last face by the one below
      if (side == 0) {
#pragma unroll
        for (int x = 0; x < 3; x++) *gp(B.snb + ((long)x * 3 + d) * nnn, mb) = sb0[x] + sb[x];
      } else if (bnd[1]) {
#pragma unroll
        for (int x = 0; x < 3; x++) *gp(B.snb + ((long)x * 3 + d) * nnn, mh) = sb1[x] + sb[x];
      }
    }
  }
  double w[5];
  load_v(a, n, w);
  const double ir = 1. / w[0], T = q0[3];
  double Tb = vb[3];
  if (a.ph.iflu == 1) Tb += bpl(a, B, B_LM)[m] * (1.5 / T - 1. / (T + a.ph.asuth));
  const double pb = qb[4] + Tb * a.ph.gam * ir, ep = a.ph.gam1 * pb;
  double r0 = qb[0] - Tb * T * ir;
#pragma unroll
  for (int x = 0; x < 3; x++) {
    const double xb = qb[1 + x] + vb[x];
    B.vb[(1 + x) * a.ldv + n] = (xb - ep * w[1 + x]) * ir;
    r0 -= (xb - 0.5 * ep * w[1 + x]) * q0[x] * ir;
  }
  B.vb[n] = r0;
  B.vb[4 * a.ldv + n] = ep;
}

// Ghost rules transposed: adjoints of the ghost's W, q and T onto the
// adjacent cell's conservative state, one Dual pass and one thread per input.
template <int FAR>
__global__ void __launch_bounds__(128) k_adjb_ghost(AdjArgs a, AdjBar B, long nf, const int64_t *__restrict__ g,
                                                    const int64_t *__restrict__ in, const double *__restrict__ nrm) {
  const long t = blockIdx.x * 128L + threadIdx.x;
  if (t >= 5 * nf) return;
  const long f = t % nf;
  const int k = (int)(t / nf);
  const Blk &b = a.b;
  const long mg = g[f] - b.npc, ni = in[f], nnn = b.nnn;
  // the interior face in the ghost's direction whose MUSCL states reach it
  // (where the block has one)
  int d;
  bool lo;
  if (!face_ghost(b, mg, d, lo)) return;
  const long inc = b.inc(d);
  const MusclW mw = muscl_w(a);
  double wb[5], qb[5], tb;
#pragma unroll
  for (int e = 0; e < 5; e++) {
    const double *Lb = bpl(a, B, B_F + 10 * d + e), *Rb = Lb + 5 * nnn;
    wb[e] = bpl(a, B, B_W + e)[mg];
    qb[e] = lo ? mw.l0 * Lb[mg + 2 * inc] : mw.r3 * Rb[mg - inc];
  }
  qb[4] += bpl(a, B, B_W + 5)[mg];
#pragma unroll
  for (int q = 0; q < 3; q++) qb[1 + q] += bpl(a, B, B_V + q)[mg];
  tb = bpl(a, B, B_V + 3)[mg];
  double vi[5];
  load_v(a, ni, vi);
  Dual vD[5], wg[5], qg[5], tg;
#pragma unroll
  for (int x = 0; x < 5; x++) vD[x] = mk(vi[x], k == x);
  if (FAR)
    far_ghost(a.ph, a.w0, nrm[f], nrm[nf + f], nrm[2 * nf + f], vD, wg, qg, tg);
  else
    wall_ghost(a.ph, vD, wg, qg, tg);
  double acc = tb * tg.d;
#pragma unroll
  for (int e = 0; e < 5; e++) acc += wb[e] * wg[e].d + qb[e] * qg[e].d;
  atomicAdd(B.vb + k * a.ldv + ni, acc);
}

// the entries of vb, snb and volb that no pass writes: snb of every entry
// (the face pass writes the faces), vb and volb of the ghosts; and the value
// planes of the ghosts, as neither list need name all of them
__global__ void __launch_bounds__(256) k_adjb_clear(Blk b, long ldv, double *vb, double *snb, double *volb,
                                                    double *ws) {
  const long m = blockIdx.x * 256L + threadIdx.x;
  if (m >= b.nnn) return;
#pragma unroll
  for (int x = 0; x < 9; x++) snb[x * b.nnn + m] = 0.;
  if (b.real(b.id1 + (int)(m % b.nid), b.jd1 + (int)((m / b.nid) % (b.nijd / b.nid)), b.kd1 + (int)(m / b.nijd)))
    return;
#pragma unroll
  for (int e = 0; e < 5; e++) vb[e * ldv + b.npc + m] = 0.;
  volb[b.npc + m] = 0.;
  for (int p = 0; p < NVPLANE; p++) ws[p * b.nnn + m] = 0.;
}

__global__ void k_adj_zero(double *p, long cnt) {
  long i = blockIdx.x * 256L + threadIdx.x;
  if (i < cnt) p[i] = 0.;
}

// ---------------------------------------------------------------------------
// metric adjoint (norm.f90 half-diagonal cross products, svol.f90 volumes)

struct MArgs {
  Blk b;
  const double *x, *y, *z;
  double sg[3];
  double *xb, *yb, *zb;
};

// One node: the faces it is a corner of (four per direction), each with its
// metric sn = sg d1 x d2 (d1, d2 the half-diagonals P(pq) - P(0) and P(q) -
// P(p), p < q the face's own directions) and its part of the volumes, the
// face sum (P(0) + P(p) + P(q) + P(pq)) . sn with weight 1/12 in the cell
// below and -1/12 in the one above, transposed onto the node.  Every face is
// formed by its four corners instead of scattered to them: 60 operations
// against 24 atomic adds.
__global__ void __launch_bounds__(256) k_madj_nodes(MArgs M, const double *__restrict__ snb,
                                                    const double *__restrict__ volb) {
  const Blk &b = M.b;
  const long o = blockIdx.x * 256L + threadIdx.x, nnn = b.nnn;
  if (o >= nnn) return;
  const int nn[3] = {(int)b.nid, (int)(b.nijd / b.nid), (int)(nnn / b.nijd)};
  const int c[3] = {(int)(o % b.nid), (int)((o / b.nid) % nn[1]), (int)(o / b.nijd)};
  const double *P[3] = {M.x + b.npc, M.y + b.npc, M.z + b.npc};
  double nb[3] = {0., 0., 0.};
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int p = d == 0 ? 1 : 0, q = d == 2 ? 1 : 2;
    const long id = b.inc(d), ip = b.inc(p), iq = b.inc(q);
#pragma unroll
    for (int corner = 0; corner < 4; corner++) {  // the node is P(0), P(p), P(q), P(pq) of the face
      const int cp = corner & 1, cq = corner >> 1;
      const int fp = c[p] - cp, fq = c[q] - cq;
      if (fp < 0 || fq < 0 || fp >= nn[p] - 1 || fq >= nn[q] - 1) continue;
      const long f = o - cp * ip - cq * iq;
      double d1[3], d2[3], cs[3];
#pragma unroll
      for (int x = 0; x < 3; x++) {
        const double p0 = P[x][f], p1 = P[x][f + ip], p2 = P[x][f + iq], p3 = P[x][f + ip + iq];
        d1[x] = p3 - p0;
        d2[x] = p2 - p1;
        cs[x] = ((p0 + p1) + p2) + p3;
      }
      double fb = 0.;  // adjoint of the face sum
      if (c[d] > 0) fb += volb[b.npc + f - id];
      if (c[d] < nn[d] - 1) fb -= volb[b.npc + f];
      fb *= 0.25 / 3.;
      double tb[3];
#pragma unroll
      for (int x = 0; x < 3; x++) tb[x] = M.sg[d] * (snb[((long)x * 3 + d) * nnn + f] + fb * cs[x]);
      const double sgn = M.sg[d] * fb;
#pragma unroll
      for (int x = 0; x < 3; x++) {
        const int y = (x + 1) % 3, z = (x + 2) % 3;
        const double sn = d1[y] * d2[z] - d1[z] * d2[y];
        // d1b = d2 x tb on P(pq) - P(0); d2b = tb x d1 on P(q) - P(p)
        const double e = cp == cq ? d2[y] * tb[z] - d2[z] * tb[y] : tb[y] * d1[z] - tb[z] * d1[y];
        nb[x] += sgn * sn + (cq ? e : -e);
      }
    }
  }
  M.xb[o] = nb[0];
  M.yb[o] = nb[1];
  M.zb[o] = nb[2];
}

inline unsigned nblk(long n, int t) { return (unsigned)((n + t - 1) / t); }

int adj_setup(const char *what, const codens_block *cb, const codens_phys *cp, const codens_scheme *sc,
              const double *v, int64_t ldv, const double *sn, const double *vol, const double *winf, long nwall,
              const int64_t *wg, const int64_t *wi, long nfar, const int64_t *fg, const int64_t *fi,
              const double *fn, AdjArgs &a) {
  int rc = codens_check_block(cb, what);
  if (rc) return rc;
  if (!cp || !sc || !v || !sn || !vol || (nfar && (!fg || !fi || !fn || !winf)) || (nwall && (!wg || !wi)) ||
      ldv <= 0 || nwall < 0 || nfar < 0) {
    codens_set_error("%s: null or invalid argument", what);
    return CODENS_EINVAL;
  }
  if (sc->ilim != 0) {
    codens_set_error("%s: the adjoint covers unlimited MUSCL (ilim = 0) only", what);
    return CODENS_EINVAL;
  }
  a.b = make_blk(cb);
  a.ph.gam = cp->gam; a.ph.gam1 = cp->gam1; a.ph.pinfl = cp->pinfl; a.ph.pr = cp->pr; a.ph.cp = cp->cp;
  a.ph.usrey = 1. / cp->reynz; a.ph.asuth = 110.4 / cp->tnz; a.ph.iflu = cp->iflu;
  a.muscl = (double)sc->muscl; a.xk = sc->xk; a.ldv = (long)ldv;
  a.v = v; a.sn = sn; a.vol = vol; a.w0 = winf;
  a.vd = nullptr; a.snd = nullptr; a.vold = nullptr; a.wd = nullptr;
  return CODENS_OK;
}

template <typename T>
void forward_chain(const AdjArgs &a, long nwall, const int64_t *wg, const int64_t *wi, long nfar,
                   const int64_t *fg, const int64_t *fi, const double *fn, hipStream_t st) {
  const Blk &b = a.b;
  long ncell = (long)(b.i2 - b.i1) * (b.j2 - b.j1) * (b.k2 - b.k1);
  hipLaunchKernelGGL(k_adj_thermo<T>, dim3(nblk(ncell, 256)), dim3(256), 0, st, a);
  if (nwall) hipLaunchKernelGGL((k_adj_ghost<T, 0>), dim3(nblk(nwall, 256)), dim3(256), 0, st, a, nwall, wg, wi, fn);
  if (nfar) hipLaunchKernelGGL((k_adj_ghost<T, 1>), dim3(nblk(nfar, 256)), dim3(256), 0, st, a, nfar, fg, fi, fn);
  hipLaunchKernelGGL(k_adj_grad<T>, dim3(nblk(ncell, 256)), dim3(256), 0, st, a);
  if (nwall) hipLaunchKernelGGL(k_adj_tq_ghost<T>, dim3(nblk(nwall, 256)), dim3(256), 0, st, a, nwall, wg, wi);
  if (nfar) hipLaunchKernelGGL(k_adj_tq_ghost<T>, dim3(nblk(nfar, 256)), dim3(256), 0, st, a, nfar, fg, fi);
}

long nfaces(const Blk &b, int d) {
  return (long)(b.i2 - b.i1 + (d == 0)) * (b.j2 - b.j1 + (d == 1)) * (b.k2 - b.k1 + (d == 2));
}

}  // namespace

extern "C" int codens_adj_residual_jvp(const codens_block *cb, const codens_phys *cp, const codens_scheme *sc,
                                       const double *v, const double *vdot, int64_t ldv, const double *sn,
                                       const double *sndot, const double *vol, const double *voldot,
                                       const double *winf, int64_t nwall, const int64_t *wall_ghost,
                                       const int64_t *wall_inner, int64_t nfar, const int64_t *far_ghost,
                                       const int64_t *far_inner, const double *far_nrm, double *u, double *udot,
                                       void *stream) {
  const char *what = "codens_adj_residual_jvp";
  AdjArgs a;
  int rc = adj_setup(what, cb, cp, sc, v, ldv, sn, vol, winf, (long)nwall, wall_ghost, wall_inner, (long)nfar,
                     far_ghost, far_inner, far_nrm, a);
  if (rc) return rc;
  if (!vdot || !sndot || !voldot || !u || !udot) {
    codens_set_error("%s: null argument", what);
    return CODENS_EINVAL;
  }
  long nnn = a.b.nnn;
  double *ws = (double *)codens_workspace(sizeof(double) * 2 * NPLANE * nnn, 8);
  if (!ws) {
    codens_set_error("%s: workspace allocation failed", what);
    return CODENS_EHIP;
  }
  hipStream_t st = (hipStream_t)stream;
  a.ws = ws; a.wd = ws + NPLANE * nnn;
  a.vd = vdot; a.snd = sndot; a.vold = voldot;
  hipLaunchKernelGGL(k_adj_zero, dim3(nblk(2 * NPLANE * nnn, 256)), dim3(256), 0, st, ws, 2 * NPLANE * nnn);
  forward_chain<Dual>(a, nwall, wall_ghost, wall_inner, nfar, far_ghost, far_inner, far_nrm, st);
  for (int d = 0; d < 3; d++)
    hipLaunchKernelGGL(k_adj_faces<Dual>, dim3(nblk(nfaces(a.b, d), 256)), dim3(256), 0, st, a, d);
  long ncell = (long)(a.b.i2 - a.b.i1) * (a.b.j2 - a.b.j1) * (a.b.k2 - a.b.k1);
  hipLaunchKernelGGL(k_adj_gather<Dual>, dim3(nblk(ncell, 256)), dim3(256), 0, st, a, u, udot);
  return codens_check_launch(what);
}

extern "C" int codens_adj_residual_vjp(const codens_block *cb, const codens_phys *cp, const codens_scheme *sc,
                                       const double *v, int64_t ldv, const double *sn, const double *vol,
                                       const double *winf, int64_t nwall, const int64_t *wall_ghost,
                                       const int64_t *wall_inner, int64_t nfar, const int64_t *far_ghost,
                                       const int64_t *far_inner, const double *far_nrm, const double *ubar,
                                       double *vbar, double *snbar, double *volbar, void *stream) {
  const char *what = "codens_adj_residual_vjp";
  AdjArgs a;
  int rc = adj_setup(what, cb, cp, sc, v, ldv, sn, vol, winf, (long)nwall, wall_ghost, wall_inner, (long)nfar,
                     far_ghost, far_inner, far_nrm, a);
  if (rc) return rc;
  if (!ubar || !vbar || !snbar || !volbar) {
    codens_set_error("%s: null argument", what);
    return CODENS_EINVAL;
  }
  long nnn = a.b.nnn;
  double *ws = (double *)codens_workspace(sizeof(double) * (NVPLANE + NBPLANE) * nnn, 8);
  if (!ws) {
    codens_set_error("%s: workspace allocation failed", what);
    return CODENS_EHIP;
  }
  hipStream_t st = (hipStream_t)stream;
  a.ws = ws;
  AdjBar B{ws + NVPLANE * nnn, ubar, vbar, snbar, volbar};
  const Blk &b = a.b;
  const long ncell = (long)(b.i2 - b.i1) * (b.j2 - b.j1) * (b.k2 - b.k1);
  hipLaunchKernelGGL(k_adjb_clear, dim3(nblk(nnn, 256)), dim3(256), 0, st, b, (long)ldv, vbar, snbar, volbar, ws);
  forward_chain<double>(a, nwall, wall_ghost, wall_inner, nfar, far_ghost, far_inner, far_nrm, st);
  const unsigned nf0 = nblk(nfaces(b, 0), 128), nf1 = nblk(nfaces(b, 1), 128), nf2 = nblk(nfaces(b, 2), 128);
  hipLaunchKernelGGL(k_adjb_faces, dim3(nf0 + nf1 + nf2), dim3(128), 0, st, a, B, nf0, nf1);
  hipLaunchKernelGGL(k_adjb_tq, dim3(nblk(ncell, 256)), dim3(256), 0, st, a, B);
  if (nwall + nfar)
    hipLaunchKernelGGL(k_adjb_tq_ghost, dim3(nblk(nwall + nfar, 128)), dim3(128), 0, st, a, B, (long)nwall, wall_ghost,
                       wall_inner, (long)nfar, far_ghost, far_inner);
  hipLaunchKernelGGL(k_adjb_cells, dim3(nblk(ncell, 256)), dim3(256), 0, st, a, B);
  if (nwall)
    hipLaunchKernelGGL(k_adjb_ghost<0>, dim3(nblk(5 * nwall, 128)), dim3(128), 0, st, a, B, (long)nwall, wall_ghost,
                       wall_inner, far_nrm);
  if (nfar)
    hipLaunchKernelGGL(k_adjb_ghost<1>, dim3(nblk(5 * nfar, 128)), dim3(128), 0, st, a, B, (long)nfar, far_ghost,
                       far_inner, far_nrm);
  return codens_check_launch(what);
}

extern "C" int codens_adj_metric_vjp(const codens_block *cb, const double *x, const double *y, const double *z,
                                     const double *sg3, const double *snbar, const double *volbar, double *xbar,
                                     double *ybar, double *zbar, void *stream) {
  const char *what = "codens_adj_metric_vjp";
  int rc = codens_check_block(cb, what);
  if (rc) return rc;
  if (!x || !y || !z || !sg3 || !snbar || !volbar || !xbar || !ybar || !zbar) {
    codens_set_error("%s: null argument", what);
    return CODENS_EINVAL;
  }
  MArgs M;
  M.b = make_blk(cb);
  M.x = x; M.y = y; M.z = z;
  for (int d = 0; d < 3; d++) M.sg[d] = sg3[d];
  M.xb = xbar; M.yb = ybar; M.zb = zbar;
  hipLaunchKernelGGL(k_madj_nodes, dim3(nblk(M.b.nnn, 256)), dim3(256), 0, (hipStream_t)stream, M, snbar, volbar);
  return codens_check_launch(what);
}
