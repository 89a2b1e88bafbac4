// Matrix-free point-Jacobi implicit phase (implimf_3d) on gfx950.
//
// implimf_3d.f90 keeps nine flux-increment arrays dF = F(v+d) - F(v) between
// sub-iterations.  Here every sub-iteration is one kernel that re-derives dF
// of a cell and of its six neighbours from v and the previous increment d:
// per sub-iteration a cell moves u, v, d_old, sn, diag, coefe and d_new through
// HBM (33 doubles) instead of also streaming nine dF arrays in and out.  In
// FP64, on all but small blocks, two sub-iterations share that pass
// (k_impl_sweep2).
// Because every read of d and dF in a sub-iteration sees the previous
// sub-iteration's values (implimf_3d.f90:230-431), the cells are independent
// and any traversal order gives the reference's result.
#include "common.hpp"

#include <algorithm>

#include <array>
#include <cmath>
#include <map>
#include <mutex>

using namespace codens;

// Increment buffer view: element (e, n) at p[e*ld + n - off].  T = double
// for the FP64 phase, float for the FP32 defect-correction form.
template <typename T>
struct TView {
  T *p;
  long ld, off;
  __device__ inline T &at(int e, long n) const { return p[e * ld + n - off]; }
};
using DView = TView<double>;

// sn(m, d, c) of a block's metric slice in either precision
template <typename T>
__device__ inline T snt(const T *__restrict__ sn, long nnn, long m, int d, int c) {
  return sn[((long)c * 3 + d) * nnn + m];
}

template <typename T>
struct DFluxT {  // mass-flux increment (d of rho u, rho v, rho w) and dF
  T mx, my, mz, xx, xy, xz, yy, yz, zz, ex, ey, ez;
};
using DFlux = DFluxT<double>;

// implimf_3d.f90:434-465 for one cell: dF = F(v + d) - F(v), p(v) from the EOS
// as zpres.f90:72-73 computes it, as the 14-vector of the sub-iterations: the
// mass-flux increments (d of rho u, rho v, rho w), the nine dF (xx xy xz yy yz
// zz, energy x y z), d of rho and of rho E.  The velocities are formed with one
// reciprocal of each density instead of the reference's divisions (about 1e-16
// relative per value; the sub-iteration result moves by ~3e-14).
//
// Here and in the face sums the fused multiply-adds are written out, so that
// every kernel that runs sub-iterations rounds alike and gives the same bits:
// left to the compiler, the all-blocks kernel fused other products of the k
// faces than the per-block one.
__device__ __forceinline__ void dflux_q(const Phys &ph, const double V[5], const double D[5], double q[14]) {
#pragma clang fp contract(off)
  const double w0 = V[0] + D[0], w1 = V[1] + D[1], w2 = V[2] + D[2], w3 = V[3] + D[3], w4 = V[4] + D[4];
  const double ri = 1. / w0, r0 = 1. / V[0];
  const double u = w1 * ri, v = w2 * ri, w = w3 * ri;
  const double kn = fma(w, w, fma(u, u, v * v));
  const double xn = fma(-(0.5 * w0), kn, w4) - ph.pinfl, pn = ph.gam1 * xn;
  const double a = V[1] * r0, b = V[2] * r0, c = V[3] * r0;
  const double k0 = fma(V[3], c, fma(V[1], a, V[2] * b));
  const double x0 = fma(-0.5, k0, V[4]) - ph.pinfl, p = ph.gam1 * x0;
  const double e5 = fma(ph.gam1, x0, V[4]) - ph.pinfl, en = fma(ph.gam1, xn, w4) - ph.pinfl;
  const double wu = w0 * u, wv = w0 * v;
  q[0] = D[1]; q[1] = D[2]; q[2] = D[3];
  q[3] = fma(w0, u * u, pn) - fma(V[1], a, p);
  q[4] = fma(wu, v, -(V[2] * a));
  q[5] = fma(wu, w, -(V[3] * a));
  q[6] = fma(w0, v * v, pn) - fma(V[2], b, p);
  q[7] = fma(wv, w, -(V[3] * b));
  q[8] = fma(w0, w * w, pn) - fma(V[3], c, p);
  q[9] = fma(u, en, -(e5 * a));
  q[10] = fma(v, en, -(e5 * b));
  q[11] = fma(w, en, -(e5 * c));
  q[12] = D[0];
  q[13] = D[4];
}

// The same increment dF = F(v + d) - F(v) in difference form, for the FP32
// sub-iterations: every term is a product with a change (dm - q drho)/(rho +
// drho) of a velocity, of the kinetic energy or of the pressure, so that its
// rounding is relative to |d|.  The form above subtracts two fluxes of size
// |F|, whose rounding in FP32 (6e-8 |F|) does not shrink with d and would
// hold the FP64 residual of the defect correction at about 1e-7 of its
// start.  Algebraically the same increment.
template <typename T>
__device__ inline DFluxT<T> dflux_delta(const Phys &ph, const T V[5], const T D[5]) {
  // no FMA contraction: the same rounding in every tile shape's kernel
#pragma clang fp contract(off)
  const T gam1 = (T)ph.gam1, pinfl = (T)ph.pinfl;
  T r0 = T(1) / V[0], rn = T(1) / (V[0] + D[0]);
  T u = V[1] * r0, v = V[2] * r0, w = V[3] * r0;
  T du = (D[1] - u * D[0]) * rn, dv = (D[2] - v * D[0]) * rn, dw = (D[3] - w * D[0]) * rn;
  T rho1 = V[0] + D[0];
  T q2 = u * u + v * v + w * w;
  T dq2 = T(2) * (u * du + v * dv + w * dw) + (du * du + dv * dv + dw * dw);
  T dk = T(0.5) * (D[0] * q2 + rho1 * dq2);                // change of rho |u|^2 / 2
  T p = gam1 * (V[4] - T(0.5) * V[0] * q2 - pinfl);
  T dp = gam1 * (D[4] - dk);
  // change of rho q_a q_b
  auto dprod = [&](T qa, T qb, T dqa, T dqb) {
#pragma clang fp contract(off)
    return D[0] * qa * qb + rho1 * (qa * dqb + dqa * qb + dqa * dqb);
  };
  T h0 = V[4] + p - pinfl, dh = D[4] + dp;                  // E + p - pinfl and its change
  DFluxT<T> r;
  r.mx = D[1]; r.my = D[2]; r.mz = D[3];
  r.xx = dprod(u, u, du, du) + dp;
  r.xy = dprod(u, v, du, dv);
  r.xz = dprod(u, w, du, dw);
  r.yy = dprod(v, v, dv, dv) + dp;
  r.yz = dprod(v, w, dv, dw);
  r.zz = dprod(w, w, dw, dw) + dp;
  r.ex = dh * (u + du) + h0 * du;
  r.ey = dh * (v + dv) + h0 * dv;
  r.ez = dh * (w + dw) + h0 * dw;
  return r;
}

// implimf_eu.f90:289-312 for one cell: dF from the momenta with
// wi1 = 1/(rho + d1), the base flux with the caller's pressure p, and the z
// energy increment without its w factor, as the reference has it.
__device__ inline DFlux dflux_eu(const Phys &ph, const double V[5], const double D[5], double p) {
  const double gam1 = ph.gam1, pinfl = ph.pinfl;
  double wi1 = 1. / (V[0] + D[0]);
  double ui = V[1] + D[1], vi = V[2] + D[2], wi = V[3] + D[3], wi5 = V[4] + D[4];
  double pres = gam1 * (wi5 - .5 * wi1 * (ui * ui + vi * vi + wi * wi) - pinfl);
  double norm = 1. / V[0];
  double a = V[1] * norm, bb = V[2] * norm, c = V[3] * norm;
  double fxx = V[1] * a + p, fxy = V[2] * a, fxz = V[3] * a;
  double fyy = V[2] * bb + p, fyz = V[3] * bb, fzz = V[3] * c + p;
  double e5 = V[4] + p - pinfl;
  double fex = e5 * V[1] * norm, fey = e5 * V[2] * norm, fez = e5 * V[3] * norm;
  double h = wi5 + pres - pinfl;
  DFlux r;
  r.mx = D[1]; r.my = D[2]; r.mz = D[3];
  r.xx = wi1 * (ui * ui) + pres - fxx;
  r.xy = wi1 * ui * vi - fxy;
  r.xz = wi1 * ui * wi - fxz;
  r.ex = wi1 * ui * h - fex;
  r.yy = wi1 * (vi * vi) + pres - fyy;
  r.yz = wi1 * vi * wi - fyz;
  r.ey = wi1 * vi * h - fey;
  r.zz = wi1 * (wi * wi) + pres - fzz;
  r.ez = wi1 * h - fez;
  return r;
}

#define CELL3(b) CELL3_AT(b, xcd_block())
// the same, for the tile XB of a block's own grid
#define CELL3_AT(b, XB)                              \
  int c[3];                                          \
  const dim3 xb = (XB);                              \
  c[0] = (b).i1 + xb.x * TX + threadIdx.x;     \
  c[1] = (b).j1 + xb.y * TY + threadIdx.y;     \
  c[2] = (b).k1 + xb.z;                        \
  if (c[0] >= (b).i2 || c[1] >= (b).j2) return;

// implimf_3d.f90:113-224: spectral-radius coefficients of the faces and the
// diagonal; coefe[d] holds the low face of every real cell.  A workgroup
// owns a TX x TY tile of real cells and marches a slab of k-planes (of
// coef_slab's depth, CK_KS in the all-blocks launch), so that each face is
// evaluated once.  Per plane, the velocity, sound speed, rv and
// volume of every cell of the tile and of its 1-cell ring (i0-1..i0+TX,
// j0-1..j0+TY) go to LDS; each thread evaluates the low i and j faces of its
// cell, the ring's threads the tile's high faces, and the k face below its
// cell from its own column's previous plane.  A face's coefficient is one
// expression of its two cells whichever tile evaluates it:
// 0.5 (|V.S| + |S| c) + (rv_lo + rv_hi) |S|^2 / (vol_lo + vol_hi), with V
// and c averaged (high + low) / 2 and no contraction.  Velocities and rv use
// one reciprocal of each density (the reference divides each time; the
// coefficients move by ~1e-16 relative).  A cell's diagonal adds its six
// faces in the order of implimf_3d.f90:206-215 (i low, i high, j low, j high,
// k low, k high) and is complete once the next plane has evaluated the k face
// above it.
//
// Bound by memory: on 200 x 120 x 100 117 us, 3.8 TB/s of the 23 planes that it
// cannot do without, where loads one after another behind the divisions that
// used the first of them, per-thread 64-bit addresses (127 registers) and
// slabs of 8 in two rounds, the second half empty, took 133 us; 75 x 61 x 43
// 19 -> 14 us.  With the FP32 copies 147 us on 256 x 128 x 64, where the
// coefficients in FP64 (90 us) and a pass that rounded them and the operands
// (119 us) read them twice.  Blocks of 2 to 4 cells in i leave nearly all lanes
// idle and lose by it: with one sub-iteration 2 x 300 x 200 178 us, 157 in two
// passes, 4 x 64 x 400 89 and 90.
constexpr int CK_KS = 8;  // planes per workgroup in the all-blocks launch
constexpr int CK_PL = (TX + 2) * (TY + 2);

struct CoefCell {  // the per-cell operands of a face coefficient
  double u, v, w, c, rv, vol;
};

// what they are made of, at byte offset off of the plane whose first storage
// entry is n0
struct CoefRaw {
  double r, m1, m2, m3, c, mu, mut, vol;
};

__device__ __forceinline__ CoefRaw coef_load(const double *__restrict__ v, long ldv, const double *__restrict__ mu,
                                             const double *__restrict__ mut, const double *__restrict__ vol,
                                             const double *__restrict__ cson, long n0, unsigned off) {
  return CoefRaw{ldp(v + n0, off),    ldp(v + (ldv + n0), off), ldp(v + (2 * ldv + n0), off),
                 ldp(v + (3 * ldv + n0), off), ldp(cson + n0, off), ldp(mu + n0, off),
                 ldp(mut + n0, off),  ldp(vol + n0, off)};
}

__device__ __forceinline__ CoefCell coef_cell(const Phys &ph, const CoefRaw &x, bool real) {
  const double r = 1.0 / x.r;
  return CoefCell{x.m1 * r, x.m2 * r, x.m3 * r, x.c,
                  real ? ph.gam * (x.mu / ph.pr + x.mut / ph.prt) * r : 0., x.vol};
}

// coefficient of the face between cells lo and hi (normal s of the face)
__device__ __forceinline__ double coef_face(const CoefCell &hi, const CoefCell &lo, double s1, double s2, double s3) {
#pragma clang fp contract(off)
  double cnds = s1 * s1 + s2 * s2 + s3 * s3;
  double uu = 0.5 * (hi.u + lo.u), vv = 0.5 * (hi.v + lo.v), ww = 0.5 * (hi.w + lo.w);
  double cc = 0.5 * (hi.c + lo.c), rsum = hi.rv + lo.rv, vsum = hi.vol + lo.vol;
  double vnf = uu * s1 + vv * s2 + ww * s3;
  return 0.5 * (fabs(vnf) + sqrt(cnds) * cc) + rsum * cnds / vsum;
}

// LDS of one workgroup: the plane's cell operands and the i and j face
// coefficients of the tile
struct CoefLds {
  double L[6][CK_PL];
  double CI[(TX + 1) * TY], CJ[TX * (TY + 1)];
};

// FP32 copies of the sub-iterations' operands, written next to the
// coefficients (block-local planes of nnn)
struct F32Copies {
  const double *u, *ff;  // ff: null if not used
  float *vF, *uF, *fF, *snF;
};

// the tile xb (x, y: TX x TY columns, z: slab of ks planes) of block b.  T =
// float rounds the coefficients and copies the operands to FP32 on the way:
// they are the ones that this pass reads, u excepted.
template <typename T>
__device__ __forceinline__ void coef_tiled_body(const Blk &b, dim3 xb, const Phys &ph, const double *__restrict__ v,
                                                long ldv, const double *__restrict__ mu,
                                                const double *__restrict__ mut, const double *__restrict__ dt,
                                                const double *__restrict__ vol, const double *__restrict__ cson,
                                                const double *__restrict__ sn, double dtpas, int kfmg,
                                                T *__restrict__ coefe, T *__restrict__ diag, int ks, CoefLds &S,
                                                const F32Copies &F) {
#pragma clang fp contract(off)
  auto &L = S.L;
  double *CI = S.CI, *CJ = S.CJ;
  const int tx = threadIdx.x, ty = threadIdx.y, t = tx + TX * ty;
  const int i0 = b.i1 + xb.x * TX, j0 = b.j1 + xb.y * TY;
  const int kb = b.k1 + xb.z * ks, ke = min(kb + ks, b.k2);
  const int i = i0 + tx, j = j0 + ty;
  // own: a real cell; load: a real cell or the ghost past the block's high
  // i or j end, whose faces with the last real cells this thread evaluates
  // when the tile is partial (it is then inside the tile)
  const bool own = i < b.i2 && j < b.j2, load = i <= b.i2 && j <= b.j2;
  // ring cell of this thread (t < 2 TX + 2 TY): columns i0-1, i0+TX, rows
  // j0-1, j0+TY, loaded where it lies in the block's storage
  int ri = 0, rj = 0, rslot = 0;
  const bool ring = t < 2 * TX + 2 * TY;
  if (ring) {
    int rx, ry;
    if (t < TX) { ri = i0 + t; rj = j0 - 1; rx = t + 1; ry = 0; }
    else if (t < 2 * TX) { ri = i0 + t - TX; rj = j0 + TY; rx = t - TX + 1; ry = TY + 1; }
    else if (t < 2 * TX + TY) { ri = i0 - 1; rj = j0 + t - 2 * TX; rx = 0; ry = t - 2 * TX + 1; }
    else { ri = i0 + TX; rj = j0 + t - 2 * TX - TY; rx = TX + 1; ry = t - 2 * TX - TY + 1; }
    rslot = ry * (TX + 2) + rx;
  }
  const int id2 = b.id1 + (int)b.nid - 1, jd2 = b.jd1 + (int)(b.nijd / b.nid) - 1;
  const bool rneed = ring && ri >= b.id1 && ri <= id2 && rj >= b.jd1 && rj <= jd2;
  const int slot = (ty + 1) * (TX + 2) + (tx + 1);
  // byte offsets in a plane of the own cell (clamped to the cells whose faces
  // are evaluated), the ring cell and the ring thread's high face; the
  // index in the block of the plane's first cell
  auto plane = [&](int x, int y) { return ((unsigned)(x - b.id1) + (unsigned)(y - b.jd1) * (unsigned)b.nid) * 8u; };
  const unsigned po = plane(min(i, b.i2), min(j, b.j2)), pr = rneed ? plane(ri, rj) : 0u;
  long mk = (long)(kb - 1 - b.kd1) * b.nijd;
  auto sn3 = [&](int d, unsigned off, double s[3]) {
#pragma unroll
    for (int c = 0; c < 3; c++) s[c] = ldp(sn + ((3 * c + d) * b.nnn + mk), off);
  };
  CoefCell below{}, cur{};
  below = coef_cell(ph, coef_load(v, ldv, mu, mut, vol, cson, b.npc + mk, po), kb > b.k1);
  double part = 0.;  // the diagonal of the cell below, all but its k high face
  // the tile's high face of a ring thread: i face at i0+TX of row j0+t
  // (t < TY), j face at j0+TY of column i0+t-TY (TY <= t < TY + TX), where it
  // bounds a real cell of the tile; its LDS slot and CI/CJ entry
  int hdir = -1, hs = 0, hc = 0, hfi = 0, hfj = 0;
  if (t < TY) {
    hfj = j0 + t; hfi = i0 + TX;
    if (hfi <= b.i2 && hfj < b.j2) { hdir = 0; hs = (t + 1) * (TX + 2) + TX + 1; hc = t * (TX + 1) + TX; }
  } else if (t < TY + TX) {
    hfi = i0 + t - TY; hfj = j0 + TY;
    if (hfj <= b.j2 && hfi < b.i2) { hdir = 1; hs = (TY + 1) * (TX + 2) + (t - TY) + 1; hc = TY * TX + (t - TY); }
  }
  // the low i face of this thread's cell where it bounds a real cell (rows
  // j < j2, up to the block's high boundary face i = i2), the low j face
  // likewise
  const bool fi = i <= b.i2 && j < b.j2, fj = i < b.i2 && j <= b.j2;
  const unsigned pf = hdir >= 0 ? plane(hfi, hfj) : 0u;
  const double *sf = sn + (hdir == 1 ? b.nnn : 0L) + pf / 8;  // the high face's normal in plane 0
  for (int k = kb; k <= ke; k++) {
    const bool top = k == ke;  // the k face above the slab's last plane only
    mk += b.nijd;
    // every global load of the plane, issued before any is used so that their
    // latencies overlap (offsets are clamped into the plane, so that all
    // threads load; what a thread does not need it does not use)
    const long nk = b.npc + mk;
    const CoefRaw xo = coef_load(v, ldv, mu, mut, vol, cson, nk, po);
    CoefRaw xr{1., 0., 0., 0., 0., 0., 0., 0.};
    double sk[3], si[3] = {0., 0., 0.}, sj[3] = {0., 0., 0.}, sh[3] = {0., 0., 0.}, dtn = 1.;
    sn3(2, po, sk);
    if (!top) {
      sn3(0, po, si);
      sn3(1, po, sj);
      dtn = ldp(dt + nk, po);
      if (ring) {
        xr = coef_load(v, ldv, mu, mut, vol, cson, nk, pr);
#pragma unroll
        for (int c = 0; c < 3; c++) sh[c] = sf[(3 * c * b.nnn + mk)];
      }
    }
    cur = coef_cell(ph, xo, own && k < b.k2);
    const bool rl = !top && rneed;
    const CoefCell rq = coef_cell(ph, xr, b.real(ri, rj, k));
    if (!top) {
      if (load) {
        L[0][slot] = cur.u; L[1][slot] = cur.v; L[2][slot] = cur.w;
        L[3][slot] = cur.c; L[4][slot] = cur.rv; L[5][slot] = cur.vol;
      }
      if (rl) {
        L[0][rslot] = rq.u; L[1][rslot] = rq.v; L[2][rslot] = rq.w;
        L[3][rslot] = rq.c; L[4][rslot] = rq.rv; L[5][rslot] = rq.vol;
      }
    }
    lds_sync();
    constexpr bool F32 = sizeof(T) == sizeof(float);
    double cv[F32 ? 5 : 1], cu[F32 ? 5 : 1], cf[F32 ? 5 : 1];
    if constexpr (F32) {  // their latency overlaps the faces
      if (own && !top) {
#pragma unroll
        for (int e = 0; e < 5; e++) {
          cv[e] = ldp(v + (e * ldv + nk), po);
          cu[e] = ldp(F.u + (e * ldv + nk), po);
          if (F.ff) cf[e] = ldp(F.ff + (e * ldv + nk), po);
        }
      }
    }
    double ckl = 0.;
    if (own) {
      ckl = coef_face(cur, below, sk[0], sk[1], sk[2]);
      if (k > kb) {  // the cell below is complete
        double dg = part + ckl;
        if (kfmg == 3) dg = dg + 1.5 * below.vol / dtpas;
        *gp(diag + (mk - b.nijd), po / (8 / sizeof(T))) = (T)dg;
      }
    }
    if (!top) {
      auto lds = [&](int s) {
        CoefCell q;
        q.u = L[0][s]; q.v = L[1][s]; q.w = L[2][s]; q.c = L[3][s]; q.rv = L[4][s]; q.vol = L[5][s];
        return q;
      };
      if (fi) CI[ty * (TX + 1) + tx] = coef_face(lds(slot), lds(slot - 1), si[0], si[1], si[2]);
      if (fj) CJ[ty * TX + tx] = coef_face(lds(slot), lds(slot - (TX + 2)), sj[0], sj[1], sj[2]);
      if (hdir == 0) CI[hc] = coef_face(lds(hs), lds(hs - 1), sh[0], sh[1], sh[2]);
      else if (hdir == 1) CJ[hc] = coef_face(lds(hs), lds(hs - (TX + 2)), sh[0], sh[1], sh[2]);
    }
    if constexpr (F32) {
      auto put_sn = [&](int d, unsigned off, const double x[3]) {
#pragma unroll
        for (int c = 0; c < 3; c++) *gp(F.snF + ((3 * c + d) * b.nnn + mk), off / 2) = (float)x[c];
      };
      // the low faces of real cells and the block's high boundary faces
      if (own && (!top || ke == b.k2)) put_sn(2, po, sk);
      if (!top && fi) put_sn(0, po, si);
      if (!top && fj) put_sn(1, po, sj);
      if (!top && hdir == 0 && hfi == b.i2) put_sn(0, pf, sh);
      if (!top && hdir == 1 && hfj == b.j2) put_sn(1, pf, sh);
    }
    lds_sync();
    if constexpr (F32) {
      if (own && !top) {
#pragma unroll
        for (int e = 0; e < 5; e++) {
          *gp(F.vF + (e * b.nnn + mk), po / 2) = (float)cv[e];
          *gp(F.uF + (e * b.nnn + mk), po / 2) = (float)cu[e];
          if (F.ff) *gp(F.fF + (e * b.nnn + mk), po / 2) = (float)cf[e];
        }
      }
    }
    if (!top && own) {
      double c0 = CI[ty * (TX + 1) + tx], c1 = CI[ty * (TX + 1) + tx + 1];
      double c2 = CJ[ty * TX + tx], c3 = CJ[(ty + 1) * TX + tx];
      const unsigned pt = po / (8 / sizeof(T));
      *gp(coefe + mk, pt) = (T)c0;
      *gp(coefe + (b.nnn + mk), pt) = (T)c2;
      *gp(coefe + (2 * b.nnn + mk), pt) = (T)ckl;
      part = cur.vol / dtn;
      part = part + c0 + c1 + c2 + c3 + ckl;
    }
    below = cur;
  }
}

template <typename T>
__global__ void __launch_bounds__(TX *TY) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_impl_coef_tiled(Blk b, Phys ph, const double *__restrict__ v, long ldv,
                                                            const double *__restrict__ mu,
                                                            const double *__restrict__ mut,
                                                            const double *__restrict__ dt,
                                                            const double *__restrict__ vol,
                                                            const double *__restrict__ cson,
                                                            const double *__restrict__ sn, double dtpas, int kfmg,
                                                            T *__restrict__ coefe, T *__restrict__ diag, int ks,
                                                            F32Copies F) {
  __shared__ CoefLds S;
  coef_tiled_body<T>(b, xcd_block(), ph, v, ldv, mu, mut, dt, vol, cson, sn, dtpas, kfmg, coefe, diag, ks, S, F);
}

// The next slab depth after x with fewer slabs in nz planes (of the depths with
// the same number of slabs the smallest takes the fewest steps, and there are
// at most 2 sqrt(nz) numbers), nz + 1 after the last
static int next_slab(int nz, int x) {
  const int slabs = (nz + x - 1) / x;
  return slabs > 1 ? (nz + slabs - 2) / (slabs - 1) : nz + 1;
}

// Slab depth of k_impl_coef_tiled on the tiles g.x x g.y: of four workgroups
// per compute unit, the fewest steps over their rounds (a slab of ks planes
// takes ks + 1)
static int coef_slab(const Blk &b, dim3 g) {
  const int nz = b.k2 - b.k1, places = codens_resident_workgroups(4);
  int ks = 1;
  long best = 0;
  for (int x = 1; x <= nz; x = next_slab(nz, x)) {
    const long c = ((long)g.x * g.y * ((nz + x - 1) / x) + places - 1) / places * (x + 1);
    if (x == 1 || c < best) { ks = x; best = c; }
  }
  return ks;
}

// implimf_eu.f90:124-170: coefficients of the Euler implicit phase,
// coefe = 0.5 |V.S| + |S| c and diag = vol (fact + 1/dt) + sum of the face
// coefficients, direction by direction; fact = 1.5/dt1min when kfmg = 3.
__global__ void __launch_bounds__(TX *TY) k_impl_coef_eu(Blk b, const double *__restrict__ v, long ldv,
                                                         const double *__restrict__ dt,
                                                         const double *__restrict__ vol,
                                                         const double *__restrict__ cson,
                                                         const double *__restrict__ sn, double fact,
                                                         double *__restrict__ coefe, double *__restrict__ diag) {
  CELL3(b)
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc;
  double norm = 1. / v[n];
  double u0 = v[ldv + n] * norm, v0 = v[2 * ldv + n] * norm, w0 = v[3 * ldv + n] * norm;
  double dg = vol[n] * (fact + 1. / dt[n]);
#pragma unroll
  for (int d = 0; d < 3; d++) {
    long inc = b.inc(d);
    double cf[2];
#pragma unroll
    for (int side = 0; side < 2; side++) {
      long nn = side == 0 ? n - inc : n + inc;
      long mf = side == 0 ? m : m + inc;
      double s1 = snv(sn, b.nnn, mf, d, 0), s2 = snv(sn, b.nnn, mf, d, 1), s3 = snv(sn, b.nnn, mf, d, 2);
      double cnds = s1 * s1 + s2 * s2 + s3 * s3;
      double norm1 = 1. / v[nn];
      double un = v[ldv + nn] * norm1, vn_ = v[2 * ldv + nn] * norm1, wn = v[3 * ldv + nn] * norm1;
      double uu, vv, ww, cc;
      if (side == 0) {  // face m: cells n (own) and n-inc
        uu = 0.5 * (u0 + un); vv = 0.5 * (v0 + vn_); ww = 0.5 * (w0 + wn); cc = 0.5 * (cson[n] + cson[nn]);
      } else {          // face m+inc: cells n+inc and n (own)
        uu = 0.5 * (un + u0); vv = 0.5 * (vn_ + v0); ww = 0.5 * (wn + w0); cc = 0.5 * (cson[nn] + cson[n]);
      }
      cf[side] = 0.5 * fabs(uu * s1 + vv * s2 + ww * s3) + sqrt(cnds) * cc;
    }
    coefe[d * b.nnn + m] = cf[0];
    dg = dg + cf[0] + cf[1];
  }
  diag[m] = dg;
}

// ---------------------------------------------------------------------------
// Tiled sub-iteration.  A workgroup owns an SW_TX x SW_TY column tile of real
// cells over SW_KS planes and marches k: the 14-vector q of a cell (mass-flux
// increments d2..d4, the nine dF, d1, d5) is formed once per sweep and kept
// in LDS for the i/j neighbours of its plane and in registers for the k
// neighbours; the k face term is carried from one plane to the next.
// LDS: 14 x (SW_TY+2) x (SW_TX+2) doubles = 44,352 bytes.  A 64 x 4 tile of
// 256 threads runs two workgroups per CU at its ~237 VGPRs (one workgroup
// waits at its plane barrier while the other computes): 125.6 us on the
// 2.1M-cell block against 133.1 for 64 x 8, despite its larger halo.
#ifndef CODENS_SW_TY
#define CODENS_SW_TY 4
#endif
#ifndef CODENS_SW_KS
#define CODENS_SW_KS 8
#endif
constexpr int SW_TX = 64, SW_TY = CODENS_SW_TY, SW_KS = CODENS_SW_KS;
static_assert(2 * SW_TX + 2 * SW_TY <= SW_TX * SW_TY, "one halo cell per thread at most");
constexpr int SW_HALO = 2 * SW_TX + 2 * SW_TY;

template <typename T>
struct Q14T {
  T q[14];
};
using Q14 = Q14T<double>;

template <typename T>
__device__ inline void q_set(const DFluxT<T> &F, const T D[5], Q14T<T> &Q) {
  Q.q[0] = F.mx; Q.q[1] = F.my; Q.q[2] = F.mz;
  Q.q[3] = F.xx; Q.q[4] = F.xy; Q.q[5] = F.xz; Q.q[6] = F.yy; Q.q[7] = F.yz; Q.q[8] = F.zz;
  Q.q[9] = F.ex; Q.q[10] = F.ey; Q.q[11] = F.ez;
  Q.q[12] = D[0]; Q.q[13] = D[4];
}

// the 14-vector of a cell: the reference's form in FP64, the difference form
// in FP32, implimf_eu's own flux increments (with the caller's p)
template <bool EU, typename T>
__device__ inline void q_form(const Phys &ph, const T V[5], const T D[5], double p, Q14T<T> &Q) {
  if constexpr (EU) q_set<T>(dflux_eu(ph, V, D, p), D, Q);
  else if constexpr (sizeof(T) == sizeof(float)) q_set<T>(dflux_delta<T>(ph, V, D), D, Q);
  else dflux_q(ph, V, D, Q.q);
}

template <bool EU, typename T, class DIN>
__device__ inline void q_model(const Phys &ph, const T *__restrict__ v, long ldv, const DIN &d,
                               const double *__restrict__ ps, long n, Q14T<T> &Q) {
  T V[5], D[5];
#pragma unroll
  for (int e = 0; e < 5; e++) {
    V[e] = v[e * ldv + n];
    D[e] = d.at(e, n);
  }
  q_form<EU, T>(ph, V, D, EU ? ps[n] : 0., Q);
}

template <typename T>
__device__ inline void q_zero(Q14T<T> &Q) {
#pragma unroll
  for (int c = 0; c < 14; c++) Q.q[c] = T(0);
}

// The same 14-vector in two phases, so that the loads of several cells can
// be in flight together: the inputs of a cell (zero for a cell outside the
// real region), then q from them.
template <typename T>
struct VD {
  T V[5], D[5];
  double p;
};

template <bool EU, typename T, class DIN>
__device__ inline void vd_load(const T *__restrict__ v, long ldv, const DIN &d, const double *__restrict__ ps,
                               long n, bool real, VD<T> &x) {
#pragma unroll
  for (int e = 0; e < 5; e++) {
    x.V[e] = real ? v[e * ldv + n] : T(1);
    x.D[e] = real ? d.at(e, n) : T(0);
  }
  x.p = (EU && real) ? ps[n] : 0.;
}

template <bool EU, typename T>
__device__ inline void vd_q(const Phys &ph, const VD<T> &x, bool real, Q14T<T> &Q) {
  if (!real) {
    q_zero(Q);
    return;
  }
  q_form<EU, T>(ph, x.V, x.D, x.p, Q);
}

// d of component e from the 14-vector
template <typename T>
__device__ inline T q_d(const T *q, int e) {
  return e == 0 ? q[12] : (e == 4 ? q[13] : q[e - 1]);
}

__device__ __forceinline__ double fma_t(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return fmaf(a, b, c); }

// Twice the face term tn (implimf_3d.f90:276-292), component by component, q
// of the other cell taken by get(c).  The half is exact and goes into the fused
// multiply-add that uses the term.
__host__ __device__ constexpr int tn_comp(int e, int x) {
  constexpr int C[5][3] = {{0, 1, 2}, {3, 4, 5}, {4, 6, 7}, {5, 7, 8}, {9, 10, 11}};
  return C[e][x];
}
template <typename T, class Get>
__device__ __forceinline__ void tn2_fma(const T A[14], const T s[3], T tn[5], Get get) {
#pragma clang fp contract(off)
  T x[12];
#pragma unroll
  for (int c = 0; c < 12; c++) x[c] = A[c] + get(c);
#pragma unroll
  for (int e = 0; e < 5; e++)
    tn[e] = fma_t(x[tn_comp(e, 2)], s[2], fma_t(x[tn_comp(e, 0)], s[0], x[tn_comp(e, 1)] * s[1]));
}

// First sub-iteration: d and dF are zero, so d = -(u (+ff)) / diag.
template <typename T>
__device__ __forceinline__ void sweep1_body(const Blk &b, dim3 tile, int ityprk, const T *__restrict__ u,
                                            const T *__restrict__ ff, long ldv, const T *__restrict__ diag,
                                            const TView<T> &dnew) {
  CELL3_AT(b, tile)
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc;
  T dg = diag[m];
#pragma unroll
  for (int e = 0; e < 5; e++) {
    T r = ityprk == 0 ? -u[e * ldv + n] : -u[e * ldv + n] - ff[e * ldv + n];
    dnew.at(e, n) = r / dg;
  }
}

template <typename T>
__global__ void __launch_bounds__(TX *TY) k_impl_sweep1(Blk b, int ityprk, const T *__restrict__ u,
                                                        const T *__restrict__ ff, long ldv,
                                                        const T *__restrict__ diag, TView<T> dnew) {
  sweep1_body<T>(b, xcd_block(), ityprk, u, ff, ldv, diag, dnew);
}

constexpr int SW_PL = (SW_TY + 2) * (SW_TX + 2);  // LDS plane stride between the 14 components

// twice the term of the face between the LDS cells a (own side) and o (other
// side), components read straight from LDS
template <int P, typename T>
__device__ __forceinline__ T lds_tn2(const T *a, const T *o, int e, const T s[3]) {
#pragma clang fp contract(off)
  const int x = tn_comp(e, 0) * P, y = tn_comp(e, 1) * P, z = tn_comp(e, 2) * P;
  return fma_t(a[z] + o[z], s[2], fma_t(a[x] + o[x], s[0], (a[y] + o[y]) * s[1]));
}
template <int P, typename T>
__device__ inline T lds_d(const T *a, int e) {
  return e == 0 ? a[12 * P] : (e == 4 ? a[13 * P] : a[(e - 1) * P]);
}

#ifdef CODENS_SW_WAVES
#define SW_ATTR __attribute__((amdgpu_waves_per_eu(CODENS_SW_WAVES, CODENS_SW_WAVES)))
#else
#define SW_ATTR
#endif
// EU selects the flux increments of implimf_eu (which read ps); the face
// terms, coefficients and update are common to both implicit phases.
template <bool EU, typename T, int TXS, int TYS, class DIN>
__device__ __forceinline__ void sweep_body(const Blk b, int lg, int ntx, int nty, int ks, const Phys ph, int ityprk,
                                           const T *__restrict__ u, const T *__restrict__ ff,
                                           const T *__restrict__ v, long ldv, const double *__restrict__ ps,
                                           const T *__restrict__ sn, const T *__restrict__ coefe,
                                           const T *__restrict__ diag, const DIN dold, const TView<T> dnew,
                                           T *sq) {
#pragma clang fp contract(off)
  constexpr int PL = (TYS + 2) * (TXS + 2), HALO = 2 * TXS + 2 * TYS;
  static_assert(HALO <= TXS * TYS, "one halo cell per thread at most");
#include "sweep_tile.inc"
}

template <bool EU, typename T, int TXS = SW_TX, int TYS = SW_TY>
__global__ void __launch_bounds__(TXS *TYS) SW_ATTR k_impl_sweep_tiled(Blk b, Phys ph, int ityprk, int ntx, int nty,
                                                                   int nkz, int ks, const T *__restrict__ u,
                                                                   const T *__restrict__ ff,
                                                                   const T *__restrict__ v, long ldv,
                                                                   const double *__restrict__ ps,
                                                                   const T *__restrict__ sn,
                                                                   const T *__restrict__ coefe,
                                                                   const T *__restrict__ diag, TView<T> dold,
                                                                   TView<T> dnew, int rev) {
#pragma clang fp contract(off)
  // XCD-aware tile order: the hardware deals workgroups to the 8 XCDs round
  // robin; give each XCD a contiguous run of tiles so that j/k neighbours
  // share its L2.  rev runs each XCD's tiles in reverse: alternate
  // sub-iterations then begin where the previous one ended, on the data it
  // left in the last-level cache (the tile order does not change any value).
  constexpr int PL = (TYS + 2) * (TXS + 2), HALO = 2 * TXS + 2 * TYS;
  static_assert(HALO <= TXS * TYS, "one halo cell per thread at most");
  __shared__ T sq[14 * PL];
  int nwg = ntx * nty * nkz;
  int hw = blockIdx.x;
  int lg = (nwg % 8 == 0) ? (hw % 8) * (nwg / 8) + hw / 8 : hw;
  if (rev) lg = nwg - 1 - lg;
#include "sweep_tile.inc"
}

// ---------------------------------------------------------------------------
// Two sub-iterations A and B in one pass over the operands, which are most of
// a sub-iteration's traffic (33 doubles per cell, of which the increments are
// ten).  A workgroup's 32 x 16 threads each own a cell; A is right on all but
// the outermost ring, B on all but two, so the tile writes 28 x 12 cells.
// Marching k, plane k of A gives plane k - 1 of B its last part, so that B
// uses the operands of plane k right after A, and carries five sums and a
// reciprocal per cell to the next plane.  A's and B's 14-vectors of a plane lie
// in LDS buffers of their own; a wave holds two rows.
//
// Every cell's operations are those of sweep_tile.inc in the same order, so
// that a pair gives the bits of two single sweeps (the minmod chains turn a
// change of the last bit of the state into 1e-7 of the next residual).  The term of an
// i face is formed by the cell above it and passed down a lane.
//
// One workgroup per CU (135 KB of LDS, 254 registers, two waves per SIMD).  On
// 256 x 128 x 64 a pair takes 175 us and moves 670 MB, against 2 x 125 us for
// single sweeps of 674 MB each, at 5.4 TB/s, what a large copy reaches; a pair's
// waves issue or wait for arithmetic and LDS half of the time.  With workgroup
// barriers in place of the flags below it took 225 us, with flags that waited
// for the loads in flight 192, and before that with the i and j faces' operands
// loaded at the top of their plane instead of during the plane below 199.
constexpr int S2_TX = 32, S2_TY = 16, S2_NC = S2_TX * S2_TY;
// cells that a tile writes; FIRST, where A needs no neighbour, one ring more
constexpr int s2_ox(bool first) { return S2_TX - (first ? 2 : 4); }
constexpr int s2_oy(bool first) { return S2_TY - (first ? 2 : 4); }
constexpr int S2_STASH = 5, S2_LDS = (28 + S2_STASH) * S2_NC;
constexpr int S2_KS = 16;  // k planes per workgroup in the all-blocks launch

// the value of the lane above
__device__ __forceinline__ double lane_above(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// component of q that holds d of equation e
__device__ __forceinline__ constexpr int q_comp(int e) { return e == 0 ? 12 : (e == 4 ? 13 : e - 1); }

// a flag that waves of a workgroup pass to each other (an LDS pointer: an access
// through a generic one waits for the global loads in flight too)
using LdsFlag = __attribute__((address_space(3))) int;

// gp and ldp without the empty asm, whose scalar operands the pair kernel has no
// registers for (the opaque offsets suffice there; the fused residual is 2%
// slower without it)
template <typename T>
__device__ __forceinline__ GPtr<T> gp2(T *base, unsigned off) {
  return (GPtr<T>)((GPtr<char>)(uint64_t)base + off);
}
template <typename T>
__device__ __forceinline__ T ldp2(const T *base, unsigned off) {
  return *gp2(base, off);
}

// FIRST: A is sub-iteration 1, which starts from d = 0 and is (-u - ff)/diag.
template <bool FF, bool FIRST>
__device__ __forceinline__ void sweep2_body(const Blk &b, int lg, int ntx, int nty, int ks, const Phys &ph,
                                            const double *__restrict__ u, const double *__restrict__ ff,
                                            const double *__restrict__ v, long ldv, const double *__restrict__ sn,
                                            const double *__restrict__ coefe, const double *__restrict__ diag,
                                            const DView dold, const DView dnew, double *sx, LdsFlag *flag) {
#pragma clang fp contract(off)
  auto scalar = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
  const int bx = scalar(lg % ntx), by = scalar((lg / ntx) % nty), bz = scalar(lg / (ntx * nty));
  const int t = threadIdx.x, tx = t % S2_TX, ty = t / S2_TX;
  constexpr int RING = FIRST ? 1 : 2;
  const int i = b.i1 + bx * s2_ox(FIRST) - RING + tx, j = b.j1 + by * s2_oy(FIRST) - RING + ty;
  const int kb = b.k1 + bz * ks, ke = min(kb + ks, b.k2);
  const int ka = max(kb - 1, b.k1), kz = min(ke, b.k2 - 1);  // planes of A
  const bool own = i >= b.i1 && i < b.i2 && j >= b.j1 && j < b.j2;
  const bool out = own && tx >= RING && tx < S2_TX - RING && ty >= RING && ty < S2_TY - RING;
  const bool ireal = i + 1 < b.i2, jreal = j + 1 < b.j2;
  // offset in a plane of this thread's cell, or of the nearest cell whose low
  // faces exist (the first ghost past the real cells closes their last face)
  auto plane = [&](int x, int y) { return ((unsigned)(x - b.id1) + (unsigned)(y - b.jd1) * (unsigned)b.nid) * 8u; };
  const unsigned pl0 = plane(min(max(i, b.i1), b.i2), min(max(j, b.j1), b.j2 - 1));
  // LDS slots of the neighbours (the thread's own at the tile's edge, where
  // the result is not used)
  const int tl = max(t - 1, 0), tr = min(t + 1, S2_NC - 1), td = max(t - S2_TX, tx), tu = min(t + S2_TX, S2_NC - S2_TX + tx);
  double *const qA = sx, *const qB = sx + 14 * S2_NC, *const stash = sx + 28 * S2_NC + t;
  // B's q of the plane below (own slot) and of the plane.  A pair meets twice a
  // plane, so one buffer serves; FIRST meets once and takes qA's as a second
  double *qP = qB, *qC = FIRST ? qA : qB;
  auto st = [&](int x) -> double & { return stash[x * S2_NC]; };  // V of the plane
  const long nnn = b.nnn, nijd = b.nijd;
  double qn[14], tkA[5], base[5], skl[3], ckl, rdb = 0.;  // qn: q of A's next plane
  long mk = (long)(ka - b.kd1) * nijd;
  auto load_vd = [&](long m, unsigned off, double V[5], double D[5]) {
#pragma unroll
    for (int e = 0; e < 5; e++) {
      V[e] = ldp2(v + (e * ldv + b.npc + m), off);
      if (!FIRST) D[e] = ldp2(dold.p + (e * dold.ld + (b.npc - dold.off) + m), off);
    }
  };
  // own slots start as the plane below A's first: q of A there, zero of B
  {
    const unsigned pl = opaque(pl0);
    double V[5], D[5], q[14];
#pragma unroll
    for (int c = 0; c < 14; c++) q[c] = qn[c] = 0.;
#pragma unroll
    for (int c = 0; c < 3; c++) skl[c] = ldp2(sn + ((c * 3 + 2) * nnn + mk), pl);
    ckl = ldp2(coefe + (2 * nnn + mk), pl);
    if (!FIRST && own && ka > b.k1) {
      load_vd(mk - nijd, pl, V, D);
      dflux_q(ph, V, D, q);
    }
    if (own) {
      load_vd(mk, pl, V, D);
      if (!FIRST) dflux_q(ph, V, D, qn);
#pragma unroll
      for (int e = 0; e < 5; e++) st(e) = V[e];
    }
    tn2_fma(qn, skl, tkA, [&](int c) { return q[c]; });
#pragma unroll
    for (int c = 0; c < 14; c++) {
      if (!FIRST) qA[c * S2_NC + t] = q[c];
      qB[c * S2_NC + t] = 0.;
    }
#pragma unroll
    for (int e = 0; e < 5; e++) base[e] = 0.;
  }
  // A wave takes rows from the waves below and above it only, so it waits for
  // those two to have written theirs instead of at a workgroup barrier: the
  // waves of a SIMD then drift apart and one computes while the other waits
  // for its loads.  Every wave runs the same number of phases and raises its
  // flag in each before it waits, so every wait ends.  A row is overwritten
  // only after its readers have raised the flag of the following phase: a
  // buffer is written again two phases later (two meetings a plane, or one and
  // two buffers in turn).  The flags are relaxed atomics, so that the fences
  // around them order the rows.
  const int wv = __builtin_amdgcn_readfirstlane(t / 64);
  int phase = 0;
  auto raised = [&](int w) { return __hip_atomic_load(flag + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  auto meet = [&]() {
    phase++;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __hip_atomic_store(flag + wv, phase, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (wv > 0) while (raised(wv - 1) < phase) __builtin_amdgcn_s_sleep(0);
    if (wv < S2_NC / 64 - 1) while (raised(wv + 1) < phase) __builtin_amdgcn_s_sleep(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  struct IJ {
    double sil[3], sjl[3], sjh[3], cil, cih, cjl, cjh, uu[5];
  } o, on;
  auto load_ij = [&](long m, unsigned pl, IJ &o) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      o.sil[c] = ldp2(sn + (c * 3 * nnn + m), pl);
      o.sjl[c] = ldp2(sn + ((c * 3 + 1) * nnn + m), pl);
      o.sjh[c] = ldp2(sn + ((c * 3 + 1) * nnn + m + b.nid), pl);
    }
    o.cil = ldp2(coefe + m, pl);
    o.cih = ldp2(coefe + m, pl + 8u);
    o.cjl = ldp2(coefe + (nnn + m), pl);
    o.cjh = ldp2(coefe + (nnn + m + b.nid), pl);
#pragma unroll
    for (int e = 0; e < 5; e++) o.uu[e] = ldp2(u + (e * ldv + b.npc + m), pl);
  };
  load_ij(mk, opaque(pl0), o);
  for (int k = ka; k <= kz; k++, mk += nijd) {
    const bool kreal = k + 1 < b.k2;
    const unsigned pl = opaque(pl0);
    // the loads of the plane but its i and j faces', which came with the plane
    // below
    double skh[3], fv[5] = {0., 0., 0., 0., 0.}, Vn[5], Dn[5];
#pragma unroll
    for (int c = 0; c < 3; c++) skh[c] = ldp2(sn + ((c * 3 + 2) * nnn + mk + nijd), pl);
    const double ckh = kreal ? ldp2(coefe + (2 * nnn + mk + nijd), pl) : 0.;
    const double dg = ldp2(diag + mk, pl);
    if constexpr (FF) {
#pragma unroll
      for (int e = 0; e < 5; e++) fv[e] = ldp2(ff + (e * ldv + b.npc + mk), pl);
    }
    if (own && kreal) load_vd(mk + nijd, pl, Vn, Dn);
    double q[14], w[5], tn[5], dlo[5], dhi[5];
    // the i and j faces and the lower k face of the plane's cell, its q in
    // buffer Q: w = -u - ff + ... as sweep_tile.inc sums it
    auto faces = [&](const double *Q, const double tk[5]) {
      tn2_fma(q, o.sil, tn, [&](int c) { return Q[c * S2_NC + tl]; });
#pragma unroll
      for (int e = 0; e < 5; e++) {
        const double th = lane_above(tn[e]);
        w[e] = fma(o.cil, Q[q_comp(e) * S2_NC + tl], fma(0.5, tn[e], -o.uu[e] - fv[e]));
        if (ireal) w[e] = fma(o.cih, Q[q_comp(e) * S2_NC + tr], w[e]);
        w[e] = fma(-0.5, th, w[e]);
      }
      tn2_fma(q, o.sjl, tn, [&](int c) { return Q[c * S2_NC + td]; });
#pragma unroll
      for (int e = 0; e < 5; e++) {
        w[e] = fma(o.cjl, Q[q_comp(e) * S2_NC + td], fma(0.5, tn[e], w[e]));
        if (jreal) w[e] = fma(o.cjh, Q[q_comp(e) * S2_NC + tu], w[e]);
      }
      tn2_fma(q, o.sjh, tn, [&](int c) { return Q[c * S2_NC + tu]; });
#pragma unroll
      for (int e = 0; e < 5; e++) w[e] = fma(ckl, dlo[e], fma(0.5, tk[e], fma(-0.5, tn[e], w[e])));
    };
    const double rd = 1. / dg;
    if constexpr (FIRST) {
#pragma unroll
      for (int e = 0; e < 5; e++) dhi[e] = (-o.uu[e] - fv[e]) / dg;
    } else {
      // A on plane k
#pragma unroll
      for (int e = 0; e < 5; e++) dlo[e] = qA[q_comp(e) * S2_NC + t];  // of the plane below
#pragma unroll
      for (int c = 0; c < 14; c++) {
        q[c] = qn[c];
        qA[c * S2_NC + t] = q[c];
        qn[c] = 0.;
      }
      meet();
      faces(qA, tkA);
      // the plane above, the face between and what its increment adds
      if (own && kreal) dflux_q(ph, Vn, Dn, qn);
      tn2_fma(qn, skh, tkA, [&](int c) { return q[c]; });
#pragma unroll
      for (int e = 0; e < 5; e++) {
        if (kreal) w[e] = fma(ckh, qn[q_comp(e)], w[e]);
        w[e] = fma(-0.5, tkA[e], w[e]);
      }
#pragma unroll
      for (int e = 0; e < 5; e++) dhi[e] = w[e] * rd;  // A's increment
    }
#pragma unroll
    for (int c = 0; c < 14; c++) q[c] = 0.;
    if (own) {
      double V[5];
#pragma unroll
      for (int e = 0; e < 5; e++) V[e] = st(e);
      dflux_q(ph, V, dhi, q);
      if (kreal) {
#pragma unroll
        for (int e = 0; e < 5; e++) st(e) = Vn[e];
      }
    }
    // B: plane k - 1 is complete with the face to plane k
    double tk[5];
    tn2_fma(q, skl, tk, [&](int c) { return qP[c * S2_NC + t]; });
#pragma unroll
    for (int e = 0; e < 5; e++) {
      dlo[e] = qP[q_comp(e) * S2_NC + t];
      dhi[e] = fma(-0.5, tk[e], fma(ckl, dhi[e], base[e])) * rdb;
    }
    if (out && k > kb) {
#pragma unroll
      for (int e = 0; e < 5; e++) *gp2(dnew.p + (e * dnew.ld + (b.npc - dnew.off) + mk - nijd), pl) = dhi[e];
    }
#pragma unroll
    for (int c = 0; c < 14; c++) qC[c * S2_NC + t] = q[c];
    load_ij(mk + nijd, pl, on);  // of the plane above (a ghost's past the last: not used)
    meet();
    faces(qC, tk);
    if (FIRST) {
      double *const x = qP;
      qP = qC;
      qC = x;
    }
    o = on;
#pragma unroll
    for (int e = 0; e < 5; e++) base[e] = w[e];
    rdb = rd;
    ckl = ckh;
#pragma unroll
    for (int c = 0; c < 3; c++) skl[c] = skh[c];
  }
  if (out && ke == b.k2) {  // the block's last plane: its upper face is a ghost's
    double q[14], tk[5];
#pragma unroll
    for (int c = 0; c < 14; c++) q[c] = qP[c * S2_NC + t];
    tn2_fma(q, skl, tk, [&](int) { return 0.; });
#pragma unroll
    for (int e = 0; e < 5; e++)
      *gp2(dnew.p + (e * dnew.ld + (b.npc - dnew.off) + mk - nijd), opaque(pl0)) =
          fma(-0.5, tk[e], base[e]) * rdb;
  }
}

template <bool FF, bool FIRST>
__global__ void __launch_bounds__(S2_NC) __attribute__((amdgpu_waves_per_eu(2)))
k_impl_sweep2(Blk b, Phys ph, int ntx, int nty, int ks, const double *__restrict__ u, const double *__restrict__ ff,
              const double *__restrict__ v, long ldv, const double *__restrict__ sn, const double *__restrict__ coefe,
              const double *__restrict__ diag, DView dold, DView dnew, int rev) {
  __shared__ double sx[S2_LDS];
  __shared__ int flag[S2_NC / 64];
  if (threadIdx.x < S2_NC / 64) flag[threadIdx.x] = 0;
  __syncthreads();
  unsigned lg = xcd_linear();
  if (rev) lg = gridDim.x - 1 - lg;
  sweep2_body<FF, FIRST>(b, (int)lg, ntx, nty, ks, ph, u, ff, v, ldv, sn, coefe, diag, dold, dnew, sx, (LdsFlag *)flag);
}

// ---------------------------------------------------------------------------
// A sub-iteration of a small block.  The tiled kernel's workgroup there waits
// for its loads three times (the planes below, its own, the one above) with
// one or two waves on a compute unit, 7 us on 32 x 16 x 8; here eight lanes
// share a cell and everything is loaded at once: lane 0 of a cell forms its q,
// lanes 1..6 that of a neighbour and the term of the face to it, then lane e
// sums equation e in the order of sweep_tile.inc.  The operations are those of
// the pair kernel, so the bits are those of the other kernels.  A wave holds
// eight cells of a row, lane = role * 8 + cell.  It computes each q seven
// times and loads it from the L2, so it pays only while the chip is not full: a
// sub-iteration of 32 x 16 x 8 takes 3.8 us against 7.0 in tiles, 64 x 32 x 16
// 8.9 against 9.6, 48 x 40 x 36 15.4 against 12.0.  The line lies below where the
// two cross, as a block above it reports a timed tile shape
// (codens_sweep_tile_of), which it did before this kernel.
constexpr int SM_CELLS = 8;
constexpr long SMALL_BLOCK = 16384;  // real cells

template <bool FIRST>
__global__ void __launch_bounds__(64) k_impl_sweep_small(Blk b, Phys ph, int ityprk, const double *__restrict__ u,
                                                         const double *__restrict__ ff,
                                                         const double *__restrict__ v, long ldv,
                                                         const double *__restrict__ sn,
                                                         const double *__restrict__ coefe,
                                                         const double *__restrict__ diag, DView dold, DView dnew) {
#pragma clang fp contract(off)
  __shared__ double own[12][SM_CELLS], tnf[5][6][SM_CELLS], dnb[5][6][SM_CELLS], cf[6][SM_CELLS];
  const int lane = threadIdx.x, c = lane % SM_CELLS, role = lane / SM_CELLS, f = max(role - 1, 0) % 6;
  const int nx = b.i2 - b.i1, ny = b.j2 - b.j1, nz = b.k2 - b.k1;
  const int cell = blockIdx.x * SM_CELLS + c;
  const bool in = cell < nx * ny * nz;
  const int x = in ? cell : 0;
  const int ci = x % nx, cj = (x / nx) % ny, ck = x / (nx * ny);
  const long n = b.idx(b.i1 + ci, b.j1 + cj, b.k1 + ck), m = n - b.npc, nnn = b.nnn;
  // this lane's cell and face
  const int d = f / 2;
  const bool high = f % 2, nb = role >= 1 && role <= 6;
  const long inc = d == 0 ? 1 : (d == 1 ? b.nid : b.nijd);
  const int at = d == 0 ? ci : (d == 1 ? cj : ck), len = d == 0 ? nx : (d == 1 ? ny : nz);
  const bool real = !nb || (high ? at + 1 < len : at > 0);
  const long nr = nb && real ? (high ? n + inc : n - inc) : n, mf = high ? m + inc : m;
  const int e = min(role, 4);
  double V[5], D[5], s[3], q[14];
#pragma unroll
  for (int x = 0; x < 5; x++) {
    V[x] = v[x * ldv + nr];
    D[x] = FIRST ? -u[x * ldv + nr] : dold.at(x, nr);
  }
  const double gr = FIRST ? diag[nr - b.npc] : 1.;
  if (FIRST && ityprk) {
#pragma unroll
    for (int x = 0; x < 5; x++) D[x] = D[x] - ff[x * ldv + nr];
  }
#pragma unroll
  for (int x = 0; x < 3; x++) s[x] = sn[(x * 3 + d) * nnn + mf];
  const double co = coefe[d * nnn + (real ? mf : m)], uu = u[e * ldv + n], dg = diag[m];
  const double fv = ityprk ? ff[e * ldv + n] : 0.;
  if (FIRST) {
#pragma unroll
    for (int x = 0; x < 5; x++) D[x] = D[x] / gr;
  }
  dflux_q(ph, V, D, q);
  if (!real) {
#pragma unroll
    for (int x = 0; x < 14; x++) q[x] = 0.;
  }
  if (role == 0) {
#pragma unroll
    for (int x = 0; x < 12; x++) own[x][c] = q[x];
  }
  __syncthreads();
  if (nb) {
    double tn[5];
    tn2_fma(q, s, tn, [&](int x) { return own[x][c]; });
#pragma unroll
    for (int x = 0; x < 5; x++) {
      tnf[x][f][c] = tn[x];
      dnb[x][f][c] = q[q_comp(x)];
    }
    cf[f][c] = co;
  }
  __syncthreads();
  if (role < 5 && in) {
    double w = -uu - fv;
#pragma unroll
    for (int x = 0; x < 3; x++) {
      const int p = x == 0 ? ci : (x == 1 ? cj : ck), l = x == 0 ? nx : (x == 1 ? ny : nz);
      w = fma(cf[2 * x][c], dnb[e][2 * x][c], fma(0.5, tnf[e][2 * x][c], w));
      if (p + 1 < l) w = fma(cf[2 * x + 1][c], dnb[e][2 * x + 1][c], w);
      w = fma(-0.5, tnf[e][2 * x + 1][c], w);
    }
    dnew.at(e, n) = w * (1. / dg);
  }
}

// ---------------------------------------------------------------------------
// Tile shape of the tiled sub-iteration, per block shape: 64 x 4, 32 x 8 or
// 16 x 16, all of 256 threads.  Every cell's arithmetic is the same in all,
// so the increments are identical bit for bit; what differs is how many
// lanes idle on the i and j edges of a block, the LDS halo per cell and the
// length of the rows each wave reads.  By default the first call for a
// block shape times each on the caller's own data (one untimed and two
// timed launches each, on the caller's stream, writing the same result the
// real launch writes next) and keeps the fastest; while the stream is being
// captured into a graph, an unseen block shape takes tile_model's choice.
// codens_sweep_tile forces one shape.
namespace {
// shapes 0 (SW_TX x SW_TY), 1 (32 x 2 SW_TY) and 2 (16 x 16), all of 256
// threads; the all-blocks launch holds the first two (N_BATCH_TILES)
constexpr int N_SWEEP_TILES = 3, N_BATCH_TILES = 2;
std::mutex g_tile_mu;
int g_tile_mode = -1;
std::map<std::array<int, 5>, int> g_tile_best;

inline int tile_tx(int tile) { return tile == 2 ? 16 : (tile == 1 ? 32 : SW_TX); }
inline int tile_ty(int tile) { return tile == 2 ? 16 : (tile == 1 ? 2 * SW_TY : SW_TY); }

// The shape with the least modelled time among the first n: the lanes the
// shape launches over the block's i-j extent (idle lanes past its edges
// included) times the shape's measured time per lane on a block that none
// of them leaves idle lanes in (256 x 128 x 64 on MI355X: 64 x 4 134.7 us,
// 32 x 8 139.2 us, 16 x 16 154.3 us).  The narrower shapes read more halo
// cells per cell and shorter runs of each row.
int tile_model(const Blk &b, int n = N_BATCH_TILES) {
  static const double per_lane[N_SWEEP_TILES] = {1.0, 139.2 / 134.7, 154.3 / 134.7};
  int nx = b.i2 - b.i1, ny = b.j2 - b.j1;
  double best = 0.;
  int pick = 0;
  for (int t = 0; t < n; t++) {
    int tx = tile_tx(t), ty = tile_ty(t);
    double lanes = (double)((nx + tx - 1) / tx * tx) * ((ny + ty - 1) / ty * ty);
    double cost = lanes * per_lane[t];
    if (t == 0 || cost < best) { best = cost; pick = t; }
  }
  return pick;
}

template <bool EU, typename T>
void launch_sweep(int tile, const Blk &b, hipStream_t st, Phys ph, int ityprk, const T *u, const T *ff, const T *v,
                  long ldv, const double *ps, const T *sn, const T *coefe, const T *diag, TView<T> in,
                  TView<T> out, int rev = 0) {
  const int tx = tile_tx(tile), ty = tile_ty(tile);
  const int ntx0 = (b.i2 - b.i1 + tx - 1) / tx, nty0 = (b.j2 - b.j1 + ty - 1) / ty;
  const int ks = slab_depth((long)ntx0 * nty0, b.k2 - b.k1, SW_KS);
  const int nkz = (b.k2 - b.k1 + ks - 1) / ks;
  if (tile == 2) {
    constexpr int X = 16, Y = 16;
    int ntx = (b.i2 - b.i1 + X - 1) / X, nty = (b.j2 - b.j1 + Y - 1) / Y;
    hipLaunchKernelGGL((k_impl_sweep_tiled<EU, T, X, Y>), dim3(ntx * nty * nkz), dim3(X, Y), 0, st, b, ph,
                       ityprk, ntx, nty, nkz, ks, u, ff, v, ldv, ps, sn, coefe, diag, in, out, rev);
  } else if (tile == 1) {
    constexpr int X = 32, Y = 2 * SW_TY;
    int ntx = (b.i2 - b.i1 + X - 1) / X, nty = (b.j2 - b.j1 + Y - 1) / Y;
    hipLaunchKernelGGL((k_impl_sweep_tiled<EU, T, X, Y>), dim3(ntx * nty * nkz), dim3(X, Y), 0, st, b, ph,
                       ityprk, ntx, nty, nkz, ks, u, ff, v, ldv, ps, sn, coefe, diag, in, out, rev);
  } else {
    int ntx = (b.i2 - b.i1 + SW_TX - 1) / SW_TX, nty = (b.j2 - b.j1 + SW_TY - 1) / SW_TY;
    hipLaunchKernelGGL((k_impl_sweep_tiled<EU, T, SW_TX, SW_TY>), dim3(ntx * nty * nkz), dim3(SW_TX, SW_TY),
                       0, st, b, ph, ityprk, ntx, nty, nkz, ks, u, ff, v, ldv, ps, sn, coefe, diag, in, out, rev);
  }
}

// The two-sub-iteration kernel on a block: its tiles, and the slab depth with
// the fewest steps over the rounds of one workgroup per compute unit (a slab
// of ks planes takes ks + 2 steps and about one more to start).
struct Pair {
  int ntx, nty, ks;
  long wgs, steps;  // workgroups; steps of one after another on a compute unit
};
Pair pair_of(const Blk &b, bool first = false) {
  const int nz = b.k2 - b.k1, ncu = codens_resident_workgroups(1), ox = s2_ox(first), oy = s2_oy(first);
  Pair p{(b.i2 - b.i1 + ox - 1) / ox, (b.j2 - b.j1 + oy - 1) / oy, 1, 0, 0};
  for (int ks = 1; ks <= nz; ks = next_slab(nz, ks)) {
    const long w = (long)p.ntx * p.nty * ((nz + ks - 1) / ks);
    const long c = (w + ncu - 1) / ncu * (std::min(ks + 2, nz) + 1);
    if (ks == 1 || c < p.steps) { p.ks = ks; p.wgs = w; p.steps = c; }
  }
  return p;
}

// Whether a block's sub-iterations run in pairs: the modelled time (us) of a
// pair against that of two single sweeps.  Measured on MI355X over 310 block
// shapes of 2 to 300 cells a side: a step of the pair kernel takes 4.4 to 5.2 us
// (less on blocks of fewer rows than its tile).  A single sweep's workgroup
// takes 3.4 us a plane and 4 to start, and the launch fills the chip's places in
// rounds, of which a partly filled last one takes 0.9 of a full one at most;
// where the places are full of active lanes the memory limits, with idle lanes
// 0.4 of that.  Two singles / a pair:
//   256 x 128 x 64 245 / 174 us, 200 x 120 x 100 367 / 192, 128 x 128 x 32 58 / 52,
//   75 x 61 x 43 41 / 33, 48 x 40 x 36 19 / 24, 16 x 16 x 400 19 / 33,
//   4 x 64 x 400 47 / 60
// (the pair kernel's tiles of 28 x 12 cells leave most of their lanes idle on
// the last two).  Of the 310 shapes the rule runs 6 in pairs where that is
// slower by more than 2% (14% at most), and 13 singly (29% at most).
// FP32 sweeps run singly: 61 us on 256 x 128 x 64, whose 349 MB move at 5.7 TB/s.
constexpr double PAIR_STEP = 4.8;

// A single sweep whose workgroups (of planes planes) would fill the chip's
// places `fill` times, a share `active` of their lanes on cells
double single_model(double fill, double planes, double active) {
  const double rounds = fill <= 1. ? 1. : std::min(std::ceil(fill), fill + 0.9);
  const double latency = rounds * (3.4 * planes + 4.);
  const double memory = std::max(1., fill) * (planes + 1.) * 2.8 * (0.8 + 1.2 * active * std::min(1., fill));
  return std::max(latency, memory);
}

bool pair_model(const Blk &b) {
  const int nx = b.i2 - b.i1, ny = b.j2 - b.j1, nz = b.k2 - b.k1;
  const double places = codens_resident_workgroups(2);
  double one = 0.;  // with the shape that takes least
  for (int t = 0; t < N_SWEEP_TILES; t++) {
    const int tx = tile_tx(t), ty = tile_ty(t);
    const long txy = (long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
    const int ks = slab_depth(txy, nz, SW_KS);
    const double wgs = (double)txy * ((nz + ks - 1) / ks);
    const double x = single_model(wgs / places, ks, (double)nx * ny * nz / (wgs * ks * tx * ty));
    if (t == 0 || x < one) one = x;
  }
  return PAIR_STEP * pair_of(b).steps < 2. * one;
}

// two sub-iterations in -> out; first: sub-iterations 1 and 2, in not read
void launch_sweep2(bool first, const Blk &b, hipStream_t st, Phys ph, int ityprk, const double *u, const double *ff,
                   const double *v, long ldv, const double *sn, const double *coefe, const double *diag, DView in,
                   DView out, int rev) {
  const Pair p = pair_of(b, first);
  auto *k = first ? (ityprk ? k_impl_sweep2<true, true> : k_impl_sweep2<false, true>)
                  : (ityprk ? k_impl_sweep2<true, false> : k_impl_sweep2<false, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)p.wgs), dim3(S2_NC), 0, st, b, ph, p.ntx, p.nty, p.ks, u, ff, v, ldv, sn, coefe,
                     diag, in, out, rev);
}

template <bool EU, typename T>
int pick_tile(const Blk &b, hipStream_t st, Phys ph, int ityprk, const T *u, const T *ff, const T *v, long ldv,
              const double *ps, const T *sn, const T *coefe, const T *diag, TView<T> in, TView<T> out) {
  std::array<int, 5> key = {b.i2 - b.i1, b.j2 - b.j1, b.k2 - b.k1, (int)EU, (int)sizeof(T)};
  {
    std::lock_guard<std::mutex> lk(g_tile_mu);
    if (g_tile_mode >= 0) return g_tile_mode;
    auto it = g_tile_best.find(key);
    if (it != g_tile_best.end()) return it->second;
  }
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return tile_model(b);
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return tile_model(b);
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return tile_model(b);
  }
  int pick = tile_model(b);
  float best = -1.f;
  for (int t = 0; t < N_SWEEP_TILES; t++) {
    launch_sweep<EU, T>(t, b, st, ph, ityprk, u, ff, v, ldv, ps, sn, coefe, diag, in, out);
    (void)hipEventRecord(e0, st);
    for (int r = 0; r < 2; r++)
      launch_sweep<EU, T>(t, b, st, ph, ityprk, u, ff, v, ldv, ps, sn, coefe, diag, in, out);
    (void)hipEventRecord(e1, st);
    float ms = 0.f;
    if (hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
      pick = tile_model(b);
      best = -1.f;
      break;
    }
    if (best < 0.f || ms < best) { best = ms; pick = t; }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  std::lock_guard<std::mutex> lk(g_tile_mu);
  g_tile_best[key] = pick;
  return pick;
}
}  // namespace

// Launches of lmx sub-iterations: the first (from d = 0), singles, pairs.  In
// pairs an even number of them begins with a pair too (the FIRST form: on 256 x
// 128 x 64 139 us, on 200 x 120 x 100 136, against 33 and 42 for k_impl_sweep1 and
// 131 and 194 for a single sweep).
struct SweepPlan {
  bool first2;
  int single, pairs, n;
};
static SweepPlan sweep_plan(int lmx, bool pairs) {
  const bool first2 = pairs && lmx > 1 && lmx % 2 == 0;
  const int rest = std::max(0, lmx - (first2 ? 2 : 1)), np = pairs ? rest / 2 : 0;
  return {first2, rest - 2 * np, np, lmx > 0 ? 1 + rest - np : 0};
}

static int forced_tile() {
  std::lock_guard<std::mutex> lk(g_tile_mu);
  return g_tile_mode;
}

// tile of a block without timing anything: the forced mode, the choice
// already timed for its shape, or the model's
static int known_tile(const Blk &b, bool eu, int tsize) {
  std::array<int, 5> key = {b.i2 - b.i1, b.j2 - b.j1, b.k2 - b.k1, eu ? 1 : 0, tsize};
  std::lock_guard<std::mutex> lk(g_tile_mu);
  if (g_tile_mode >= 0) return g_tile_mode;
  auto it = g_tile_best.find(key);
  return it != g_tile_best.end() ? it->second : tile_model(b);
}

extern "C" int codens_sweep_tile(int32_t mode, int32_t *previous) {
  if (mode < -1 || mode >= N_SWEEP_TILES) {
    codens_set_error("codens_sweep_tile: mode %d is not -1 (timed choice), 0 (64 x 4), 1 (32 x 8) or 2 (16 x 16)",
                     mode);
    return CODENS_EINVAL;
  }
  std::lock_guard<std::mutex> lk(g_tile_mu);
  if (previous) *previous = g_tile_mode;
  g_tile_mode = mode;
  return CODENS_OK;
}

extern "C" int codens_sweep_tile_of(const codens_block *cb, int32_t eu, int32_t fp32, int32_t *tile) {
  int rc = codens_check_block(cb, "codens_sweep_tile_of");
  if (rc) return rc;
  if (!tile) {
    codens_set_error("codens_sweep_tile_of: null argument");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  std::array<int, 5> key = {b.i2 - b.i1, b.j2 - b.j1, b.k2 - b.k1, eu ? 1 : 0, fp32 ? 4 : 8};
  std::lock_guard<std::mutex> lk(g_tile_mu);
  auto it = g_tile_best.find(key);
  *tile = g_tile_mode >= 0 ? g_tile_mode : (it != g_tile_best.end() ? it->second : -1);
  return CODENS_OK;
}

// implimf_3d.f90:473-486
__device__ __forceinline__ void update_body(const Blk &b, dim3 tile, double *v, long ldv,
                                            const double *__restrict__ d, int nvar) {
  CELL3_AT(b, tile)
  long n = b.idx(c[0], c[1], c[2]);
  for (int e = 0; e < nvar; e++) v[e * ldv + n] = v[e * ldv + n] + d[e * ldv + n];
}

__global__ void __launch_bounds__(TX *TY) k_impl_update(Blk b, double *v, long ldv, double *d, int nvar) {
  // d = 0 on the ghosts; the last sub-iteration wrote every real cell
  if (shell_layers(b, b.k2 - b.k1, b.npc, b.npc + b.nnn - 1, d, ldv, 5)) return;
  update_body(b, xcd_block(false, b.k2 - b.k1), v, ldv, d, nvar);
}

__global__ void k_zero5(double *d, long ldv, long n0, long n1) {
  long n = n0 + blockIdx.x * 256L + threadIdx.x;
  if (n > n1) return;
#pragma unroll
  for (int e = 0; e < 5; e++) d[e * ldv + n] = 0.;
}

// Shared host sequence of both implicit phases: zero d, coefficients, lmx
// sub-iterations (ping-pong between the caller's d and the workspace, the
// last one landing in d), then v += d on nvar planes.
// ws_ext: scratch of 9 nnn doubles supplied by the caller (then nothing is
// allocated, no timing event is created and the sub-iteration tile is the
// forced or already chosen one, else the model's); nullptr: the library's
// workspace.
static int implimf_common(bool eu, const codens_block *cb, const codens_phys *cp, const double *u, const double *dt,
                          double *v, int64_t ldv, int nvar, double *d, const double *ff, const double *mu,
                          const double *mut, int32_t lmx, const double *sn, const double *vol, double dtpas,
                          double dt1min, int32_t kfmg, int32_t ityprk, const double *ps, const double *cson,
                          void *stream, const char *what, double *ws_ext = nullptr) {
  int rc = codens_check_block(cb, what);
  if (rc) return rc;
  if (!cp || !u || !dt || !v || !d || (!eu && (!mu || !mut)) || (eu && !ps) || !sn || !vol || !cson ||
      (ityprk && !ff) || lmx < 0 || nvar < 5) {
    codens_set_error("%s: invalid argument", what);
    return CODENS_EINVAL;
  }
  if (eu && kfmg == 3 && !(dt1min > 0.)) {
    codens_set_error("%s: dt1min must be positive when kfmg = 3", what);
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  Phys ph = make_phys(cp);
  hipStream_t st = (hipStream_t)stream;
  const bool fixed = ws_ext != nullptr;
  double *ws = fixed ? ws_ext : (double *)codens_workspace(sizeof(double) * 9 * b.nnn, 2);
  if (!ws) {
    codens_set_error("%s: workspace allocation failed", what);
    return CODENS_EHIP;
  }
  double *coefe = ws, *diag = ws + 3 * b.nnn, *W = ws + 4 * b.nnn;
  long n0 = b.npc, n1 = b.npc + b.nnn - 1;
  auto tname = [fixed](const char *n) { return fixed ? (const char *)nullptr : n; };
  if (lmx < 1) hipLaunchKernelGGL(k_zero5, dim3((b.nnn + 255) / 256), dim3(256), 0, st, d, (long)ldv, n0, n1);
  dim3 g = cell_grid(b), t(TX, TY);
  {
    CodensTimed _tm(tname("implimf_coef"), st);
    if (eu) {
      hipLaunchKernelGGL(k_impl_coef_eu, g, t, 0, st, b, v, (long)ldv, dt, vol, cson, sn,
                         kfmg == 3 ? 1.5 / dt1min : 0., coefe, diag);
    } else {
      const int ks = coef_slab(b, g);
      dim3 gc(g.x, g.y, (unsigned)((b.k2 - b.k1 + ks - 1) / ks));
      hipLaunchKernelGGL(k_impl_coef_tiled<double>, gc, t, 0, st, b, ph, v, (long)ldv, mu, mut, dt, vol, cson, sn,
                         dtpas, (int)kfmg, coefe, diag, ks, F32Copies{});
    }
  }
  DView A = {d, (long)ldv, 0}, B = {W, b.nnn, b.npc};
  int tile = 0;
  // sub-iteration 1 starts from d = 0: d = -u/diag (k_impl_sweep1, or the
  // second one on a small block); the others run in pairs, one left over on its
  // own, alternate launches in reverse tile order; a small block, a forced tile
  // shape, the Euler form, or a block where pairs do not pay (pair_model),
  // runs them one by one.  The launches alternate between the two buffers, the
  // last one landing in d.
  const long cells = (long)(b.i2 - b.i1) * (b.j2 - b.j1) * (b.k2 - b.k1);
  const bool choose = !eu && forced_tile() < 0, small = choose && cells <= SMALL_BLOCK;
  const SweepPlan plan = sweep_plan(lmx, choose && !small && pair_model(b));
  const double *fx = ityprk ? ff : u, *psx = eu ? ps : v;
  for (int s = 0; s < plan.n; s++) {
    DView out = ((plan.n - 1 - s) % 2 == 0) ? A : B;
    DView in = ((plan.n - 1 - s) % 2 == 0) ? B : A;
    if (s == 0 && small && plan.single > 0) continue;  // formed by the second
    if (s == 0 && plan.first2) {
      CodensTimed _tm(tname("implimf_sweep1"), st);
      launch_sweep2(true, b, st, ph, (int)ityprk, u, fx, v, (long)ldv, sn, coefe, diag, in, out, 0);
    } else if (s == 0) {
      CodensTimed _tm(tname("implimf_sweep1"), st);
      hipLaunchKernelGGL(k_impl_sweep1<double>, g, t, 0, st, b, (int)ityprk, u, fx, (long)ldv, diag, out);
    } else if (s <= plan.single && small) {
      CodensTimed _tm(tname("implimf_sweep"), st);
      hipLaunchKernelGGL(s == 1 ? k_impl_sweep_small<true> : k_impl_sweep_small<false>, dim3((unsigned)((cells + SM_CELLS - 1) / SM_CELLS)), dim3(64), 0, st, b, ph,
                         (int)ityprk, u, fx, (const double *)v, (long)ldv, sn, coefe, diag, in, out);
    } else if (s <= plan.single) {
      if (s == 1 && fixed)
        tile = known_tile(b, eu, (int)sizeof(double));
      else if (s == 1)
        tile = eu ? pick_tile<true, double>(b, st, ph, (int)ityprk, u, fx, v, (long)ldv, psx, sn, coefe, diag, in, out)
                  : pick_tile<false, double>(b, st, ph, (int)ityprk, u, fx, v, (long)ldv, psx, sn, coefe, diag, in,
                                             out);
      CodensTimed _tm(tname("implimf_sweep"), st);
      if (eu)
        launch_sweep<true, double>(tile, b, st, ph, (int)ityprk, u, fx, v, (long)ldv, psx, sn, coefe, diag, in, out,
                                   s % 2);
      else
        launch_sweep<false, double>(tile, b, st, ph, (int)ityprk, u, fx, v, (long)ldv, psx, sn, coefe, diag, in, out,
                                    s % 2);
    } else {
      CodensTimed _tm(tname("implimf_sweep2"), st);
      launch_sweep2(false, b, st, ph, (int)ityprk, u, fx, v, (long)ldv, sn, coefe, diag, in, out, s % 2);
    }
  }
  {
    CodensTimed _tm(tname("implimf_update"), st);
    hipLaunchKernelGGL(k_impl_update, with_shell(b, g), t, 0, st, b, v, (long)ldv, d, nvar);
  }
  return codens_check_launch(what);
}

int codens_implimf_3d_with(const codens_block *b, const codens_phys *ph, const double *u, const double *dt, double *v,
                           int64_t ldv, double *d, const double *ff, const double *mu, const double *mut, int32_t lmx,
                           const double *sn_blk, const double *vol, double dtpas, int32_t kfmg, int32_t ityprk,
                           const double *cson, void *stream, double *ws, const char *what) {
  return implimf_common(false, b, ph, u, dt, v, ldv, 5, d, ff, mu, mut, lmx, sn_blk, vol, dtpas, 1.0, kfmg, ityprk,
                        nullptr, cson, stream, what, ws);
}

// ---------------------------------------------------------------------------
// implimf_3d for all blocks of a layout.  Each pass (coefficients, first
// sub-iteration, the lmx-1 tiled sub-iterations, update) is one
// flattened launch over every block; a device table gives each block its
// extents and its first workgroup per pass, and a workgroup runs the
// per-block kernel's own body on its block's tile.  Block l's coefficients,
// diagonal and ping-pong increment (9 planes of nnn) start at 9 npc of the
// workspace.  The sub-iterations of small blocks then share the chip instead
// of each filling a few CUs.
enum { IB_ZERO, IB_CELL, IB_SWEEP, IB_COEF, IB_SWEEP2, IB_FIRST2, IB_SHELL, IB_N };

struct ImplEnt {
  Blk b;
  unsigned start[IB_N];         // first workgroup of this block, per pass
  unsigned gx[IB_N], gy[IB_N];  // this block's grid, per pass
  int tile;                     // sub-iteration tile shape of this block (0: 64 x 4, 1: 32 x 8)
  int ks_coef, ks_sweep, ks_sweep2;  // k planes per workgroup
};

__global__ void __launch_bounds__(256) k_zero5_batch(const ImplEnt *__restrict__ tab, int nb, double *d, long ldv) {
  const ImplEnt &E = tab[tab_find(tab, nb, IB_ZERO, blockIdx.x)];
  const long n0 = E.b.npc, n = n0 + (blockIdx.x - E.start[IB_ZERO]) * 256L + threadIdx.x;
  if (n >= n0 + E.b.nnn) return;
#pragma unroll
  for (int e = 0; e < 5; e++) d[e * ldv + n] = 0.;
}

__global__ void __launch_bounds__(TX *TY) k_impl_coef_batch(const ImplEnt *__restrict__ tab, int nb, Phys ph,
                                                            const double *__restrict__ v, long ldv,
                                                            const double *__restrict__ mu,
                                                            const double *__restrict__ mut,
                                                            const double *__restrict__ dt,
                                                            const double *__restrict__ vol,
                                                            const double *__restrict__ cson,
                                                            const double *__restrict__ sn_all, double dtpas, int kfmg,
                                                            double *ws) {
  __shared__ CoefLds S;
  const unsigned wg = xcd_linear();
  const ImplEnt &E = tab[tab_find(tab, nb, IB_COEF, wg)];
  const Blk b = uniform_blk(E.b);
  double *c = ws + 9 * b.npc;
  coef_tiled_body<double>(b, tab_tile(E, IB_COEF, wg), ph, v, ldv, mu, mut, dt, vol, cson, sn_all + 9 * b.npc, dtpas,
                          kfmg, c, c + 3 * b.nnn, E.ks_coef, S, F32Copies{});
}

__global__ void __launch_bounds__(TX *TY) k_impl_sweep1_batch(const ImplEnt *__restrict__ tab, int nb, int ityprk,
                                                              const double *__restrict__ u,
                                                              const double *__restrict__ ff, long ldv, double *ws,
                                                              double *d, int out_d) {
  const unsigned wg = xcd_linear();
  const ImplEnt &E = tab[tab_find(tab, nb, IB_CELL, wg)];
  const Blk b = E.b;
  double *c = ws + 9 * b.npc;
  DView out = out_d ? DView{d, ldv, 0} : DView{c + 4 * b.nnn, b.nnn, b.npc};
  sweep1_body<double>(b, tab_tile(E, IB_CELL, wg), ityprk, u, ff, ldv, c + 3 * b.nnn, out);
}

__global__ void __launch_bounds__(SW_TX *SW_TY) k_impl_sweep_batch(const ImplEnt *__restrict__ tab, int nb, Phys ph,
                                                                   int ityprk, const double *__restrict__ u,
                                                                   const double *__restrict__ ff,
                                                                   const double *__restrict__ v, long ldv,
                                                                   const double *__restrict__ sn_all, double *ws,
                                                                   double *d, int out_d, int rev) {
  constexpr int PL0 = (SW_TY + 2) * (SW_TX + 2), PL1 = (2 * SW_TY + 2) * (32 + 2);
  __shared__ double sq[14 * (PL0 > PL1 ? PL0 : PL1)];  // one buffer for both shapes
  const unsigned wg = rev ? gridDim.x - 1 - xcd_linear() : xcd_linear();
  const ImplEnt &E = tab[tab_find(tab, nb, IB_SWEEP, wg)];
  const Blk b = E.b;
  double *c = ws + 9 * b.npc;
  DView A = {d, ldv, 0}, B = {c + 4 * b.nnn, b.nnn, b.npc};
  const int lg = (int)(wg - E.start[IB_SWEEP]), ntx = (int)E.gx[IB_SWEEP], nty = (int)E.gy[IB_SWEEP];
  const double *sn = sn_all + 9 * b.npc;
  if (E.tile == 1)
    sweep_body<false, double, 32, 2 * SW_TY>(b, lg, ntx, nty, E.ks_sweep, ph, ityprk, u, ff, v, ldv, v, sn, c,
                                             c + 3 * b.nnn, out_d ? B : A, out_d ? A : B, sq);
  else
    sweep_body<false, double, SW_TX, SW_TY>(b, lg, ntx, nty, E.ks_sweep, ph, ityprk, u, ff, v, ldv, v, sn, c,
                                            c + 3 * b.nnn, out_d ? B : A, out_d ? A : B, sq);
}

// two sub-iterations of every block
template <bool FF, bool FIRST>
__global__ void __launch_bounds__(S2_NC) __attribute__((amdgpu_waves_per_eu(2)))
k_impl_sweep2_batch(const ImplEnt *__restrict__ tab, int nb, Phys ph, const double *__restrict__ u,
                    const double *__restrict__ ff, const double *__restrict__ v, long ldv,
                    const double *__restrict__ sn_all, double *ws, double *d, int out_d, int rev) {
  __shared__ double sx[S2_LDS];
  __shared__ int flag[S2_NC / 64];
  if (threadIdx.x < S2_NC / 64) flag[threadIdx.x] = 0;
  __syncthreads();
  // one workgroup of a compute unit is in flight, so 32 on an XCD: in groups of
  // those 3.71 ms over 48 blocks of 40M cells, with an eighth of the grid each 3.79
  const unsigned wg = rev ? gridDim.x - 1 - xcd_grouped(32) : xcd_grouped(32);
  constexpr int PASS = FIRST ? IB_FIRST2 : IB_SWEEP2;
  const ImplEnt &E = tab[tab_find(tab, nb, PASS, wg)];
  const Blk b = uniform_blk(E.b);
  double *c = ws + 9 * b.npc;
  DView A = {d, ldv, 0}, B = {c + 4 * b.nnn, b.nnn, b.npc};
  sweep2_body<FF, FIRST>(b, (int)(wg - E.start[PASS]), (int)E.gx[PASS], (int)E.gy[PASS], E.ks_sweep2, ph, u, ff,
                  v, ldv, sn_all + 9 * b.npc, c, c + 3 * b.nnn, out_d ? B : A, out_d ? A : B, sx, (LdsFlag *)flag);
}

// the update in the first workgroups, d = 0 on the ghosts in those from cells on
__global__ void __launch_bounds__(TX *TY) k_impl_update_batch(const ImplEnt *__restrict__ tab, int nb, unsigned cells,
                                                              double *v, long ldv, double *d, int nvar) {
  if (blockIdx.x >= cells) {
    const unsigned sh = blockIdx.x - cells;
    const ImplEnt &E = tab[tab_find(tab, nb, IB_SHELL, sh)];
    const Blk b = E.b;
    shell_entries(b, (long)(sh - E.start[IB_SHELL]), b.npc, b.npc + b.nnn - 1, d, ldv, 5);
    return;
  }
  const unsigned wg = xcd_linear(cells);
  const ImplEnt &E = tab[tab_find(tab, nb, IB_CELL, wg)];
  update_body(E.b, tab_tile(E, IB_CELL, wg), v, ldv, d, nvar);
}

extern "C" int codens_implimf_3d_batch(int32_t nblk, const codens_block *blocks, const codens_phys *cp,
                                       const double *u, const double *dt, double *v, int64_t ldv, double *d,
                                       const double *ff, const double *mu, const double *mut, int32_t lmx,
                                       const double *sn_all, const double *vol, double dtpas, int32_t kfmg,
                                       int32_t ityprk, const double *cson, void *stream) {
  const char *what = "codens_implimf_3d_batch";
  if (nblk <= 0 || !blocks || !cp || !u || !dt || !v || !d || !mu || !mut || !sn_all || !vol || !cson ||
      (ityprk && !ff) || lmx < 0) {
    codens_set_error("%s: null or invalid argument", what);
    return CODENS_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  std::vector<ImplEnt> ent(nblk);
  std::vector<int32_t> key;
  std::vector<std::pair<long, long>> span(nblk);
  unsigned tot[IB_N] = {0};
  double one_wgs = 0., lanes = 0., cells = 0., two = 0., longest = 0.;
  int deepest = 0;
  auto slabs = [](int nz, int ks) { return (nz + ks - 1) / ks; };
  for (int l = 0; l < nblk; l++) {
    int rc = codens_check_block(&blocks[l], what);
    if (rc) return rc;
    const int32_t *w = (const int32_t *)&blocks[l];
    key.insert(key.end(), w, w + sizeof(codens_block) / sizeof(int32_t));
    Blk b = make_blk(&blocks[l]);
    span[l] = {b.npc, b.npc + b.nnn};
    ImplEnt &E = ent[l];
    E.b = b;
    dim3 cg = cell_grid(b);
    {
      std::lock_guard<std::mutex> lk(g_tile_mu);
      // the all-blocks launch holds shapes 0 and 1 (a forced 16 x 16 takes
      // the model's choice between them)
      E.tile = (g_tile_mode >= 0 && g_tile_mode < N_BATCH_TILES) ? g_tile_mode : tile_model(b);
    }
    const int tx = tile_tx(E.tile), ty = tile_ty(E.tile);
    unsigned ntx = (b.i2 - b.i1 + tx - 1) / tx, nty = (b.j2 - b.j1 + ty - 1) / ty;
    // full slabs: the launch has workgroups to spare, and these kernels give
    // the same values at any slab depth
    E.ks_coef = CK_KS;
    E.ks_sweep = SW_KS;
    const int nz = b.k2 - b.k1, ns2 = slabs(nz, S2_KS);
    auto over = [](int n, int o) { return (unsigned)((n + o - 1) / o); };
    const unsigned n2x = over(b.i2 - b.i1, s2_ox(false)), n2y = over(b.j2 - b.j1, s2_oy(false));
    E.ks_sweep2 = slabs(nz, ns2);  // even slabs of at most S2_KS planes
    // pairs or singles, for all blocks alike, as in pair_model: the steps of a
    // pair on a chip that is full, and at least those of the longest workgroup
    // (three blocks of 12 to 40 cells a side: two singles 55 us, a pair 77)
    const double wgs = (double)ntx * nty * slabs(nz, SW_KS);
    one_wgs += wgs;
    lanes += (double)ntx * nty * nz * SW_TX * SW_TY;
    cells += (double)(b.i2 - b.i1) * (b.j2 - b.j1) * nz;
    deepest = std::max(deepest, std::min(SW_KS, nz));
    two += (double)n2x * n2y * slabs(nz, E.ks_sweep2) * (E.ks_sweep2 + 2);
    longest = std::max(longest, E.ks_sweep2 + 2.);
    const unsigned nkz = (unsigned)((b.k2 - b.k1 + E.ks_sweep - 1) / E.ks_sweep);
    unsigned g[IB_N][3] = {{(unsigned)((b.nnn + 255) / 256), 1, 1},
                           {cg.x, cg.y, cg.z},
                           {ntx, nty, nkz},
                           {cg.x, cg.y, (unsigned)((b.k2 - b.k1 + E.ks_coef - 1) / E.ks_coef)},
                           {n2x, n2y, (unsigned)slabs(nz, E.ks_sweep2)},
                           {over(b.i2 - b.i1, s2_ox(true)), over(b.j2 - b.j1, s2_oy(true)),
                            (unsigned)slabs(nz, E.ks_sweep2)},
                           {shell_wgs(b), 1, 1}};
    for (int p = 0; p < IB_N; p++) {
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
  const double fill = one_wgs / codens_resident_workgroups(2);
  const double one = single_model(fill, fill <= 1. ? deepest : lanes / (SW_TX * SW_TY) / one_wgs, cells / lanes);
  const bool pairs =
      forced_tile() < 0 && PAIR_STEP * std::max(two / codens_resident_workgroups(1), longest) < 2. * one;
  for (int l = 0; l < nblk; l++) key.push_back(ent[l].tile);
  ImplEnt *tab = (ImplEnt *)codens_device_table(1, key, ent.data(), sizeof(ImplEnt) * nblk, st, what);
  if (!tab) return CODENS_EHIP;
  double *ws = (double *)codens_workspace(sizeof(double) * 9 * tot_n, 2);
  if (!ws) {
    codens_set_error("%s: workspace allocation failed", what);
    return CODENS_EHIP;
  }
  Phys ph = make_phys(cp);
  const ImplEnt *ct = tab;
  const int nb = nblk;
  const double *fx = ityprk ? ff : u;
  if (lmx < 1) hipLaunchKernelGGL(k_zero5_batch, dim3(tot[IB_ZERO]), dim3(256), 0, st, ct, nb, d, (long)ldv);
  {
    CodensTimed _tm("implimf_coef", st);
    hipLaunchKernelGGL(k_impl_coef_batch, dim3(tot[IB_COEF]), dim3(TX, TY), 0, st, ct, nb, ph, (const double *)v,
                       (long)ldv, mu, mut, dt, vol, cson, sn_all, dtpas, (int)kfmg, ws);
  }
  // the launches of implimf_common: sub-iteration 1, singles, then pairs
  const SweepPlan plan = sweep_plan(lmx, pairs);
  for (int s = 0; s < plan.n; s++) {
    const int out_d = (plan.n - 1 - s) % 2 == 0;
    if (s == 0 && plan.first2) {
      CodensTimed _tm("implimf_sweep1", st);
      hipLaunchKernelGGL((ityprk ? k_impl_sweep2_batch<true, true> : k_impl_sweep2_batch<false, true>),
                         dim3(tot[IB_FIRST2]), dim3(S2_NC), 0, st, ct, nb, ph, u, fx, (const double *)v, (long)ldv,
                         sn_all, ws, d, out_d, 0);
    } else if (s == 0) {
      CodensTimed _tm("implimf_sweep1", st);
      hipLaunchKernelGGL(k_impl_sweep1_batch, dim3(tot[IB_CELL]), dim3(TX, TY), 0, st, ct, nb, (int)ityprk, u, fx,
                         (long)ldv, ws, d, out_d);
    } else if (s <= plan.single) {
      CodensTimed _tm("implimf_sweep", st);
      hipLaunchKernelGGL(k_impl_sweep_batch, dim3(tot[IB_SWEEP]), dim3(SW_TX * SW_TY), 0, st, ct, nb, ph,
                         (int)ityprk, u, fx, (const double *)v, (long)ldv, sn_all, ws, d, out_d, s % 2);
    } else {
      CodensTimed _tm("implimf_sweep2", st);
      hipLaunchKernelGGL((ityprk ? k_impl_sweep2_batch<true, false> : k_impl_sweep2_batch<false, false>),
                         dim3(tot[IB_SWEEP2]), dim3(S2_NC), 0, st, ct, nb, ph, u, fx, (const double *)v, (long)ldv, sn_all, ws, d, out_d,
                         s % 2);
    }
  }
  {
    CodensTimed _tm("implimf_update", st);
    hipLaunchKernelGGL(k_impl_update_batch, dim3(tot[IB_CELL] + tot[IB_SHELL]), dim3(TX, TY), 0, st, ct, nb,
                       tot[IB_CELL], v, (long)ldv, d, 5);
  }
  return codens_check_launch(what);
}

// ---------------------------------------------------------------------------
// FP32 defect-correction form

// d = the FP32 increment widened to FP64, v += d (real cells)
__global__ void __launch_bounds__(TX *TY) k_impl_update_f32(Blk b, double *v, long ldv, double *d,
                                                            const float *__restrict__ df) {
  if (shell_layers(b, b.k2 - b.k1, b.npc, b.npc + b.nnn - 1, d, ldv, 5)) return;  // d = 0 on the ghosts
  CELL3_AT(b, xcd_block(false, b.k2 - b.k1))
  long n = b.idx(c[0], c[1], c[2]), m = n - b.npc;
#pragma unroll
  for (int e = 0; e < 5; e++) {
    double x = (double)df[e * b.nnn + m];
    d[e * ldv + n] = x;
    v[e * ldv + n] = v[e * ldv + n] + x;
  }
}

extern "C" int codens_implimf_3d_f32(const codens_block *cb, const codens_phys *cp, const double *u,
                                     const double *dt, double *v, int64_t ldv, double *d, const double *ff,
                                     const double *mu, const double *mut, int32_t lmx, const double *sn,
                                     const double *vol, double dtpas, int32_t kfmg, int32_t ityprk, const double *ps,
                                     const double *cson, void *stream) {
  const char *what = "codens_implimf_3d_f32";
  int rc = codens_check_block(cb, what);
  if (rc) return rc;
  if (!cp || !u || !dt || !v || !d || !mu || !mut || !sn || !vol || !cson || (ityprk && !ff) || lmx < 0) {
    codens_set_error("%s: invalid argument", what);
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  Phys ph = make_phys(cp);
  hipStream_t st = (hipStream_t)stream;
  const long nnn = b.nnn;
  // float planes: v 5, u 5, ff 5, sn 9, coefe 3 + diag 1, two increments 5 + 5
  float *wf = (float *)codens_workspace(sizeof(float) * 38 * nnn, 6);
  if (!wf) {
    codens_set_error("%s: workspace allocation failed", what);
    return CODENS_EHIP;
  }
  float *vF = wf, *uF = wf + 5 * nnn, *fF = wf + 10 * nnn, *snF = wf + 15 * nnn, *cF = wf + 24 * nnn;
  float *dgF = cF + 3 * nnn, *dA = wf + 28 * nnn, *dB = wf + 33 * nnn;
  dim3 g1((unsigned)((nnn + 255) / 256)), t1(256);
  if (lmx < 1) hipLaunchKernelGGL(k_zero5, g1, t1, 0, st, d, (long)ldv, (long)b.npc, (long)(b.npc + nnn - 1));
  dim3 g = cell_grid(b), t(TX, TY);
  {
    CodensTimed _tm("implimf32_coef", st);
    const int ks = coef_slab(b, g);
    dim3 gc(g.x, g.y, (unsigned)((b.k2 - b.k1 + ks - 1) / ks));
    hipLaunchKernelGGL(k_impl_coef_tiled<float>, gc, t, 0, st, b, ph, v, (long)ldv, mu, mut, dt, vol, cson, sn, dtpas,
                       (int)kfmg, cF, dgF, ks, F32Copies{u, ityprk ? ff : nullptr, vF, uF, fF, snF});
  }
  // storage-indexed views of the block-local float planes (entry n at n - npc)
  const float *vS = vF - b.npc, *uS = uF - b.npc, *fS = fF - b.npc;
  TView<float> A = {dA, nnn, b.npc}, B = {dB, nnn, b.npc};
  TView<float> last = A;
  int tile = 0;
  // as in the FP64 phase: sub-iteration 1 from d = 0, then the tiled sweeps
  for (int s = 1; s <= lmx; s++) {
    TView<float> out = (s % 2) ? A : B, in = (s % 2) ? B : A;
    if (s == 1) {
      CodensTimed _tm("implimf32_sweep1", st);
      hipLaunchKernelGGL(k_impl_sweep1<float>, g, t, 0, st, b, (int)ityprk, uS, ityprk ? fS : uS, nnn, dgF, out);
    } else {
      if (s == 2)
        tile = pick_tile<false, float>(b, st, ph, (int)ityprk, uS, ityprk ? fS : uS, vS, nnn, (const double *)nullptr,
                                       snF, cF, dgF, in, out);
      CodensTimed _tm("implimf32_sweep", st);
      launch_sweep<false, float>(tile, b, st, ph, (int)ityprk, uS, ityprk ? fS : uS, vS, nnn, (const double *)nullptr,
                                 snF, cF, dgF, in, out, s % 2 == 0);
    }
    last = out;
  }
  if (lmx > 0) {
    CodensTimed _tm("implimf32_update", st);
    hipLaunchKernelGGL(k_impl_update_f32, with_shell(b, g), t, 0, st, b, v, (long)ldv, d, (const float *)last.p);
  }
  return codens_check_launch(what);
}

extern "C" int codens_implimf_3d(const codens_block *cb, const codens_phys *cp, const double *u, const double *dt,
                                 double *v, int64_t ldv, double *d, const double *ff, const double *mu,
                                 const double *mut, int32_t lmx, const double *sn, const double *vol, double dtpas,
                                 int32_t kfmg, int32_t ityprk, const double *ps, const double *cson,
                                 void *stream) {
  // p of the real cells is re-derived from v with the zpres formula; ps unused
  return implimf_common(false, cb, cp, u, dt, v, ldv, 5, d, ff, mu, mut, lmx, sn, vol, dtpas, 0., kfmg, ityprk,
                        ps, cson, stream, "codens_implimf_3d");
}

extern "C" int codens_implimf_eu(const codens_block *cb, const codens_phys *cp, const double *u, const double *dt,
                                 double *v, int64_t ldv, int32_t nvar, double *d, const double *ff, int32_t lmx,
                                 const double *sn, const double *vol, double dt1min, int32_t kfmg, int32_t ityprk,
                                 const double *ps, const double *cson, void *stream) {
  return implimf_common(true, cb, cp, u, dt, v, ldv, nvar, d, ff, nullptr, nullptr, lmx, sn, vol, 1., dt1min, kfmg,
                        ityprk, ps, cson, stream, "codens_implimf_eu");
}
