// Viscous stresses and heat flux (zvisqc -> zgrad2 + zfluto) on gfx950.
// A workgroup owns a TX x TY tile of real cells and marches a slab of up to
// ZV_KS k-planes (fewer on small blocks, slab_depth).
// Per plane, the velocities (rho u)/rho (one division each, as
// zgrad2.f90:161-180 forms vx, vy, vz) and T of the tile and of its 1-cell
// ring go to LDS for the i and j neighbours; the own column's planes k-1
// and k+1 stay in registers.  Each cell gathers the Green-Gauss sums of its
// six faces (instead of the reference's +/- face scatter) in zgrad2's order
// (k, j, i; low face, then high), scales them by 1/(2 vol) and forms tau
// and q in registers: neither the velocity planes nor the twelve gradient
// arrays reach HBM.
#include "common.hpp"

using namespace codens;

// Bound by memory: 26 planes, on 256 x 128 x 64 91 us (4.8 TB/s), on 161 x 97 x
// 64 48 us on the same fields again and 63 on others (3.3 TB/s: its 600
// workgroups put three on some compute units and two on the others, of the four
// that fit), on blocks of 230,000 cells 17 us.  A plane's loads are all issued
// before one is used, the planes alternate between two LDS buffers with one
// barrier each, which waits for the LDS traffic only and not for the stores of
// the plane before (99, 66 and 19.7 us with the loads behind each other's
// divisions and two barriers that drained the stores).  The tile is the one
// that leaves fewest lanes idle over the block's i-j extent.
constexpr int ZV_KS = 8;

// velocity and temperature of a cell: loaded, then formed
struct ZvRaw {
  double r, m[3], t;
};
__device__ __forceinline__ ZvRaw zv_load(const double *__restrict__ v, long ldv, const double *__restrict__ temp,
                                         long n0, unsigned off) {
  ZvRaw x;
  x.r = ldp(v + n0, off);
#pragma unroll
  for (int e = 0; e < 3; e++) x.m[e] = ldp(v + ((e + 1) * ldv + n0), off);
  x.t = ldp(temp + n0, off);
  return x;
}
__device__ __forceinline__ void zv_q(const ZvRaw &x, double q[4]) {
  const double y = rcp64(x.r);
#pragma unroll
  for (int e = 0; e < 3; e++) q[e] = div_rcp(x.m[e], x.r, y);
  q[3] = x.t;
}

template <int X, int Y>
__global__ void __launch_bounds__(X *Y) k_zvisqc_tiled(Blk b, Phys ph, const double *__restrict__ sn,
                                                       const double *__restrict__ vol, const double *__restrict__ v,
                                                       long ldv, const double *__restrict__ temp,
                                                       const double *__restrict__ mu, const double *__restrict__ mut,
                                                       double *__restrict__ tq, int ks) {
  constexpr int PL = (X + 2) * (Y + 2);
  __shared__ double Lb[2][4][PL];
  const dim3 xb = xcd_block();
  const int t = threadIdx.x, tx = t % X, ty = t / X;
  const int i0 = b.i1 + xb.x * X, j0 = b.j1 + xb.y * Y;
  const int kb = b.k1 + xb.z * ks, ke = min(kb + ks, b.k2);
  const int i = i0 + tx, j = j0 + ty;
  const bool own = i < b.i2 && j < b.j2;
  // ring cell of this thread (t < 2 X + 2 Y), loaded where it lies in the
  // block's storage (the faces of real cells reach only the ghost layer)
  int ri = 0, rj = 0, rslot = 0;
  const bool ring = t < 2 * X + 2 * Y;
  if (ring) {
    int rx, ry;
    if (t < X) { ri = i0 + t; rj = j0 - 1; rx = t + 1; ry = 0; }
    else if (t < 2 * X) { ri = i0 + t - X; rj = j0 + Y; rx = t - X + 1; ry = Y + 1; }
    else if (t < 2 * X + Y) { ri = i0 - 1; rj = j0 + t - 2 * X; rx = 0; ry = t - 2 * X + 1; }
    else { ri = i0 + X; rj = j0 + t - 2 * X - Y; rx = X + 1; ry = t - 2 * X - Y + 1; }
    rslot = ry * (X + 2) + rx;
  }
  const int id2 = b.id1 + (int)b.nid - 1, jd2 = b.jd1 + (int)(b.nijd / b.nid) - 1;
  const bool rneed = ring && ri >= b.id1 && ri <= id2 && rj >= b.jd1 && rj <= jd2;
  const int slot = (ty + 1) * (X + 2) + (tx + 1);
  // own cell's slot also holds a cell past a partial tile's edge (the ghost
  // layer), which the neighbouring real cell reads
  const bool load = i <= b.i2 && j <= b.j2;
  // byte offsets in a plane of the own cell (clamped to the ghost layer: every
  // thread loads) and of the ring cell
  auto plane = [&](int x, int y) { return ((unsigned)(x - b.id1) + (unsigned)(y - b.jd1) * (unsigned)b.nid) * 8u; };
  const unsigned po = plane(min(i, b.i2), min(j, b.j2)), pr = rneed ? plane(ri, rj) : 0u;
  const long N = b.nnn;
  long mk = (long)(kb - b.kd1) * b.nijd;
  double qm[4], qc[4], qp[4], sk[3];  // sk: the k face below
  {
    const ZvRaw xm = zv_load(v, ldv, temp, b.npc + mk - b.nijd, po), xc = zv_load(v, ldv, temp, b.npc + mk, po);
#pragma unroll
    for (int cc = 0; cc < 3; cc++) sk[cc] = ldp(sn + ((3 * cc + 2) * N + mk), po);
    loads_issued();
    zv_q(xm, qm);
    zv_q(xc, qc);
  }
  for (int k = kb; k < ke; k++, mk += b.nijd) {
    double (*const Lq)[PL] = Lb[(k - kb) % 2];
    const long nk = b.npc + mk;
    // everything the plane needs
    ZvRaw xr;
    if (ring) xr = zv_load(v, ldv, temp, nk, pr);
    const ZvRaw xp = zv_load(v, ldv, temp, nk + b.nijd, po);
    double sl[3][3], sh[3][3];
#pragma unroll
    for (int cc = 0; cc < 3; cc++) {
      const double *const s = sn + (3 * cc * N + mk);
      sl[0][cc] = ldp(s, po);
      sh[0][cc] = ldp(s + 1, po);
      sl[1][cc] = ldp(s + N, po);
      sh[1][cc] = ldp(s + (N + b.nid), po);
      sl[2][cc] = sk[cc];
      sh[2][cc] = ldp(s + (2 * N + b.nijd), po);
    }
    const double vn = ldp(vol + nk, po), mun = ldp(mu + nk, po), mutn = ldp(mut + nk, po);
    loads_issued();
    if (load) {
#pragma unroll
      for (int q = 0; q < 4; q++) Lq[q][slot] = qc[q];
    }
    if (rneed) {
      double qr[4];
      zv_q(xr, qr);
#pragma unroll
      for (int q = 0; q < 4; q++) Lq[q][rslot] = qr[q];
    }
    zv_q(xp, qp);
    lds_sync();
    if (own) {
      double G[12];
#pragma unroll
      for (int q = 0; q < 12; q++) G[q] = 0.;
#pragma unroll
      for (int dd = 0; dd < 3; dd++) {
        const int d = 2 - dd;  // k faces, then j, then i (zgrad2.f90:181-457)
        const int a = d == 0 ? i : (d == 1 ? j : k), a1 = b.lo(d), a2 = b.hi(d);
        const int so = d == 0 ? 1 : (X + 2);
        double qlo[4], qhi[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
          qlo[q] = d == 2 ? qm[q] : Lq[q][slot - so];
          qhi[q] = d == 2 ? qp[q] : Lq[q][slot + so];
        }
        {  // low face (S at m): subtract
          bool bnd = (a == a1);
#pragma unroll
          for (int cc = 0; cc < 3; cc++) {
            double s = sl[d][cc];
#pragma unroll
            for (int q = 0; q < 4; q++) {
              double tt = bnd ? s * 2 * qlo[q] : (qc[q] + qlo[q]) * s;
              G[3 * q + cc] -= tt;
            }
          }
        }
        {  // high face (S at m+inc): add
          bool bnd = (a + 1 == a2);
#pragma unroll
          for (int cc = 0; cc < 3; cc++) {
            double s = sh[d][cc];
#pragma unroll
            for (int q = 0; q < 4; q++) {
              double tt = bnd ? s * 2 * qhi[q] : (qhi[q] + qc[q]) * s;
              G[3 * q + cc] += tt;
            }
          }
        }
      }
      // zgrad2.f90:463-485 (guard for non-positive volumes)
      double ts = copysign(0.5, -vn);
      double vols = (0.5 + ts) * 0.00001 + (0.5 - ts) * vn;
      double c0 = .5 / (vols + DBL_MIN);
#pragma unroll
      for (int q = 0; q < 12; q++) G[q] *= c0;
      // zfluto.f90:104-121
      double mt = mun + mutn;
      const double ds3 = 2. / 3.;
      double xx = G[0], xy = G[1], xz = G[2], yx = G[3], yy = G[4], yz = G[5], zx = G[6], zy = G[7], zz = G[8];
      *gp(tq + nk, po) = ds3 * mt * (2 * xx - yy - zz);
      *gp(tq + (ldv + nk), po) = mt * (xy + yx);
      *gp(tq + (2 * ldv + nk), po) = mt * (xz + zx);
      *gp(tq + (3 * ldv + nk), po) = ds3 * mt * (2 * yy - xx - zz);
      *gp(tq + (4 * ldv + nk), po) = mt * (yz + zy);
      *gp(tq + (5 * ldv + nk), po) = ds3 * mt * (2 * zz - xx - yy);
      double kq = ph.cp * (mun / ph.pr + mutn / ph.prt);
      *gp(tq + (6 * ldv + nk), po) = kq * G[9];
      *gp(tq + (7 * ldv + nk), po) = kq * G[10];
      *gp(tq + (8 * ldv + nk), po) = kq * G[11];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      qm[q] = qc[q];
      qc[q] = qp[q];
    }
#pragma unroll
    for (int cc = 0; cc < 3; cc++) sk[cc] = sh[2][cc];
  }
}

template <int X, int Y>
static void launch_zvisqc(const Blk &b, const Phys &ph, const double *sn, const double *vol, const double *v, long ldv,
                          const double *temp, const double *mu, const double *mut, double *tq, hipStream_t st) {
  dim3 g((b.i2 - b.i1 + X - 1) / X, (b.j2 - b.j1 + Y - 1) / Y, 1);
  const int ks = slab_depth((long)g.x * g.y, b.k2 - b.k1, ZV_KS);
  g.z = (unsigned)((b.k2 - b.k1 + ks - 1) / ks);
  hipLaunchKernelGGL((k_zvisqc_tiled<X, Y>), g, dim3(X * Y), 0, st, b, ph, sn, vol, v, ldv, temp, mu, mut, tq, ks);
}

extern "C" int codens_zvisqc(const codens_block *cb, const codens_phys *cp, const double *sn, const double *vol,
                             const double *v, int64_t ldv, const double *temp, const double *mu,
                             const double *mut, double *tq, void *stream) {
  int rc = codens_check_block(cb, "codens_zvisqc");
  if (rc) return rc;
  if (!cp || !sn || !vol || !v || !temp || !mu || !mut || !tq) {
    codens_set_error("codens_zvisqc: null argument");
    return CODENS_EINVAL;
  }
  Blk b = make_blk(cb);
  CodensTimed _tm("zvisqc", (hipStream_t)stream);
  // the shape with fewest lanes over the block's i-j extent, the wider one on a
  // tie (its rows are longer)
  auto lanes = [&](int x, int y) {
    return (long)((b.i2 - b.i1 + x - 1) / x * x) * ((b.j2 - b.j1 + y - 1) / y * y);
  };
  const long l64 = lanes(64, 4), l32 = lanes(32, 8), l16 = lanes(16, 16);
  auto *launch = l64 <= l32 && l64 <= l16 ? launch_zvisqc<64, 4> : l32 <= l16 ? launch_zvisqc<32, 8> : launch_zvisqc<16, 16>;
  launch(b, make_phys(cp), sn, vol, v, (long)ldv, temp, mu, mut, tq, (hipStream_t)stream);
  return codens_check_launch("codens_zvisqc");
}
