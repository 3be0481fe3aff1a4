// gp_vstep.hip — velocity stepping with and without continuous collision
// detection (integrators.rs:42-175, dynamics.rs:366-742), FP64, runtime
// topology, n_steps steps per launch: one instance per lane (vs_step_kernel)
// or per wave (vs_wave_kernel, below), the same bits.
//
// Per instance and step:
//  1. free velocity v_free = v + dt M^-1 (tau + springs - c(q, v)) by the
//     articulated-body algorithm without contact forces (dynamics.rs:375-395);
//  2. contacts: contact points inside a half-space and sphere colliders
//     touching one (collision_detection, dynamics.rs:546-606);
//  3. contact Jacobian rows [n; t; b] (v_o + w x p) over the joints from the
//     contact's body to the root (compose_contact_jacobian, dynamics.rs:747-820);
//  4. Y = M^-1 J^T, one articulated-body solve per row of J (zero velocity,
//     zero gravity, no springs: the solve returns M^-1 x);
//  5. G = J Y, g = J v_free and the impulse program of dynamics.rs:668-704:
//     minimise 1/2 x'Gx + g'x with (0.95 x_n, x_t, x_b) in the second-order
//     cone per contact, by a primal-dual interior-point method with
//     Nesterov-Todd scaling and Mehrotra's predictor-corrector;
//  6. v_next = v_free + Y x, q advanced with v_next.
// With continuous collision detection the step is cut at the earliest time
// a separated contact point, or the sphere of a body without contacts, would
// reach a half-space with v_next, and the rest of the step is stepped again;
// a sphere that ended a cut touches that half-space in the next round.
//
// One instance per lane: every per-lane array is a [k][Bp] column block of the
// bucket's scratch (vs_layout), so each access of a wavefront is one coalesced
// 512-byte line. One instance per wave: the arrays are in LDS (vw_layout).
#include "gp_cone.h"
#include "gp_plain_impl.h"

#ifndef GP_DYN_LDS
extern __shared__ __align__(16) unsigned char gp_dyn_lds[];
#define GP_DYN_LDS gp_dyn_lds
#endif

namespace gp {

namespace {

struct VsLane {
  const BucketArgs& a;
  int lane;
  VsLayout L;
  double* base;  // the instance's first working value, and the distance to its next
  int pitch;
  __device__ __forceinline__ Strided col(size_t off) const { return Strided{base + off * (size_t)pitch, pitch}; }
  __device__ __forceinline__ PlainCtx ctx() const { return PlainCtx{a, lane, base, pitch}; }
};

__device__ inline v3<double> mcol(const m3<double>& R, int k) { return {R.a[k], R.a[3 + k], R.a[6 + k]}; }

// world frames of every body from the parent-relative transforms the last
// plain_dynamics call left in scratch (PF_E = R^T, PF_R)
__device__ __forceinline__ void world_frames(const VsLane& V) {
  const BucketArgs& a = V.a;
  const PlainCtx X = V.ctx();
  for (int i = 0; i < a.nb; ++i) {
    const m3<double> E = X.ldm(PF_E, i);
    const m3<double> Rm{{E.a[0], E.a[3], E.a[6], E.a[1], E.a[4], E.a[7], E.a[2], E.a[5], E.a[8]}};
    const v3<double> p = X.ld3(PF_R, i);
    const int pr = a.parent[i];
    if (pr < 0) {
      X.stm(PF_RW, i, Rm);
      X.st3(PF_TW, i, p);
    } else {
      const m3<double> Rp = X.ldm(PF_RW, pr);
      X.stm(PF_RW, i, mul(Rp, Rm));
      X.st3(PF_TW, i, X.ld3(PF_TW, pr) + mul(Rp, p));
    }
  }
}

// The impulse program for nc contacts (G, g in scratch) -> x. Returns false
// when no finite iterate was produced.
__device__ bool cone_program(const VsLane& V, int nc) {
  const int m = 3 * nc;
  const VsLayout& L = V.L;
  Strided G = V.col(L.g), g = V.col(L.gv), Lc = V.col(L.l), x = V.col(L.x), z = V.col(L.z), s = V.col(L.s),
          rd = V.col(L.rd), lt = V.col(L.lt), xb = V.col(L.xb), dx = V.col(L.dx), dz = V.col(L.dz), ds = V.col(L.ds),
          xi = V.col(L.xi), rhs = V.col(L.rhs), Wc = V.col(L.w), Wic = V.col(L.wi);
  auto d = [](int k) { return k % 3 == 0 ? kConeMu : 1.0; };
  for (int c = 0; c < nc; ++c) {
    x[3 * c] = 1.0 / kConeMu; x[3 * c + 1] = 0.0; x[3 * c + 2] = 0.0;
    z[3 * c] = 1.0; z[3 * c + 1] = 0.0; z[3 * c + 2] = 0.0;
  }
  double gnorm = 0.0;
  for (int k = 0; k < m; ++k) gnorm = fmax(gnorm, fabs(g[k]));
  for (int k = 0; k < m; ++k) xb[k] = x[k];
  double best = 1e300;
  int since_best = 0;
  // Newton direction for a right-hand side xi of the scaled complementarity
  auto solve = [&]() {
    for (int c = 0; c < nc; ++c)
      for (int i = 0; i < 3; ++i) {
        double t = 0.0;
        for (int j = 0; j < 3; ++j) t += Wic[9 * c + 3 * i + j] * xi[3 * c + j];
        rhs[3 * c + i] = -rd[3 * c + i] + d(i) * t;
      }
    for (int r = 0; r < m; ++r) {
      double t = rhs[r];
      for (int k = 0; k < r; ++k) t -= Lc[r * m + k] * dx[k];
      dx[r] = t / Lc[r * m + r];
    }
    for (int r = m - 1; r >= 0; --r) {
      double t = dx[r];
      for (int k = r + 1; k < m; ++k) t -= Lc[k * m + r] * dx[k];
      dx[r] = t / Lc[r * m + r];
    }
    for (int c = 0; c < nc; ++c) {
      double a3[3];
      for (int i = 0; i < 3; ++i) {
        a3[i] = 0.0;
        for (int j = 0; j < 3; ++j) a3[i] += Wic[9 * c + 3 * i + j] * d(j) * dx[3 * c + j];
      }
      for (int i = 0; i < 3; ++i) {
        double t = 0.0;
        for (int j = 0; j < 3; ++j) t += Wic[9 * c + 3 * i + j] * (xi[3 * c + j] - a3[j]);
        dz[3 * c + i] = t;
      }
    }
  };
  auto max_step = [&](double scale) {
    double alpha = 1.0;
    for (int c = 0; c < nc; ++c) {
      const double sc[3] = {s[3 * c], s[3 * c + 1], s[3 * c + 2]}, dsc[3] = {ds[3 * c], ds[3 * c + 1], ds[3 * c + 2]};
      const double zc[3] = {z[3 * c], z[3 * c + 1], z[3 * c + 2]}, dzc[3] = {dz[3 * c], dz[3 * c + 1], dz[3 * c + 2]};
      alpha = fmin(alpha, scale * fmin(soc_max_step(sc, dsc), soc_max_step(zc, dzc)));
    }
    return alpha;
  };
  for (int it = 0; it < kConeMaxIter; ++it) {
    double gap = 0.0, rmax = 0.0, xmax = 0.0;
    for (int k = 0; k < m; ++k) s[k] = d(k) * x[k];
    for (int r = 0; r < m; ++r) {
      double t = g[r] - d(r) * z[r];
      for (int k = 0; k < m; ++k) t += G[r * m + k] * x[k];
      rd[r] = t;
      rmax = fmax(rmax, fabs(t));
      gap += s[r] * z[r];
      xmax = fmax(xmax, fabs(x[r]));
    }
    if (!isfinite(gap) || !isfinite(rmax)) break;
    const double gap_rel = gap / ((1.0 + gnorm) * (1.0 + xmax)), res_rel = rmax / (1.0 + gnorm);
    const double merit = fmax(gap_rel, res_rel);
    if (merit < best) {
      best = merit;
      since_best = 0;
      for (int k = 0; k < m; ++k) xb[k] = x[k];
    }
    if (gap_rel <= kConeGapTol && res_rel <= kConeResTol) break;
    if (++since_best > kConeStall) break;
    const double mug = gap / nc;
    for (int c = 0; c < nc; ++c) {
      const double sc[3] = {s[3 * c], s[3 * c + 1], s[3 * c + 2]}, zc[3] = {z[3 * c], z[3 * c + 1], z[3 * c + 2]};
      double W[9], Wi[9];
      nt_scaling(sc, zc, W, Wi);
      for (int k = 0; k < 9; ++k) { Wc[9 * c + k] = W[k]; Wic[9 * c + k] = Wi[k]; }
      for (int i = 0; i < 3; ++i) lt[3 * c + i] = W[3 * i] * zc[0] + W[3 * i + 1] * zc[1] + W[3 * i + 2] * zc[2];
    }
    // K = G + D W^-2 D, Cholesky in place in Lc (lower triangle)
    for (int r = 0; r < m; ++r)
      for (int k = 0; k <= r; ++k) Lc[r * m + k] = G[r * m + k];
    for (int c = 0; c < nc; ++c)
      for (int i = 0; i < 3; ++i)
        for (int j = 0; j <= i; ++j) {
          double t = 0.0;
          for (int k = 0; k < 3; ++k) t += Wic[9 * c + 3 * i + k] * Wic[9 * c + 3 * k + j];
          Lc[(3 * c + i) * m + 3 * c + j] += d(i) * t * d(j);
        }
    bool pd = true;
    for (int j = 0; j < m && pd; ++j) {
      double t = Lc[j * m + j];
      for (int k = 0; k < j; ++k) t -= Lc[j * m + k] * Lc[j * m + k];
      if (!(t > 0.0)) { pd = false; break; }
      const double ljj = sqrt(t);
      Lc[j * m + j] = ljj;
      for (int r = j + 1; r < m; ++r) {
        double u = Lc[r * m + j];
        for (int k = 0; k < j; ++k) u -= Lc[r * m + k] * Lc[j * m + k];
        Lc[r * m + j] = u / ljj;
      }
    }
    if (!pd) break;
    // predictor
    for (int k = 0; k < m; ++k) xi[k] = -lt[k];
    solve();
    for (int k = 0; k < m; ++k) ds[k] = d(k) * dx[k];
    const double alpha_a = max_step(1.0);
    double sz = 0.0;
    for (int k = 0; k < m; ++k) sz += (s[k] + alpha_a * ds[k]) * (z[k] + alpha_a * dz[k]);
    const double ratio = sz / gap, sigma = ratio * ratio * ratio;
    // corrector: xi = lt \ (sigma mu e - lt o lt - (W^-1 ds) o (W dz))
    for (int c = 0; c < nc; ++c) {
      double a3[3], b3[3];
      for (int i = 0; i < 3; ++i) {
        a3[i] = Wic[9 * c + 3 * i] * ds[3 * c] + Wic[9 * c + 3 * i + 1] * ds[3 * c + 1] + Wic[9 * c + 3 * i + 2] * ds[3 * c + 2];
        b3[i] = Wc[9 * c + 3 * i] * dz[3 * c] + Wc[9 * c + 3 * i + 1] * dz[3 * c + 1] + Wc[9 * c + 3 * i + 2] * dz[3 * c + 2];
      }
      const double l0 = lt[3 * c], l1 = lt[3 * c + 1], l2 = lt[3 * c + 2];
      const double w0 = sigma * mug - (l0 * l0 + l1 * l1 + l2 * l2) - (a3[0] * b3[0] + a3[1] * b3[1] + a3[2] * b3[2]);
      const double w1 = -(2.0 * l0 * l1) - (a3[0] * b3[1] + b3[0] * a3[1]);
      const double w2 = -(2.0 * l0 * l2) - (a3[0] * b3[2] + b3[0] * a3[2]);
      const double y0 = (l0 * w0 - l1 * w1 - l2 * w2) / soc_det(l0, l1, l2);
      xi[3 * c] = y0;
      xi[3 * c + 1] = (w1 - y0 * l1) / l0;
      xi[3 * c + 2] = (w2 - y0 * l2) / l0;
    }
    solve();
    for (int k = 0; k < m; ++k) ds[k] = d(k) * dx[k];
    const double alpha = max_step(0.99);
    for (int k = 0; k < m; ++k) {
      x[k] += alpha * dx[k];
      z[k] += alpha * dz[k];
    }
  }
  bool ok = best < 1e300;
  for (int k = 0; k < m; ++k) {
    x[k] = xb[k];
    ok = ok && isfinite(x[k]);
  }
  return ok;
}

// motion subspace column k of body i's joint in world Plücker coordinates
// (angular w, linear velocity of the point at the world origin)
__device__ inline void world_column(int kind, const m3<double>& Rw, v3<double> o, int k, v3<double>& w,
                                    v3<double>& v0) {
  if (kind == K_REV) {
    w = mcol(Rw, 2);
    v0 = cross(o, w);
  } else if (kind == K_PRI) {
    w = v3<double>{0, 0, 0};
    v0 = mcol(Rw, 2);
  } else if (k < 3) {
    w = mcol(Rw, k);
    v0 = cross(o, w);
  } else {
    w = v3<double>{0, 0, 0};
    v0 = mcol(Rw, k - 3);
  }
}

// A rigid inertia (J about the body's origin, c = m com, in the body's frame)
// at the world's origin: J there and m com (inertia.rs:106-134)
__device__ __forceinline__ void world_inertia(const m3<double>& R, v3<double> p, const double (&J)[9], v3<double> c,
                                              double mass, double (&Jw)[9], v3<double>& cw) {
  const v3<double> Rmc = mul(R, c);
  const v3<double> mp = mass * p;
  double RJ[9];
  for (int r = 0; r < 3; ++r)
    for (int k = 0; k < 3; ++k) RJ[3 * r + k] = R.a[3 * r] * J[k] + R.a[3 * r + 1] * J[3 + k] + R.a[3 * r + 2] * J[6 + k];
  const double rm[3] = {Rmc.x, Rmc.y, Rmc.z}, pp[3] = {p.x, p.y, p.z}, mpp[3] = {mp.x, mp.y, mp.z};
  double Y[9];
  for (int r = 0; r < 3; ++r)
    for (int k = 0; k < 3; ++k) Y[3 * r + k] = rm[r] * pp[k] + rm[k] * pp[r] + mpp[r] * pp[k];
  const double trY = Y[0] + Y[4] + Y[8];
  for (int r = 0; r < 3; ++r)
    for (int k = 0; k < 3; ++k)
      Jw[3 * r + k] = RJ[3 * r] * R.a[3 * k] + RJ[3 * r + 1] * R.a[3 * k + 1] + RJ[3 * r + 2] * R.a[3 * k + 2] -
                      Y[3 * r + k] + (r == k ? trY : 0.0);
  cw = Rmc + mp;
}
// F = Ic s (momentum.rs:17-32)
__device__ __forceinline__ void composite_force(double Jxx, double Jyy, double Jzz, double Jxy, double Jxz, double Jyz,
                                                v3<double> c, double mass, v3<double> sw, v3<double> sv, v3<double>& Fa,
                                                v3<double>& Fl) {
  const v3<double> Jw{Jxx * sw.x + Jxy * sw.y + Jxz * sw.z, Jxy * sw.x + Jyy * sw.y + Jyz * sw.z,
                      Jxz * sw.x + Jyz * sw.y + Jzz * sw.z};
  Fa = Jw + cross(c, sv);
  Fl = mass * sv - cross(c, sw);
}

// Mass matrix by the composite-rigid-body algorithm in world coordinates
// (the quantity of mechanism.rs:637-696), then its Cholesky factor, lower
// triangle in place (row-major nv x nv). World frames of the current q must be
// in scratch. Composite inertias (J about the world origin, m c, m) are kept
// in the first ten articulated-inertia fields, free at this point.
__device__ bool mass_matrix_cholesky(const VsLane& V, Strided Mm) {
  const BucketArgs& a = V.a;
  const int lane = V.lane, nb = a.nb, nv = a.nv, Bp = a.Bp;
  const PlainCtx X = V.ctx();
  for (int i = 0; i < nb; ++i) {  // world inertias (inertia.rs:106-134)
    const m3<double> R = X.ldm(PF_RW, i);
    const v3<double> p = X.ld3(PF_TW, i);
    const double J[9] = {X.bpar(BF_J, i), X.bpar(BF_J + 3, i), X.bpar(BF_J + 4, i),
                         X.bpar(BF_J + 3, i), X.bpar(BF_J + 1, i), X.bpar(BF_J + 5, i),
                         X.bpar(BF_J + 4, i), X.bpar(BF_J + 5, i), X.bpar(BF_J + 2, i)};
    const double mass = X.bpar(BF_M, i);
    double Jw[9];
    v3<double> cw;
    world_inertia(R, p, J, v3<double>{X.bpar(BF_C, i), X.bpar(BF_C + 1, i), X.bpar(BF_C + 2, i)}, mass, Jw, cw);
    X.s(PF_IA, i) = Jw[0]; X.s(PF_IA + 1, i) = Jw[4]; X.s(PF_IA + 2, i) = Jw[8];
    X.s(PF_IA + 3, i) = Jw[1]; X.s(PF_IA + 4, i) = Jw[2]; X.s(PF_IA + 5, i) = Jw[5];
    X.st3(PF_IA + 6, i, cw);
    X.s(PF_IA + 9, i) = mass;
  }
  for (int i = nb - 1; i > 0; --i) {  // composite inertias, leaves to root
    const int pr = a.parent[i];
    if (pr < 0) continue;
    for (int f = 0; f < 10; ++f) X.s(PF_IA + f, pr) += X.s(PF_IA + f, i);
  }
  for (int r = 0; r < nv; ++r)
    for (int c = 0; c <= r; ++c) Mm[r * nv + c] = 0.0;
  for (int i = 0; i < nb; ++i) {
    const int ki = a.kind[i * Bp + lane], ni = ki == K_FLOAT ? 6 : (ki == K_FIXED ? 0 : 1);
    if (ni == 0) continue;
    const double Jxx = X.s(PF_IA, i), Jyy = X.s(PF_IA + 1, i), Jzz = X.s(PF_IA + 2, i);
    const double Jxy = X.s(PF_IA + 3, i), Jxz = X.s(PF_IA + 4, i), Jyz = X.s(PF_IA + 5, i);
    const v3<double> c = X.ld3(PF_IA + 6, i);
    const double mass = X.s(PF_IA + 9, i);
    const m3<double> Ri = X.ldm(PF_RW, i);
    const v3<double> oi = X.ld3(PF_TW, i);
    for (int ca = 0; ca < ni; ++ca) {
      v3<double> sw, sv;
      world_column(ki, Ri, oi, ca, sw, sv);
      v3<double> Fa, Fl;
      composite_force(Jxx, Jyy, Jzz, Jxy, Jxz, Jyz, c, mass, sw, sv, Fa, Fl);
      const int row = a.voff[i] + ca;
      for (int j = i; j >= 0; j = a.parent[j]) {
        const int kj = a.kind[j * Bp + lane], nj = kj == K_FLOAT ? 6 : (kj == K_FIXED ? 0 : 1);
        const m3<double> Rj = X.ldm(PF_RW, j);
        const v3<double> oj = X.ld3(PF_TW, j);
        for (int cb2 = 0; cb2 < nj; ++cb2) {
          const int col = a.voff[j] + cb2;
          if (col > row) continue;
          v3<double> tw, tv;
          world_column(kj, Rj, oj, cb2, tw, tv);
          Mm[row * nv + col] = dot(Fa, tw) + dot(Fl, tv);
        }
      }
    }
  }
  bool pd = true;
  for (int j = 0; j < nv; ++j) {
    double t = Mm[j * nv + j];
    for (int k = 0; k < j; ++k) t -= Mm[j * nv + k] * Mm[j * nv + k];
    if (!(t > 0.0)) {
      pd = false;
      t = 1.0;
    }
    const double ljj = sqrt(t);
    Mm[j * nv + j] = ljj;
    for (int r = j + 1; r < nv; ++r) {
      double u = Mm[r * nv + j];
      for (int k = 0; k < j; ++k) u -= Mm[r * nv + k] * Mm[j * nv + k];
      Mm[r * nv + j] = u / ljj;
    }
  }
  return pd;
}

// Contacts at the world frames in scratch: points inside a half-space, then
// touching spheres (normals, points and bodies in L.cn, L.cp, L.cb); returns
// their number.
__device__ __forceinline__ int find_contacts(const VsLane& V, int forced_body, int forced_h) {
  const BucketArgs& a = V.a;
  const int lane = V.lane, nb = a.nb, Bp = a.Bp;
  const VsLayout& L = V.L;
  const PlainCtx X = V.ctx();
  Strided cn = V.col(L.cn), cpn = V.col(L.cp), cb = V.col(L.cb);
  int nc = 0;
  auto add = [&](v3<double> n, v3<double> p, int body) {
    cn[3 * nc] = n.x; cn[3 * nc + 1] = n.y; cn[3 * nc + 2] = n.z;
    cpn[3 * nc] = p.x; cpn[3 * nc + 1] = p.y; cpn[3 * nc + 2] = p.z;
    cb[nc] = (double)body;
    ++nc;
  };
  for (int i = 0; i < nb; ++i) {
    const m3<double> Rw = X.ldm(PF_RW, i);
    const v3<double> tw = X.ld3(PF_TW, i);
    for (int cc = a.cstart[i]; cc < a.cstart[i + 1]; ++cc) {
      auto cpar = [&](int f) { return a.cp[((size_t)f * a.nc + cc) * Bp + lane]; };
      const v3<double> pw = mul(Rw, v3<double>{cpar(CF_P), cpar(CF_P + 1), cpar(CF_P + 2)}) + tw;
      for (int hh = 0; hh < a.nh; ++hh) {
        auto hpar = [&](int f) { return a.hp[((size_t)f * a.nh + hh) * Bp + lane]; };
        const v3<double> pt{hpar(HF_POINT), hpar(HF_POINT + 1), hpar(HF_POINT + 2)};
        const v3<double> n{hpar(HF_NORMAL), hpar(HF_NORMAL + 1), hpar(HF_NORMAL + 2)};
        if (dot(pw - pt, n) <= kInsideMargin) add(n, pw, i);
      }
    }
  }
  for (int i = 0; i < nb; ++i) {
    const int sl = a.sphere_of[i];
    if (sl < 0) continue;
    auto spar = [&](int f) { return a.shp[((size_t)f * a.ns + sl) * Bp + lane]; };
    if (spar(SH_ON) == 0.0) continue;
    const m3<double> Rw = X.ldm(PF_RW, i);
    const v3<double> center = mul(Rw, v3<double>{spar(SH_C), spar(SH_C + 1), spar(SH_C + 2)}) + X.ld3(PF_TW, i);
    const double r = spar(SH_R);
    for (int hh = 0; hh < a.nh; ++hh) {
      auto hpar = [&](int f) { return a.hp[((size_t)f * a.nh + hh) * Bp + lane]; };
      const v3<double> pt{hpar(HF_POINT), hpar(HF_POINT + 1), hpar(HF_POINT + 2)};
      const v3<double> n{hpar(HF_NORMAL), hpar(HF_NORMAL + 1), hpar(HF_NORMAL + 2)};
      const double dist = dot(center - pt, n);
      if (dist <= r || (i == forced_body && hh == forced_h)) add(n, center - dist * n, i);
    }
  }
  return nc;
}

// The rows [n; t; b] of contact ci's Jacobian (3 x nv), by put(row, column,
// value) for the columns of the joints from the contact's body to the root.
template <class Put>
__device__ __forceinline__ void contact_jacobian(const VsLane& V, int ci, Put put_row) {
  const BucketArgs& a = V.a;
  const int lane = V.lane, Bp = a.Bp;
  const PlainCtx X = V.ctx();
  Strided cn = V.col(V.L.cn), cpn = V.col(V.L.cp), cb = V.col(V.L.cb);
  const v3<double> n{cn[3 * ci], cn[3 * ci + 1], cn[3 * ci + 2]};
  const v3<double> p{cpn[3 * ci], cpn[3 * ci + 1], cpn[3 * ci + 2]};
  v3<double> t = cross(n, v3<double>{1.0, 0.0, 0.0});
  double tn = sqrt(dot(t, t));
  if (tn == 0.0) {
    t = cross(n, v3<double>{0.0, 1.0, 0.0});
    tn = sqrt(dot(t, t));
  }
  t = v3<double>{t.x / tn, t.y / tn, t.z / tn};
  v3<double> bb = cross(n, t);
  const double bn = sqrt(dot(bb, bb));
  bb = v3<double>{bb.x / bn, bb.y / bn, bb.z / bn};
  auto put = [&](int colk, v3<double> vel) {
    put_row(0, colk, dot(n, vel));
    put_row(1, colk, dot(t, vel));
    put_row(2, colk, dot(bb, vel));
  };
  for (int jb = (int)cb[ci]; jb >= 0; jb = a.parent[jb]) {
    const int kd = a.kind[jb * Bp + lane], vo = a.voff[jb];
    const m3<double> Rw = X.ldm(PF_RW, jb);
    const v3<double> rel = p - X.ld3(PF_TW, jb);
    if (kd == K_REV) {
      put(vo, cross(mcol(Rw, 2), rel));
    } else if (kd == K_PRI) {
      put(vo, mcol(Rw, 2));
    } else if (kd == K_FLOAT) {
      for (int k = 0; k < 3; ++k) put(vo + k, cross(mcol(Rw, k), rel));
      for (int k = 0; k < 3; ++k) put(vo + 3 + k, mcol(Rw, k));
    }
  }
}

// dynamics_discrete for one lane at (q, v) with step h: new velocities in
// L.vn. Returns false on a non-positive D or a failed impulse program.
// *n_contacts = the touching contacts (their bodies in L.cb). forced_body /
// forced_h: a sphere the collision loop has just moved onto half-space
// forced_h is in contact with it (its distance is zero in exact arithmetic;
// rounding may leave it some ulps above the plane).
__device__ bool vs_dynamics(const VsLane& V, Strided q, Strided v, Strided tau, double h, int* n_contacts,
                            int forced_body, int forced_h) {
  const BucketArgs& a = V.a;
  const int lane = V.lane, nv = a.nv, nb = a.nb, Bp = a.Bp;
  const VsLayout& L = V.L;
  const PlainCtx X = V.ctx();
  Strided vfree = V.col(L.vfree), zero = V.col(L.zero), colv = V.col(L.col), out = V.col(L.out), vn = V.col(L.vn);
  Strided J = V.col(L.j), Y = V.col(L.y), G = V.col(L.g), gv = V.col(L.gv), x = V.col(L.x);
  Strided cn = V.col(L.cn), cpn = V.col(L.cp), cb = V.col(L.cb);
  // 1. free velocity: no contact forces on this path (dynamics.rs:377-383)
  bool ok = plain_dynamics(a, lane, q, v, tau, out, false);
  for (int k = 0; k < nv; ++k) vfree[k] = v[k] + h * out[k];
  world_frames(V);
  // 2. contacts
  const int nc = find_contacts(V, forced_body, forced_h);
  *n_contacts = nc;
  if (nc == 0) {
    for (int k = 0; k < nv; ++k) vn[k] = vfree[k];
    return ok;
  }
  const int m = 3 * nc;
  // 3. Jacobian rows
  for (int ci = 0; ci < nc; ++ci) {
    for (int r = 0; r < 3; ++r)
      for (int k = 0; k < nv; ++k) J[(3 * ci + r) * nv + k] = 0.0;
    contact_jacobian(V, ci, [&](int r, int k, double x) { J[(3 * ci + r) * nv + k] = x; });
  }
  // 4. Y = M^-1 J^T with M from the composite-rigid-body algorithm and its
  // Cholesky factor (M is symmetric positive definite)
  Strided Mm = V.col(L.mm);
  ok = mass_matrix_cholesky(V, Mm) && ok;
  for (int r = 0; r < m; ++r) {
    for (int k = 0; k < nv; ++k) {  // L y = J_r
      double t = J[r * nv + k];
      for (int l = 0; l < k; ++l) t -= Mm[k * nv + l] * out[l];
      out[k] = t / Mm[k * nv + k];
    }
    for (int k = nv - 1; k >= 0; --k) {  // L^T y = .
      double t = out[k];
      for (int l = k + 1; l < nv; ++l) t -= Mm[l * nv + k] * Y[l * m + r];
      Y[k * m + r] = t / Mm[k * nv + k];
    }
  }
  // 5. G = J Y, g = J v_free, impulses
  for (int r = 0; r < m; ++r) {
    for (int c = 0; c <= r; ++c) {
      double t = 0.0;
      for (int k = 0; k < nv; ++k) t += J[r * nv + k] * Y[k * m + c];
      G[r * m + c] = t;
      G[c * m + r] = t;
    }
    double t = 0.0;
    for (int k = 0; k < nv; ++k) t += J[r * nv + k] * vfree[k];
    gv[r] = t;
  }
  ok = cone_program(V, nc) && ok;
  // 6. v_next = v_free + M^-1 J^T x
  for (int k = 0; k < nv; ++k) {
    double t = vfree[k];
    for (int r = 0; r < m; ++r) t += Y[k * m + r] * x[r];
    vn[k] = t;
  }
  return ok;
}

// earliest time within which a separated contact point, or the sphere of a
// body without contacts, reaches a half-space at the new velocities
// (integrators.rs:62-158); world frames of the current q are in scratch.
// *hit_body / *hit_h: the sphere and half-space of that time (-1: a point).
__device__ __forceinline__ double earliest_collision(const VsLane& V, int nc, int* hit_body, int* hit_h) {
  const BucketArgs& a = V.a;
  const int lane = V.lane, Bp = a.Bp;
  const PlainCtx X = V.ctx();
  Strided vn = V.col(V.L.vn), cb = V.col(V.L.cb);
  double earliest = 1e300;
  *hit_body = -1;
  *hit_h = -1;
  auto hit = [&](v3<double> p, v3<double> vel, double radius, int sphere_body) {
    for (int hh = 0; hh < a.nh; ++hh) {
      auto hpar = [&](int f) { return a.hp[((size_t)f * a.nh + hh) * Bp + lane]; };
      const v3<double> pt{hpar(HF_POINT), hpar(HF_POINT + 1), hpar(HF_POINT + 2)};
      const v3<double> n{hpar(HF_NORMAL), hpar(HF_NORMAL + 1), hpar(HF_NORMAL + 2)};
      const double vdn = dot(vel, n);
      if (vdn == 0.0) continue;
      const double dist = dot(p - pt, n) - radius;
      if (dist <= 0.0) continue;
      const double t = dist / -vdn;
      if (t < earliest && t > 0.0) {
        earliest = t;
        *hit_body = sphere_body;
        *hit_h = hh;
      }
    }
  };
  for (int i = 0; i < a.nb; ++i) {
    // world twist (w, velocity of the point at the origin) from the new velocities
    const int kd = a.kind[i * Bp + lane], vo = a.voff[i], pr = a.parent[i];
    const m3<double> Rw = X.ldm(PF_RW, i);
    const v3<double> o = X.ld3(PF_TW, i);
    v3<double> w = pr < 0 ? v3<double>{0, 0, 0} : X.ld3(PF_VEL, pr);
    v3<double> v0 = pr < 0 ? v3<double>{0, 0, 0} : X.ld3(PF_VEL + 3, pr);
    if (kd == K_REV) {
      const v3<double> ax = vn[vo] * mcol(Rw, 2);
      w = w + ax;
      v0 = v0 + cross(o, ax);
    } else if (kd == K_PRI) {
      v0 = v0 + vn[vo] * mcol(Rw, 2);
    } else if (kd == K_FLOAT) {
      const v3<double> ww = mul(Rw, v3<double>{vn[vo], vn[vo + 1], vn[vo + 2]});
      w = w + ww;
      v0 = v0 + mul(Rw, v3<double>{vn[vo + 3], vn[vo + 4], vn[vo + 5]}) + cross(o, ww);
    }
    X.st3(PF_VEL, i, w);
    X.st3(PF_VEL + 3, i, v0);
    for (int cc = a.cstart[i]; cc < a.cstart[i + 1]; ++cc) {
      auto cpar = [&](int f) { return a.cp[((size_t)f * a.nc + cc) * Bp + lane]; };
      const v3<double> pw = mul(Rw, v3<double>{cpar(CF_P), cpar(CF_P + 1), cpar(CF_P + 2)}) + o;
      hit(pw, v0 + cross(w, pw), 0.0, -1);
    }
  }
  for (int i = 0; i < a.nb; ++i) {
    const int sl = a.sphere_of[i];
    if (sl < 0) continue;
    auto spar = [&](int f) { return a.shp[((size_t)f * a.ns + sl) * Bp + lane]; };
    if (spar(SH_ON) == 0.0) continue;
    bool touching = false;
    for (int c = 0; c < nc; ++c) touching = touching || (int)cb[c] == i;
    if (touching) continue;
    const v3<double> center = mul(X.ldm(PF_RW, i), v3<double>{spar(SH_C), spar(SH_C + 1), spar(SH_C + 2)}) + X.ld3(PF_TW, i);
    hit(center, X.ld3(PF_VEL + 3, i) + cross(X.ld3(PF_VEL, i), center), spar(SH_R), i);
  }
  return earliest;
}

// ---------------------------------------------------------------- one instance per wave
// The same step with the 64 lanes of a wave sharing one instance. Per lane the
// step is a chain of dependent loads from a working set of some 30 KB an
// instance, 2 MB a wave; here it is in LDS, the impulse program's rows and
// contacts go over the lanes, and what is serial (the articulated-body
// pass, contact detection, the collision loop) is done by all lanes alike.
// Four steps of 512 standing quadrupeds: 15.7 ms by vs_step_kernel, 1.94 ms here.
// What bounds it is still the serial chain: an interior-point iteration of 12
// rows is some 40,000 cycles (the factor 12,000, its two solves 13,000 each, a
// division or a square root and an LDS round trip per row), 15 to 20 of them a
// step; a step in flight is 65 us of articulated-body pass. Rows of the factor in
// registers with every loop unrolled took 2.65 ms: a lone wave then waits
// for instructions. Two waves per SIMD (256 registers) took 2.04 ms and gain
// 15 % only where the lane kernel is the faster one.
//
// Every value is formed by the operations of vs_step_kernel in their order, so
// the results are the same bits: lanes take different rows (or contacts), never
// parts of one sum. A column-oriented triangular solve subtracts a row's
// products in the order of the row-oriented one; where that order needs the
// last solved value first (the backward solve) and in sums over rows, the sum
// is formed by all lanes from values broadcast one after another.
//
// wlanes(f): f(lane) on every lane; between two such phases, what one lane
// wrote to LDS can be read by another (one wave executes its LDS instructions
// in order; the fence keeps the compiler from moving them). The host build
// runs the lanes of a phase in turn, from the launch's first thread.
#ifdef __HIP_DEVICE_COMPILE__
template <class F> __device__ __forceinline__ void wlanes(F f) {
  f((int)threadIdx.x);
  asm volatile("" ::: "memory");
}
struct LaneD {  // one double per lane
  double r;
  __device__ __forceinline__ double& operator[](int) { return r; }
  __device__ __forceinline__ double at(int k) const {  // lane k's, k the same on all lanes
    const long long b = __builtin_bit_cast(long long, r);
    const int lo = __builtin_amdgcn_readlane((int)b, k), hi = __builtin_amdgcn_readlane((int)(b >> 32), k);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (long long)(unsigned)lo);
  }
};
#else
template <class F> __device__ inline void wlanes(F f) {
  for (int l = 0; l < 64; ++l) f(l);
}
struct LaneD {
  double r[64];
  __device__ double& operator[](int l) { return r[l]; }
  __device__ double at(int k) const { return r[k]; }
};
#endif

// LDS of one instance, in doubles. First the fields of vs_layout that the
// shared parts of the step use (per-body fields, the loop's state, contacts).
// K: the lower triangle (and diagonal) of the
// factor, and G's upper one a column to its right, in one m x pitch block
// (pitch odd: a column's entries spread over the banks). The program's vectors
// and scalings take J's place once G and g are formed.
struct VwLayout {
  VsLayout v;  // the shared fields' offsets (the others are not used)
  int pitch;
  int k, j, y, mm, gv, vfree, ic, x, z, s, rd, lt, xb, xi, rhs, w, wi, total;
};
__host__ __device__ inline VwLayout vw_layout(int nb, int nq, int nv, int cmax) {
  VwLayout L{};
  const int m = 3 * cmax;
  L.pitch = (m + 1) | 1;
  int at = NPF * nb;
  L.v.cmax = cmax;
  L.v.m = m;
  auto shared = [&](size_t& f, int n) { f = at; at += n; };
  shared(L.v.out, nv); shared(L.v.qc, nq); shared(L.v.vc, nv); shared(L.v.vn, nv);
  shared(L.v.cn, 3 * cmax); shared(L.v.cp, 3 * cmax); shared(L.v.cb, cmax);
  auto take = [&](int n) { const int o = at; at += n; return o; };
  L.k = take(m * L.pitch);
  L.y = take(nv * m);
  L.mm = take(nv * (nv | 1));
  L.gv = take(m);
  L.vfree = take(nv);
  L.ic = take(10 * nb);
  L.j = at;
  int end = at + m * nv;
  L.x = take(m); L.z = take(m); L.s = take(m); L.rd = take(m); L.lt = take(m); L.xb = take(m); L.xi = take(m);
  L.rhs = take(m);
  L.w = take(9 * cmax); L.wi = take(9 * cmax);
  L.total = at > end ? at : end;
  return L;
}

// x as rounded to a double: not contracted with what uses it (the lane kernel
// forms it outside of the loop that uses it, so the compiler does not either)
__device__ __forceinline__ double rounded(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" : "+v"(x));
#endif
  return x;
}

struct VsWave {
  const VsLane& V;
  VwLayout L;
  double* lds;
  int m;  // rows of this round's program
  __device__ __forceinline__ double& low(int r, int k) const { return lds[L.k + r * L.pitch + k]; }       // k <= r
  __device__ __forceinline__ double& up(int r, int c) const { return lds[L.k + r * L.pitch + c + 1]; }    // r <= c
  __device__ __forceinline__ double g(int r, int c) const { return r <= c ? up(r, c) : up(c, r); }
};

// mass_matrix_cholesky with the bodies, rows and factor rows over the lanes
__device__ __forceinline__ bool vw_mass_matrix(const VsWave& W) {
  const BucketArgs& a = W.V.a;
  const int lane = W.V.lane, nb = a.nb, nv = a.nv, Bp = a.Bp, mp_ = nv | 1;
  double* const ic = W.lds + W.L.ic;
  double* const Mm = W.lds + W.L.mm;
  const PlainCtx X = W.V.ctx();
  wlanes([&](int i) {
    if (i >= nb) return;
    const m3<double> R = X.ldm(PF_RW, i);
    const v3<double> p = X.ld3(PF_TW, i);
    const double J[9] = {X.bpar(BF_J, i), X.bpar(BF_J + 3, i), X.bpar(BF_J + 4, i),
                         X.bpar(BF_J + 3, i), X.bpar(BF_J + 1, i), X.bpar(BF_J + 5, i),
                         X.bpar(BF_J + 4, i), X.bpar(BF_J + 5, i), X.bpar(BF_J + 2, i)};
    const double mass = X.bpar(BF_M, i);
    v3<double> cw;
    double Jw[9];
    world_inertia(R, p, J, v3<double>{X.bpar(BF_C, i), X.bpar(BF_C + 1, i), X.bpar(BF_C + 2, i)}, mass, Jw, cw);
    double* o = ic + 10 * i;
    o[0] = Jw[0]; o[1] = Jw[4]; o[2] = Jw[8]; o[3] = Jw[1]; o[4] = Jw[2]; o[5] = Jw[5];
    o[6] = cw.x; o[7] = cw.y; o[8] = cw.z; o[9] = mass;
  });
  wlanes([&](int f) {  // composite inertias, leaves to root
    if (f >= 10) return;
    for (int i = nb - 1; i > 0; --i) {
      const int pr = a.parent[i];
      if (pr >= 0) ic[10 * pr + f] += ic[10 * i + f];
    }
  });
  wlanes([&](int row) {
    if (row >= nv) return;
    for (int c = 0; c <= row; ++c) Mm[row * mp_ + c] = 0.0;
    int i = 0;  // the body that the row belongs to
    for (int b = 1; b < nb; ++b)
      if (a.voff[b] <= row && a.kind[b * Bp + lane] != K_FIXED) i = b;
    const int ki = a.kind[i * Bp + lane], ca = row - a.voff[i];
    const double* o = ic + 10 * i;
    const double Jxx = o[0], Jyy = o[1], Jzz = o[2], Jxy = o[3], Jxz = o[4], Jyz = o[5];
    const v3<double> c{o[6], o[7], o[8]};
    const double mass = o[9];
    v3<double> sw, sv, Fa, Fl;
    world_column(ki, X.ldm(PF_RW, i), X.ld3(PF_TW, i), ca, sw, sv);
    composite_force(Jxx, Jyy, Jzz, Jxy, Jxz, Jyz, c, mass, sw, sv, Fa, Fl);
    for (int j = i; j >= 0; j = a.parent[j]) {
      const int kj = a.kind[j * Bp + lane], nj = kj == K_FLOAT ? 6 : (kj == K_FIXED ? 0 : 1);
      const m3<double> Rj = X.ldm(PF_RW, j);
      const v3<double> oj = X.ld3(PF_TW, j);
      for (int cb2 = 0; cb2 < nj; ++cb2) {
        const int col = a.voff[j] + cb2;
        if (col > row) continue;
        v3<double> tw, tv;
        world_column(kj, Rj, oj, cb2, tw, tv);
        Mm[row * mp_ + col] = dot(Fa, tw) + dot(Fl, tv);
      }
    }
  });
  bool pd = true;
  for (int j = 0; j < nv; ++j) {
    wlanes([&](int r) {
      if (r < j || r >= nv) return;
      double t = Mm[r * mp_ + j];
      for (int k = 0; k < j; ++k) t -= Mm[r * mp_ + k] * Mm[j * mp_ + k];
      Mm[r * mp_ + j] = t;
    });
    double t = Mm[j * mp_ + j];
    if (!(t > 0.0)) {
      pd = false;
      t = 1.0;
    }
    const double ljj = sqrt(t);
    wlanes([&](int r) {
      if (r < j || r >= nv) return;
      if (r == j) Mm[r * mp_ + j] = ljj;
      else Mm[r * mp_ + j] = Mm[r * mp_ + j] / ljj;
    });
  }
  return pd;
}

// cone_program with its rows and contacts over the lanes
__device__ __forceinline__ bool vw_cone_program(const VsWave& W, int nc) {
  const int m = W.m;
  const VwLayout& L = W.L;
  double *g = W.lds + L.gv, *x = W.lds + L.x, *z = W.lds + L.z, *s = W.lds + L.s, *rd = W.lds + L.rd,
         *lt = W.lds + L.lt, *xb = W.lds + L.xb, *xi = W.lds + L.xi, *rhs = W.lds + L.rhs, *Wc = W.lds + L.w,
         *Wic = W.lds + L.wi;
  auto d = [](int k) { return k % 3 == 0 ? kConeMu : 1.0; };
  LaneD dx, dz, ds;  // by row
  LaneD fa, fb;      // two products' factors, step lengths by contact
  wlanes([&](int k) {
    if (k >= m) return;
    x[k] = k % 3 == 0 ? 1.0 / kConeMu : 0.0;
    z[k] = k % 3 == 0 ? 1.0 : 0.0;
    xb[k] = x[k];
  });
  double gnorm = 0.0;
  for (int k = 0; k < m; ++k) gnorm = fmax(gnorm, fabs(g[k]));
  double best = 1e300;
  int since_best = 0;
  // Newton direction for a right-hand side xi; dx by row, dz in lane registers
  auto solve = [&]() {
    wlanes([&](int c) {
      if (c >= nc) return;
      for (int i = 0; i < 3; ++i) {
        double t = 0.0;
        for (int j = 0; j < 3; ++j) t += Wic[9 * c + 3 * i + j] * xi[3 * c + j];
        rhs[3 * c + i] = -rd[3 * c + i] + d(i) * t;
      }
    });
    wlanes([&](int r) { dx[r] = r < m ? rhs[r] : 0.0; });
    for (int k = 0; k < m; ++k) {
      const double q = dx.at(k) / W.low(k, k);
      wlanes([&](int r) {
        if (r == k) dx[r] = q;
        else if (r > k && r < m) dx[r] -= W.low(r, k) * q;
      });
    }
    double last = 0.0;  // the entry solved before, still in a register
    for (int r = m - 1; r >= 0; --r) {
      double t = dx.at(r);
      if (r + 1 < m) t -= W.low(r + 1, r) * last;
#pragma unroll 4
      for (int k = r + 2; k < m; ++k) t -= W.low(k, r) * rhs[k];
      last = t / W.low(r, r);
      rhs[r] = last;  // every lane writes the same
    }
    wlanes([&](int r) { dx[r] = r < m ? rhs[r] : 0.0; });
    wlanes([&](int c) {
      if (c >= nc) return;
      double a3[3];
      for (int i = 0; i < 3; ++i) {
        a3[i] = 0.0;
        for (int j = 0; j < 3; ++j) a3[i] += Wic[9 * c + 3 * i + j] * d(j) * rhs[3 * c + j];
      }
      double o[3];
      for (int i = 0; i < 3; ++i) {
        double t = 0.0;
        for (int j = 0; j < 3; ++j) t += Wic[9 * c + 3 * i + j] * (xi[3 * c + j] - a3[j]);
        o[i] = t;
      }
      for (int i = 0; i < 3; ++i) xi[3 * c + i] = o[i];  // dz takes xi's place
    });
    wlanes([&](int r) {
      dz[r] = r < m ? xi[r] : 0.0;
      ds[r] = r < m ? d(r) * dx[r] : 0.0;
      if (r < m) rhs[r] = ds[r];  // ds takes dx's
    });
  };
  // after solve: rhs holds ds, xi holds dz
  auto max_step = [&](double scale) {
    wlanes([&](int c) {
      if (c >= nc) return;
      const double sc[3] = {s[3 * c], s[3 * c + 1], s[3 * c + 2]}, dsc[3] = {rhs[3 * c], rhs[3 * c + 1], rhs[3 * c + 2]};
      const double zc[3] = {z[3 * c], z[3 * c + 1], z[3 * c + 2]}, dzc[3] = {xi[3 * c], xi[3 * c + 1], xi[3 * c + 2]};
      fa[c] = scale * fmin(soc_max_step(sc, dsc), soc_max_step(zc, dzc));
    });
    double alpha = 1.0;
    for (int c = 0; c < nc; ++c) alpha = fmin(alpha, fa.at(c));
    return alpha;
  };
  for (int it = 0; it < kConeMaxIter; ++it) {
    wlanes([&](int k) {
      if (k < m) s[k] = d(k) * x[k];
    });
    wlanes([&](int r) {
      if (r >= m) return;
      double t = g[r] - d(r) * z[r];
#pragma unroll 4
      for (int k = 0; k < m; ++k) t += W.g(r, k) * x[k];
      rd[r] = t;
    });
    double gap = 0.0, rmax = 0.0, xmax = 0.0;
#pragma unroll 4
    for (int r = 0; r < m; ++r) {
      rmax = fmax(rmax, fabs(rd[r]));
      gap += s[r] * z[r];
      xmax = fmax(xmax, fabs(x[r]));
    }
    if (!isfinite(gap) || !isfinite(rmax)) break;
    const double gap_rel = gap / ((1.0 + gnorm) * (1.0 + xmax)), res_rel = rmax / (1.0 + gnorm);
    const double merit = fmax(gap_rel, res_rel);
    if (merit < best) {
      best = merit;
      since_best = 0;
      wlanes([&](int k) {
        if (k < m) xb[k] = x[k];
      });
    }
    if (gap_rel <= kConeGapTol && res_rel <= kConeResTol) break;
    if (++since_best > kConeStall) break;
    const double mug = gap / nc;
    // scaling, and K = G + D W^-2 D's lower triangle
    wlanes([&](int c) {
      if (c >= nc) return;
      const double sc[3] = {s[3 * c], s[3 * c + 1], s[3 * c + 2]}, zc[3] = {z[3 * c], z[3 * c + 1], z[3 * c + 2]};
      double Ws[9], Wi[9];
      nt_scaling(sc, zc, Ws, Wi);
      for (int k = 0; k < 9; ++k) { Wc[9 * c + k] = Ws[k]; Wic[9 * c + k] = Wi[k]; }
      for (int i = 0; i < 3; ++i) lt[3 * c + i] = Ws[3 * i] * zc[0] + Ws[3 * i + 1] * zc[1] + Ws[3 * i + 2] * zc[2];
    });
    wlanes([&](int r) {
      if (r >= m) return;
#pragma unroll 4
      for (int k = 0; k <= r; ++k) W.low(r, k) = W.up(k, r);
    });
    wlanes([&](int c) {
      if (c >= nc) return;
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) {
          double t = 0.0;
          for (int k = 0; k < 3; ++k) t += Wic[9 * c + 3 * i + k] * Wic[9 * c + 3 * k + j];
          W.low(3 * c + i, 3 * c + j) += d(i) * t * d(j);
        }
    });
    bool pd = true;
    for (int j = 0; j < m; ++j) {
      wlanes([&](int r) {
        if (r < j || r >= m) return;
        double x = W.low(r, j);
#pragma unroll 4
        for (int k = 0; k < j; ++k) x -= W.low(r, k) * W.low(j, k);
        W.low(r, j) = x;
      });
      const double t = W.low(j, j);
      if (!(t > 0.0)) { pd = false; break; }
      const double ljj = sqrt(t);
      wlanes([&](int r) {
        if (r < j || r >= m) return;
        if (r == j) W.low(r, j) = ljj;
        else W.low(r, j) = W.low(r, j) / ljj;
      });
    }
    if (!pd) break;
    // predictor
    wlanes([&](int k) {
      if (k < m) xi[k] = -lt[k];
    });
    solve();
    const double alpha_a = max_step(1.0);
    wlanes([&](int k) {
      fa[k] = k < m ? s[k] + alpha_a * ds[k] : 0.0;
      fb[k] = k < m ? z[k] + alpha_a * dz[k] : 0.0;
    });
    double sz = 0.0;
    for (int k = 0; k < m; ++k) sz += fa.at(k) * fb.at(k);
    const double ratio = sz / gap, sigma = ratio * ratio * ratio;
    const double smu = rounded(sigma * mug);
    // corrector: xi = lt \ (sigma mu e - lt o lt - (W^-1 ds) o (W dz))
    wlanes([&](int c) {
      if (c >= nc) return;
      double a3[3], b3[3];
      for (int i = 0; i < 3; ++i) {
        a3[i] = Wic[9 * c + 3 * i] * rhs[3 * c] + Wic[9 * c + 3 * i + 1] * rhs[3 * c + 1] + Wic[9 * c + 3 * i + 2] * rhs[3 * c + 2];
        b3[i] = Wc[9 * c + 3 * i] * xi[3 * c] + Wc[9 * c + 3 * i + 1] * xi[3 * c + 1] + Wc[9 * c + 3 * i + 2] * xi[3 * c + 2];
      }
      const double l0 = lt[3 * c], l1 = lt[3 * c + 1], l2 = lt[3 * c + 2];
      const double w0 = smu - (l0 * l0 + l1 * l1 + l2 * l2) - (a3[0] * b3[0] + a3[1] * b3[1] + a3[2] * b3[2]);
      const double w1 = -(2.0 * l0 * l1) - (a3[0] * b3[1] + b3[0] * a3[1]);
      const double w2 = -(2.0 * l0 * l2) - (a3[0] * b3[2] + b3[0] * a3[2]);
      const double y0 = (l0 * w0 - l1 * w1 - l2 * w2) / soc_det(l0, l1, l2);
      xi[3 * c] = y0;
      xi[3 * c + 1] = (w1 - y0 * l1) / l0;
      xi[3 * c + 2] = (w2 - y0 * l2) / l0;
    });
    solve();
    const double alpha = max_step(0.99);
    wlanes([&](int k) {
      if (k >= m) return;
      x[k] += alpha * dx[k];
      z[k] += alpha * dz[k];
    });
  }
  bool ok = best < 1e300;
  wlanes([&](int k) {
    if (k < m) x[k] = xb[k];
  });
  for (int k = 0; k < m; ++k) ok = ok && isfinite(x[k]);
  return ok;
}

// vs_dynamics on a wave
__device__ __forceinline__ bool vw_dynamics(VsWave& W, Strided q, Strided v, Strided tau, double h, int* n_contacts,
                                            int forced_body, int forced_h) {
  const VsLane& V = W.V;
  const BucketArgs& a = V.a;
  const int lane = V.lane, nv = a.nv, mp_ = nv | 1;
  Strided out = V.col(V.L.out), vn = V.col(V.L.vn);
  double *J = W.lds + W.L.j, *Y = W.lds + W.L.y, *gv = W.lds + W.L.gv, *vfree = W.lds + W.L.vfree, *x = W.lds + W.L.x,
         *Mm = W.lds + W.L.mm;
  bool ok = plain_dynamics_on(V.ctx(), q, v, tau, out, false);
  wlanes([&](int k) {
    if (k < nv) vfree[k] = v[k] + h * out[k];
  });
  world_frames(V);
  const int nc = find_contacts(V, forced_body, forced_h);
  *n_contacts = nc;
  if (nc == 0) {
    for (int k = 0; k < nv; ++k) vn[k] = vfree[k];
    return ok;
  }
  const int m = W.m = 3 * nc;
  wlanes([&](int r) {
    if (r >= m) return;
    for (int k = 0; k < nv; ++k) J[r * nv + k] = 0.0;
  });
  wlanes([&](int ci) {
    if (ci < nc) contact_jacobian(V, ci, [&](int r, int k, double e) { J[(3 * ci + r) * nv + k] = e; });
  });
  ok = vw_mass_matrix(W) && ok;
  wlanes([&](int r) {  // Y = M^-1 J^T, a row of J per lane
    if (r >= m) return;
    for (int k = 0; k < nv; ++k) {  // L y = J_r
      double t = J[r * nv + k];
      for (int l = 0; l < k; ++l) t -= Mm[k * mp_ + l] * Y[l * m + r];
      Y[k * m + r] = t / Mm[k * mp_ + k];
    }
    for (int k = nv - 1; k >= 0; --k) {  // L^T y = .
      double t = Y[k * m + r];
      for (int l = k + 1; l < nv; ++l) t -= Mm[l * mp_ + k] * Y[l * m + r];
      Y[k * m + r] = t / Mm[k * mp_ + k];
    }
  });
  for (int r0 = 0; r0 < m; r0 += 8)  // G = J Y by 8 x 8 tiles of its lower triangle
    for (int c0 = 0; c0 <= r0; c0 += 8)
      wlanes([&](int l) {
        const int r = r0 + (l >> 3), c = c0 + (l & 7);
        if (r >= m || c > r) return;
        double t = 0.0;
        for (int k = 0; k < nv; ++k) t += J[r * nv + k] * Y[k * m + c];
        W.up(c, r) = t;
      });
  wlanes([&](int r) {
    if (r >= m) return;
    double t = 0.0;
    for (int k = 0; k < nv; ++k) t += J[r * nv + k] * vfree[k];
    gv[r] = t;
  });
  ok = vw_cone_program(W, nc) && ok;
  wlanes([&](int k) {  // v_next = v_free + M^-1 J^T x
    if (k >= nv) return;
    double t = vfree[k];
    for (int r = 0; r < m; ++r) t += Y[k * m + r] * x[r];
    vfree[k] = t;
  });
  for (int k = 0; k < nv; ++k) vn[k] = vfree[k];
  return ok;
}

// n_steps steps of one instance: the collision loop around dyn, its contact
// dynamics. Every step reads q and v back from the state arrays it wrote.
template <class Dyn>
__device__ __forceinline__ void vs_run(const VsLane& V, double dt, int ccd, int n_steps, Dyn dyn) {
  const BucketArgs& a = V.a;
  const int lane = V.lane, Bp = a.Bp, nv = a.nv, nq = a.nq;
  Strided q{a.q + lane, Bp}, v{a.v + lane, Bp}, tau{const_cast<double*>(a.tau) + lane, Bp};
  Strided vdot{a.vdot + lane, Bp};
  for (int step = 0; step < n_steps; ++step) {
    Strided qc = V.col(V.L.qc), vc = V.col(V.L.vc), vn = V.col(V.L.vn);
    for (int k = 0; k < nq; ++k) qc[k] = q[k];
    for (int k = 0; k < nv; ++k) vc[k] = v[k];
    bool ok = true, done = false;
    double t_remain = dt;
    int forced_body = -1, forced_h = -1, rounds = 0;
    for (int round = 0; round < kCcdMaxRounds && !done; ++round) {
      int nc = 0, hit_body = -1, hit_h = -1;
      rounds = round + 1;
      ok = dyn(qc, vc, tau, t_remain, &nc, forced_body, forced_h) && ok;
      const double earliest = ccd ? earliest_collision(V, nc, &hit_body, &hit_h) : 1e300;
      if (earliest < t_remain) {
        plain_advance(a, lane, qc, vn, earliest, qc);
        for (int k = 0; k < nv; ++k) vc[k] = vn[k];
        t_remain -= earliest;
        forced_body = hit_body;
        forced_h = hit_body >= 0 ? hit_h : -1;
      } else {
        plain_advance(a, lane, qc, vn, t_remain, qc);
        done = true;
      }
    }
    ok = ok && done;  // the collision loop gave up: a fault, the state still advances
    if (!done) plain_advance(a, lane, qc, vn, t_remain, qc);
    for (int k = 0; k < nv; ++k) {
      vdot[k] = (vn[k] - v[k]) / dt;
      v[k] = vn[k];
    }
    for (int k = 0; k < nq; ++k) q[k] = qc[k];
    ok = ok && finite_cols(q, nq) && finite_cols(v, nv);
    if (!ok) a.fault[lane] = 1;
    a.rounds[lane] = rounds;
  }
}

}  // namespace

// n_steps steps of each lane in one launch: a lane goes on to its next step
// as soon as its own step is done, so a launch lasts as long as the slowest
// lane's sum of steps rather than the sum of each step's slowest lane. The
// lane's arithmetic is the same as in n_steps launches of one step.
__global__ void __launch_bounds__(64) vs_step_kernel(BucketArgs a, double dt, int ccd, int n_steps) {
  const int lane = blockIdx.x * blockDim.x + threadIdx.x;
  if (lane >= a.B) return;
  const VsLane V{a, lane, vs_layout(a.nb, a.nq, a.nv, a.nc, a.nh, a.ns), a.scratch + lane, a.Bp};
  vs_run(V, dt, ccd, n_steps, [&](Strided q, Strided v, Strided tau, double h, int* nc, int fb, int fh) {
    return vs_dynamics(V, q, v, tau, h, nc, fb, fh);
  });
}

// One instance per wave (workgroup)
__global__ void __launch_bounds__(64) vs_wave_kernel(BucketArgs a, double dt, int ccd, int n_steps) {
#ifndef __HIP_DEVICE_COMPILE__
  if (threadIdx.x != 0) return;  // the host build's first thread runs every lane
#endif
  double* const lds = (double*)GP_DYN_LDS;
  const VwLayout L = vw_layout(a.nb, a.nq, a.nv, (a.nc + a.ns) * a.nh);
  const VsLane V{a, (int)blockIdx.x, L.v, lds, 1};
  VsWave W{V, L, lds, 0};
  vs_run(V, dt, ccd, n_steps, [&](Strided q, Strided v, Strided tau, double h, int* nc, int fb, int fh) {
    return vw_dynamics(W, q, v, tau, h, nc, fb, fh);
  });
}

size_t vs_scratch_doubles(int nb, int nq, int nv, int nc, int nh, int ns, int Bp) {
  return vs_layout(nb, nq, nv, nc, nh, ns).total * (size_t)Bp;
}

// 64-lane workgroups: one instance per lane is a long serial program, so the
// launch spreads its waves over every compute unit rather than packing four
// to a workgroup on a quarter of them
int launch_vs_step(const BucketArgs& a, double dt, int ccd, int n_steps, void* stream) {
  if (a.B == 0 || n_steps <= 0) return 0;
  dim3 block(64), grid((a.B + 63) / 64);
  hipLaunchKernelGGL(vs_step_kernel, grid, block, 0, (hipStream_t)stream, a, dt, ccd, n_steps);
  return (int)hipGetLastError();
}

// The wave's lanes hold the program's rows, the bodies and the coordinates, and
// a workgroup's LDS its working set. The line lies where the instances no longer
// have a SIMD each: until then a launch takes one instance's time, which is the
// shorter one at any number of contacts; past it the wave kernel's time doubles
// and that of instances in flight is longer than the lane kernel's. Whether
// instances touch is not known when the launch is made, and none may be slower
// than on the lane kernel alone. Instances that do touch pay for it: they
// would be faster on the wave kernel up to several thousand (the crossing lies
// between 2,048 and 16,384 standing quadrupeds). Two steps, lane / wave, ms, at 64, 1,024 and 2,048 instances:
// quadrupeds on four feet 8.3 / 1.09, 8.8 / 1.25, 9.0 / 2.2 (and 11.8 / 14.8 at
// 16,384), in flight 0.200 / 0.131, 0.206 / 0.147, 0.207 / 0.297; 8-joint arms
// with one contact 1.04 / 0.38, 1.21 / 0.44, 1.22 / 0.83, with none 0.155 / 0.098,
// 0.159 / 0.108, 0.161 / 0.213; cubes on two planes (up to 16 contacts) 12.6 / 1.1,
// 14.6 / 1.6, 14.9 / 2.0.
bool vs_wave_ok(int B, int nb, int nq, int nv, int nc, int nh, int ns) {
  constexpr int kComputeUnits = 256, kSimds = 4, kLds = 160 << 10;  // LDS of a compute unit
  const int cmax = (nc + ns) * nh;
  if (cmax < 1 || 3 * cmax > 64 || nv < 1 || nv > 64 || nb > 64) return false;
  const int bytes = vw_layout(nb, nq, nv, cmax).total * 8;
  return bytes <= (64 << 10) && B <= kComputeUnits * std::min(kSimds, kLds / bytes);
}

int launch_vs_wave(const BucketArgs& a, double dt, int ccd, int n_steps, void* stream) {
  if (a.B == 0 || n_steps <= 0) return 0;
  const unsigned lds = (unsigned)(vw_layout(a.nb, a.nq, a.nv, (a.nc + a.ns) * a.nh).total * 8);
  hipLaunchKernelGGL(vs_wave_kernel, dim3(a.B), dim3(64), lds, (hipStream_t)stream, a, dt, ccd, n_steps);
  return (int)hipGetLastError();
}

}  // namespace gp
