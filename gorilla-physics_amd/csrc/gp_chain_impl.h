// gp_chain_impl.h — the FP64 dynamics of serial chains (TopoChain, TopoWelded)
// with one instance per lane.
//
// The host turns every body's frame of a chain about its own joint axis so
// that each tree rotation is Rx(alpha) Rz(delta) (gp_runtime.cpp,
// chain_frames). A joint's transform is then two planar rotations,
// Rx(alpha) Rz(delta + q), and a translation:
//  - a motion or force vector costs 16 operations a transform, and no 3x3
//    rotation is rebuilt in any of the three sweeps (from the tree parameters
//    that took 36 operations a body and sweep);
//  - the congruence of an articulated inertia turns 2x2 blocks, whose trace is
//    invariant, instead of three 3x3 products (79 operations against 144);
//  - a revolute joint's row and column of I^A - U U^T / D are zero: they are
//    neither formed nor turned.
// The base's acceleration is the only thing that the root's transform acts
// on, so it is one vector a launch (h = R_t^T a_base, turned by q).
//
// What bounds it: FP64 issue at one wave per SIMD (65,536 instances are 1,024
// waves, the chip's SIMDs), so operations are what is saved: the 7-joint
// kernel's code holds 2,252 FP64 instructions, 4,186 with rotations rebuilt as
// matrices. Measured with the state's transfers on one MI355X, before and
// after: 65,536 7-joint arms x 20 steps 222 -> 153 us, 65,536 SO-101 arms
// (RK4) x 10 steps 347 -> 241 us, 1,024 acrobots x 400 steps 461 -> 266 us,
// 32,768 chains of 1-12 joints and quadrupeds x 20 steps 1,078 -> 746 us. The
// error against 64-bit references is unchanged (arms: 1.7e-13 of the
// accelerations' norm after 20 steps, both).
// Included by gp_fast_impl.h (it uses Soa, sel and the topologies from there).
#pragma once

namespace gp {

template <class T> struct IsChain { static constexpr bool value = false; };
template <int N> struct IsChain<TopoChain<N>> { static constexpr bool value = true; };
template <int N> struct IsChain<TopoWelded<N>> { static constexpr bool value = true; };

// One joint's tree transform: Rx(alpha) as (ca, sa), the translation in the
// parent's frame, and (cd, sd) of the angle delta that q starts from.
struct ChainT {
  double ca, sa;
  v3<double> p;
  double cd, sd;
};
// A rigid body in its frame
struct ChainI {
  s3<double> J;
  v3<double> c;
  double m;
};

// Where a chain's parameters live for a launch. All in registers for short
// chains. Longer ones: a lane-private LDS row (one odd pitch per lane, so a
// wave's 64-bit accesses spread over the banks; a lane touches its own row
// only, so no barrier) with the transforms of joints 1.. (7 values each) and
// then the inertias (10 values) of as many bodies as fit in kLdsLaneBytes, the
// CU's 160 KB over its 256 lanes at one wave per SIMD; up to kChainRegBodies
// more inertias in registers, any further ones read from the bucket's array
// (L2) where used.
constexpr int kChainRegBodies = 4;
template <class Topo, bool ALLREV>
struct ChainTier {
  static constexpr int J = Topo::N - Topo::first;  // joints
  static constexpr bool REG = J <= (ALLREV ? 4 : 3);
  static constexpr int cap = kLdsLaneBytes / 8 - 1;
  static constexpr int NT = REG ? 0 : (J - 1 < cap / 7 ? J - 1 : cap / 7);  // transforms of joints 1 .. NT
  static constexpr int NI0 = NT == J - 1 ? (cap - 7 * NT) / 10 : 0;
  static constexpr int NI = REG ? 0 : (NI0 < J - 1 ? NI0 : J - 1);          // inertias of joints 1 .. NI
  static constexpr int left = J - 1 - NI;
  static constexpr int NR = REG ? J - 1 : (left <= kChainRegBodies ? left : 0);  // then NR in registers
  static constexpr int slots = 7 * NT + 10 * NI;
  static constexpr int pitch = slots > 0 ? (slots | 1) : 0;
};

template <class Topo, bool ALLREV>
struct ChainParams {
  using Tier = ChainTier<Topo, ALLREV>;
  static constexpr int J = Tier::J, N = Topo::N, F = Topo::first;
  static constexpr int RT = Tier::REG && J > 1 ? J - 1 : 1;
  static constexpr int RI = Tier::NR > 0 ? Tier::NR : 1;
  Soa<double> bp;
  int lane;
  double* lds;
  unsigned rev;         // bit j: joint j is revolute
  v3<double> h;         // base acceleration in the root's tree frame
  double jzz, cx, cy, m0;  // what the root's body contributes
  ChainT rt[RT];        // joint 1 + k in rt[k] (register tier)
  ChainI ri[RI];        // joint 1 + NI + k in ri[k]

  __device__ __forceinline__ double ld(int f, int j) const { return bp.ld(f * N + F + j, lane); }
  __device__ __forceinline__ ChainT load_t(int j) const {
    // R_t = Rx(alpha) Rz(delta): row 0 is (cd, -sd, 0), column 2 is (0, -sa, ca)
    return ChainT{ld(BF_RT + 8, j), -ld(BF_RT + 5, j), v3<double>{ld(BF_PT, j), ld(BF_PT + 1, j), ld(BF_PT + 2, j)},
                  ld(BF_RT, j), -ld(BF_RT + 1, j)};
  }
  __device__ __forceinline__ ChainI load_i(int j) const {
    return ChainI{s3<double>{ld(BF_J, j), ld(BF_J + 1, j), ld(BF_J + 2, j), ld(BF_J + 3, j), ld(BF_J + 4, j),
                             ld(BF_J + 5, j)},
                  v3<double>{ld(BF_C, j), ld(BF_C + 1, j), ld(BF_C + 2, j)}, ld(BF_M, j)};
  }
  __device__ __forceinline__ ChainParams(const BucketArgs& a, int lane_, double* lds_base)
      : bp(a.bp, NBF * N, a.Bp), lane(lane_), lds(lds_base + (int)threadIdx.x * Tier::pitch) {
    if constexpr (ALLREV) {
      rev = ~0u;
    } else {
      const Soa<int> kindS(a.kind, a.nb, a.Bp);
      rev = 0;
#pragma unroll
      for (int j = 0; j < J; ++j) rev |= (kindS.ld(F + j, lane) == K_REV ? 1u : 0u) << j;
    }
    // the root: gravity as the base's acceleration, seen through the welded
    // body's rotation (if any) and the root's
    v3<double> g{0.0, 0.0, a.g};
    if constexpr (F > 0) {
      g = v3<double>{a.g * bp.ld((BF_RT + 6) * N, lane), a.g * bp.ld((BF_RT + 7) * N, lane),
                     a.g * bp.ld((BF_RT + 8) * N, lane)};
      m3<double> R;
#pragma unroll
      for (int k = 0; k < 9; ++k) R.a[k] = ld(BF_RT + k, 0);
      h = mulT(R, g);
    } else {
      h = v3<double>{a.g * ld(BF_RT + 6, 0), a.g * ld(BF_RT + 7, 0), a.g * ld(BF_RT + 8, 0)};
    }
    jzz = ld(BF_J + 2, 0);
    cx = ld(BF_C, 0);
    cy = ld(BF_C + 1, 0);
    m0 = ALLREV ? 0.0 : ld(BF_M, 0);
    if constexpr (Tier::REG) {
#pragma unroll
      for (int j = 1; j < J; ++j) rt[j - 1] = load_t(j);
    } else {
#pragma unroll
      for (int j = 1; j <= Tier::NT; ++j) {
        const ChainT t = load_t(j);
        double* o = lds + 7 * (j - 1);
        o[0] = t.ca; o[1] = t.sa; o[2] = t.p.x; o[3] = t.p.y; o[4] = t.p.z; o[5] = t.cd; o[6] = t.sd;
      }
#pragma unroll
      for (int j = 1; j <= Tier::NI; ++j)
#pragma unroll
        for (int k = 0; k < 10; ++k) lds[7 * Tier::NT + 10 * (j - 1) + k] = ld(BF_J + k, j);
    }
#pragma unroll
    for (int k = 0; k < Tier::NR; ++k) ri[k] = load_i(1 + Tier::NI + k);
  }
  // a compiler-only memory barrier: LDS values read after it are loaded again,
  // not held in registers from one sweep to the next
  __device__ __forceinline__ void sweep_fence() const {
    if constexpr (!Tier::REG) asm volatile("" ::: "memory");
  }
  __device__ __forceinline__ ChainT t(int j) const {
    if constexpr (Tier::REG) return rt[j - 1];
    if (j <= Tier::NT) {
      const double* o = lds + 7 * (j - 1);
      return ChainT{o[0], o[1], v3<double>{o[2], o[3], o[4]}, o[5], o[6]};
    }
    return load_t(j);
  }
  __device__ __forceinline__ ChainI inertia(int j) const {
    if (j <= Tier::NI) {
      const double* o = lds + 7 * Tier::NT + 10 * (j - 1);
      return ChainI{s3<double>{o[0], o[1], o[2], o[3], o[4], o[5]}, v3<double>{o[6], o[7], o[8]}, o[9]};
    }
    if (j <= Tier::NI + Tier::NR) return ri[j - 1 - Tier::NI];
    return load_i(j);
  }
  __device__ __forceinline__ bool revolute(int j) const { return ALLREV || ((rev >> j) & 1u); }
};

// What a joint keeps between the sweeps
struct ChainJoint {
  double c, s;                // of delta + q (prismatic: of delta)
  double cw0, cw1, cv0, cv1;  // velocity-product acceleration (its z components are 0)
  sv<double> pA;              // articulated bias force
  sv<double> U;               // I^A S
  double Dinv, u;             // 1 / (S^T I^A S), tau - S^T p^A
};

// Rx(alpha) x and Rx(alpha)^T x, Rz x and Rz^T x
__device__ __forceinline__ v3<double> rx(double c, double s, v3<double> x) {
  return {x.x, c * x.y - s * x.z, s * x.y + c * x.z};
}
__device__ __forceinline__ v3<double> rxT(double c, double s, v3<double> x) {
  return {x.x, c * x.y + s * x.z, c * x.z - s * x.y};
}
__device__ __forceinline__ v3<double> rz(double c, double s, v3<double> x) {
  return {c * x.x - s * x.y, s * x.x + c * x.y, x.z};
}
__device__ __forceinline__ v3<double> rzT(double c, double s, v3<double> x) {
  return {c * x.x + s * x.y, c * x.y - s * x.x, x.z};
}
// a symmetric 2x2 block turned by (c, s); its trace is invariant
__device__ __forceinline__ void turn2(double c, double s, double& xx, double& yy, double& xy) {
  const double p = c * xx - s * xy, q = c * xy - s * yy, tr = xx + yy;
  xx = c * p - s * q;
  xy = s * p + c * q;
  yy = tr - xx;
}

// 1 / x to the last bit or so: the hardware's estimate and two Newton steps.
// Zero, infinite and NaN x give NaN, which the callers' tests count as failed.
__device__ __forceinline__ double recip(double x) {
#ifdef __HIP_DEVICE_COMPILE__
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
#else
  return 1.0 / x;
#endif
}

// X^T I X of an articulated inertia whose joint is (c, s) about z, then alpha
// about x, then the translation r. ZROW: the angular z row and column of I are
// zero (a revolute joint's, after its rank-1 step).
template <bool ZROW>
__device__ __forceinline__ ai6<double> chain_xtix(const ChainT& t, double c, double s, v3<double> r, ai6<double> I) {
  // about z
  turn2(c, s, I.A.xx, I.A.yy, I.A.xy);
  turn2(c, s, I.C.xx, I.C.yy, I.C.xy);
  {
    const double x = I.C.xz, y = I.C.yz;
    I.C.xz = c * x - s * y;
    I.C.yz = s * x + c * y;
  }
  if constexpr (!ZROW) {
    const double x = I.A.xz, y = I.A.yz;
    I.A.xz = c * x - s * y;
    I.A.yz = s * x + c * y;
  }
  double* B = I.B.a;
  {
    const double t00 = c * B[0] - s * B[1], t01 = s * B[0] + c * B[1];
    const double t10 = c * B[3] - s * B[4], t11 = s * B[3] + c * B[4];
    const double z0 = B[2], z1 = B[5];
    B[0] = c * t00 - s * t10; B[3] = s * t00 + c * t10;
    B[1] = c * t01 - s * t11; B[4] = s * t01 + c * t11;
    B[2] = c * z0 - s * z1;   B[5] = s * z0 + c * z1;
    if constexpr (!ZROW) {
      const double x = B[6], y = B[7];
      B[6] = c * x - s * y;
      B[7] = s * x + c * y;
    }
  }
  // about x
  const double ca = t.ca, sa = t.sa;
  turn2(ca, sa, I.C.yy, I.C.zz, I.C.yz);
  {
    const double x = I.C.xy, y = I.C.xz;
    I.C.xy = ca * x - sa * y;
    I.C.xz = sa * x + ca * y;
  }
  if constexpr (ZROW) {
    const double cy = ca * I.A.yy, sy = sa * I.A.yy;
    I.A.xz = sa * I.A.xy;
    I.A.xy = ca * I.A.xy;
    I.A.yy = ca * cy;
    I.A.yz = sa * cy;
    I.A.zz = sa * sy;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const double y = B[3 * k + 1], z = B[3 * k + 2];
      B[3 * k + 1] = ca * y - sa * z;
      B[3 * k + 2] = sa * y + ca * z;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      B[6 + k] = sa * B[3 + k];
      B[3 + k] = ca * B[3 + k];
    }
  } else {
    turn2(ca, sa, I.A.yy, I.A.zz, I.A.yz);
    {
      const double x = I.A.xy, y = I.A.xz;
      I.A.xy = ca * x - sa * y;
      I.A.xz = sa * x + ca * y;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double y = B[3 * k + 1], z = B[3 * k + 2];
      B[3 * k + 1] = ca * y - sa * z;
      B[3 * k + 2] = sa * y + ca * z;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double y = B[3 + k], z = B[6 + k];
      B[3 + k] = ca * y - sa * z;
      B[6 + k] = sa * y + ca * z;
    }
  }
  // translation: B_p = B + r x C, A_p = A + r x B^T - B_p (r x)
  const s3<double> C = I.C;
  const v3<double> c0 = cross(r, v3<double>{C.xx, C.xy, C.xz});
  const v3<double> c1 = cross(r, v3<double>{C.xy, C.yy, C.yz});
  const v3<double> c2 = cross(r, v3<double>{C.xz, C.yz, C.zz});
  ai6<double> o;
  o.C = C;
  o.B = m3<double>{{B[0] + c0.x, B[1] + c1.x, B[2] + c2.x, B[3] + c0.y, B[4] + c1.y, B[5] + c2.y, B[6] + c0.z,
                    B[7] + c1.z, B[8] + c2.z}};
  const double* P = o.B.a;
  // (r x B^T)_ij = (r x row j of B)_i, (B_p r x)_ij = (row i of B_p x r)_j
  o.A.xx = I.A.xx + (r.y * B[2] - r.z * B[1]) - (P[1] * r.z - P[2] * r.y);
  o.A.yy = I.A.yy + (r.z * B[3] - r.x * B[5]) - (P[5] * r.x - P[3] * r.z);
  o.A.zz = I.A.zz + (r.x * B[7] - r.y * B[6]) - (P[6] * r.y - P[7] * r.x);
  o.A.xy = I.A.xy + (r.y * B[5] - r.z * B[4]) - (P[2] * r.x - P[0] * r.z);
  o.A.xz = I.A.xz + (r.y * B[8] - r.z * B[7]) - (P[0] * r.y - P[1] * r.x);
  o.A.yz = I.A.yz + (r.z * B[6] - r.x * B[8]) - (P[3] * r.y - P[4] * r.x);
  return o;
}

// Joint accelerations of one instance at (q, v). tau(k), and out(j, qdd) takes
// joint j's acceleration as soon as the outward sweep knows it (nothing later
// in the sweep reads q or v). False where a D is not positive.
template <class Topo, bool ALLREV, class Tau, class Out>
__device__ __forceinline__ bool chain_dynamics(const ChainParams<Topo, ALLREV>& P, const double* q, const double* v,
                                               Tau tau, Out out) {
  constexpr int J = ChainTier<Topo, ALLREV>::J;
  ChainJoint b[J];
  bool ok = true;
  auto shift = [&](const ChainT& t, int j) {  // the joint's translation in the parent's frame
    if constexpr (ALLREV) return t.p;
    const double d = P.revolute(j) ? 0.0 : q[j];
    return v3<double>{t.p.x, t.p.y - t.sa * d, t.p.z + t.ca * d};
  };
  P.sweep_fence();
  // ---- pass 1: velocities, velocity-product accelerations, rigid bias forces
  sv<double> V{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
#pragma unroll
  for (int j = 0; j < J; ++j) {
    ChainJoint& B = b[j];
    const bool rev = P.revolute(j);
    const double qd = v[j];
    double s0, c0;
    sincos_q(rev ? q[j] : 0.0, &s0, &c0);
    if (j == 0) {
      // only qd along z: no velocity product, no bias force along z
      B.c = c0;
      B.s = s0;
      V.w.z = rev ? qd : 0.0;
      V.v.z = rev ? 0.0 : qd;
      continue;
    }
    const ChainT t = P.t(j);
    B.c = t.cd * c0 - t.sd * s0;
    B.s = t.sd * c0 + t.cd * s0;
    const v3<double> r = shift(t, j);
    v3<double> w, l;
    if (j == 1) {  // the root's velocity lies along z
      w = v3<double>{0.0, t.sa * V.w.z, t.ca * V.w.z};
      l = v3<double>{-(r.y * V.w.z), r.x * V.w.z, V.v.z};
      if constexpr (ALLREV) l = v3<double>{l.x, t.ca * l.y, -(t.sa * l.y)};
      else l = rxT(t.ca, t.sa, l);
      w = v3<double>{B.s * w.y, B.c * w.y, w.z};
    } else {
      w = rzT(B.c, B.s, rxT(t.ca, t.sa, V.w));
      l = rxT(t.ca, t.sa, V.v - cross(r, V.w));
    }
    l = rzT(B.c, B.s, l);
    V = sv<double>{w, l};
    if constexpr (ALLREV) {
      V.w.z += qd;
      B.cw0 = qd * w.y;
      B.cw1 = -(qd * w.x);
      B.cv0 = qd * l.y;
      B.cv1 = -(qd * l.x);
    } else {
      V.w.z += rev ? qd : 0.0;
      V.v.z += rev ? 0.0 : qd;
      B.cw0 = rev ? qd * w.y : 0.0;
      B.cw1 = rev ? -(qd * w.x) : 0.0;
      B.cv0 = qd * sel(rev, l.y, w.y);
      B.cv1 = -(qd * sel(rev, l.x, w.x));
    }
    // v x* (I v): w x (J w) + c x g and m g + w x (w x c) with g = w x v
    const ChainI I = P.inertia(j);
    const v3<double> g = cross(V.w, V.v), wc = cross(V.w, I.c);
    const v3<double> hw = mul(I.J, V.w);
    B.pA.w = cross(V.w, hw) + cross(I.c, g);
    B.pA.v = I.m * g + cross(V.w, wc);
  }
  P.sweep_fence();
  // ---- pass 2: articulated inertias and bias forces, tip to root
  ai6<double> acc;      // the outer bodies' part of body j's inertia
  sv<double> facc;
#pragma unroll
  for (int j = J - 1; j >= 1; --j) {
    ChainJoint& B = b[j];
    const bool rev = P.revolute(j);
    ai6<double> IA;
    {
      const ChainI I = P.inertia(j);
      if (j == J - 1) {
        IA = rigid(I.J, I.c, I.m);
      } else {
        IA = acc;
        IA.A.xx += I.J.xx; IA.A.yy += I.J.yy; IA.A.zz += I.J.zz;
        IA.A.xy += I.J.xy; IA.A.xz += I.J.xz; IA.A.yz += I.J.yz;
        IA.B.a[1] -= I.c.z; IA.B.a[2] += I.c.y; IA.B.a[3] += I.c.z;
        IA.B.a[5] -= I.c.x; IA.B.a[6] -= I.c.y; IA.B.a[7] += I.c.x;
        IA.C.xx += I.m; IA.C.yy += I.m; IA.C.zz += I.m;
        B.pA = B.pA + facc;
      }
    }
    const double D = ALLREV ? IA.A.zz : sel(rev, IA.A.zz, IA.C.zz);
    B.U = ALLREV || rev ? col(IA, 2) : col(IA, 5);
    B.Dinv = recip(D);
    ok = ok && (B.Dinv > 0.0);
    double tq = tau(j);
    if constexpr (!ALLREV) {
      const double sk = rev ? 0.0 : P.ld(BF_SK, j);
      tq += -sk * (q[j] - P.ld(BF_SL, j));
    }
    B.u = tq - (ALLREV ? B.pA.w.z : sel(rev, B.pA.w.z, B.pA.v.z));
    const sv<double> uD{B.Dinv * B.U.w, B.Dinv * B.U.v};
    sv<double> pa;
    if constexpr (ALLREV) {
      // the angular z row and column of I^A - U U^T / D are zero, and the bias
      // force along z is the whole torque
      IA.A.xx -= uD.w.x * B.U.w.x;
      IA.A.xy -= uD.w.x * B.U.w.y;
      IA.A.yy -= uD.w.y * B.U.w.y;
      const double uv[3] = {B.U.v.x, B.U.v.y, B.U.v.z};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        IA.B.a[k] -= uD.w.x * uv[k];
        IA.B.a[3 + k] -= uD.w.y * uv[k];
      }
      IA.C.xx -= uD.v.x * B.U.v.x; IA.C.yy -= uD.v.y * B.U.v.y; IA.C.zz -= uD.v.z * B.U.v.z;
      IA.C.xy -= uD.v.x * B.U.v.y; IA.C.xz -= uD.v.x * B.U.v.z; IA.C.yz -= uD.v.y * B.U.v.z;
      const double* M = IA.B.a;
      pa.w.x = B.pA.w.x + IA.A.xx * B.cw0 + IA.A.xy * B.cw1 + M[0] * B.cv0 + M[1] * B.cv1 + B.u * uD.w.x;
      pa.w.y = B.pA.w.y + IA.A.xy * B.cw0 + IA.A.yy * B.cw1 + M[3] * B.cv0 + M[4] * B.cv1 + B.u * uD.w.y;
      pa.w.z = tq;
      pa.v.x = B.pA.v.x + M[0] * B.cw0 + M[3] * B.cw1 + IA.C.xx * B.cv0 + IA.C.xy * B.cv1 + B.u * uD.v.x;
      pa.v.y = B.pA.v.y + M[1] * B.cw0 + M[4] * B.cw1 + IA.C.xy * B.cv0 + IA.C.yy * B.cv1 + B.u * uD.v.y;
      pa.v.z = B.pA.v.z + M[2] * B.cw0 + M[5] * B.cw1 + IA.C.xz * B.cv0 + IA.C.yz * B.cv1 + B.u * uD.v.z;
    } else {
      IA = rank1_down(IA, B.U, uD);
      const double* M = IA.B.a;
      pa.w.x = B.pA.w.x + IA.A.xx * B.cw0 + IA.A.xy * B.cw1 + M[0] * B.cv0 + M[1] * B.cv1 + B.u * uD.w.x;
      pa.w.y = B.pA.w.y + IA.A.xy * B.cw0 + IA.A.yy * B.cw1 + M[3] * B.cv0 + M[4] * B.cv1 + B.u * uD.w.y;
      pa.w.z = B.pA.w.z + IA.A.xz * B.cw0 + IA.A.yz * B.cw1 + M[6] * B.cv0 + M[7] * B.cv1 + B.u * uD.w.z;
      pa.v.x = B.pA.v.x + M[0] * B.cw0 + M[3] * B.cw1 + IA.C.xx * B.cv0 + IA.C.xy * B.cv1 + B.u * uD.v.x;
      pa.v.y = B.pA.v.y + M[1] * B.cw0 + M[4] * B.cw1 + IA.C.xy * B.cv0 + IA.C.yy * B.cv1 + B.u * uD.v.y;
      pa.v.z = B.pA.v.z + M[2] * B.cw0 + M[5] * B.cw1 + IA.C.xz * B.cv0 + IA.C.yz * B.cv1 + B.u * uD.v.z;
    }
    const ChainT t = P.t(j);
    const v3<double> r = shift(t, j);
    acc = chain_xtix<ALLREV>(t, B.c, B.s, r, IA);
    const v3<double> fl = rx(t.ca, t.sa, rz(B.c, B.s, pa.v));
    facc = sv<double>{rx(t.ca, t.sa, rz(B.c, B.s, pa.w)) + cross(r, fl), fl};
  }
  // ---- the root, then pass 3: accelerations, root to tip
  P.sweep_fence();
  sv<double> A;
  {
    ChainJoint& B = b[0];
    const bool rev = P.revolute(0);
    // the base has no angular acceleration: only U's linear part is needed
    double D, pz;
    v3<double> Ul;
    if constexpr (J > 1) {
      D = ALLREV ? P.jzz + acc.A.zz : sel(rev, P.jzz + acc.A.zz, P.m0 + acc.C.zz);
      const v3<double> Ur{acc.B.a[6] - P.cy, acc.B.a[7] + P.cx, acc.B.a[8]};
      Ul = ALLREV ? Ur : v3<double>{sel(rev, Ur.x, acc.C.xz), sel(rev, Ur.y, acc.C.yz), sel(rev, Ur.z, D)};
      pz = ALLREV ? facc.w.z : sel(rev, facc.w.z, facc.v.z);
    } else {
      D = ALLREV ? P.jzz : sel(rev, P.jzz, P.m0);
      Ul = v3<double>{rev ? -P.cy : 0.0, rev ? P.cx : 0.0, rev ? 0.0 : D};
      pz = 0.0;
    }
    double tq = tau(0);
    if constexpr (!ALLREV) {
      const double sk = rev ? 0.0 : P.ld(BF_SK, 0);
      tq += -sk * (q[0] - P.ld(BF_SL, 0));
    }
    B.Dinv = recip(D);
    ok = ok && (B.Dinv > 0.0);
    A.v = rzT(B.c, B.s, P.h);
    const double qdd = ((tq - pz) - dot(Ul, A.v)) * B.Dinv;
    out(0, qdd);
    A.w = v3<double>{0.0, 0.0, rev ? qdd : 0.0};
    if constexpr (!ALLREV) A.v.z += rev ? 0.0 : qdd;
  }
#pragma unroll
  for (int j = 1; j < J; ++j) {
    const ChainJoint& B = b[j];
    const bool rev = P.revolute(j);
    const ChainT t = P.t(j);
    const v3<double> r = shift(t, j);
    v3<double> w, l;
    if (j == 1) {  // the root's angular acceleration lies along z
      const double wz = A.w.z;
      w = v3<double>{0.0, t.sa * wz, t.ca * wz};
      w = v3<double>{B.s * w.y, B.c * w.y, w.z};
      l = v3<double>{A.v.x - r.y * wz, A.v.y + r.x * wz, A.v.z};
    } else {
      w = rzT(B.c, B.s, rxT(t.ca, t.sa, A.w));
      l = A.v - cross(r, A.w);
    }
    l = rzT(B.c, B.s, rxT(t.ca, t.sa, l));
    w.x += B.cw0; w.y += B.cw1; l.x += B.cv0; l.y += B.cv1;
    A = sv<double>{w, l};
    const double qdd = (B.u - dot6(B.U, A)) * B.Dinv;
    out(j, qdd);
    if constexpr (ALLREV) {
      A.w.z += qdd;
    } else {
      A.w.z += rev ? qdd : 0.0;
      A.v.z += rev ? 0.0 : qdd;
    }
  }
  return ok;
}

}  // namespace gp
