// gp_tree_impl.h — trees of bodies, one body and its joint per lane: an
// instance takes as many neighbouring lanes of one wave as it has bodies, and
// a wave holds as many whole instances as fit in its 64 lanes (three hexapods
// of 19 bodies, seven quadrupeds of 9). The articulated-body algorithm (RBDA
// Table 7.1) runs its three sweeps level by level: every body of one depth at
// once, each reading its parent's velocity, world pose or acceleration on the
// way out and its children's articulated inertias and bias forces on the way
// in. The lanes exchange through LDS: each lane has a slot of kTreeSlot
// doubles, written by the lane when its level is done and read by its children
// (pass 1 and 3) or its parent (pass 2) one level later; all lanes of an
// instance are in one wave, whose LDS instructions execute in order, so no
// barrier is needed, only a compiler fence between levels. Runtime topology:
// any tree of up to 64 bodies with at most kTreeMaxChildren children per
// body, every joint type, contact points, prismatic springs; semi-implicit
// Euler (integrators.rs:276-319), n_steps steps per launch. The joint
// accelerations are those of the reference's dynamics_continuous
// (dynamics.rs:322-364). R = double: FP64 throughout; R = float: FP32 sweeps,
// FP64 joint-space solves, contact distances and q/v (as the other mixed
// kernels).
//
// What bounds it: each level's instructions issue for the whole wave with the
// other depths' lanes masked off, and each level waits for the one before
// through LDS. So: instances packed by their body count, not by a power of two
// above it, and two waves per SIMD, which 256 registers a lane allow once a
// floating joint's coordinates (one lane in a tree has them) live in LDS
// instead of every lane's registers. Measured with the state's transfers on
// one MI355X, ten steps: 8,191 trees of 16-40 bodies 1,060 -> 534 us (one wave
// per SIMD, two instances a wave before); 2,048 nine-body quadrupeds with
// twelve foot contacts 986 (plain kernel) -> 122 us.
// Included by gp_fast_impl.h (it uses Soa, pick and joint_frame from there).
#pragma once

namespace gp {

constexpr int kTreeMaxChildren = 8;
// doubles per lane in the exchange slot (an articulated inertia and a force,
// 21 + 6; odd, so a wave's 64-bit accesses spread over the banks)
constexpr int kTreeSlot = 27;

// slot <-> spatial vector / articulated inertia, in the sweeps' precision R
// from the slot's start (the slot is a row of doubles)
template <class R> __device__ __forceinline__ void put_sv(R* p, const sv<R>& x) {
  p[0] = x.w.x; p[1] = x.w.y; p[2] = x.w.z; p[3] = x.v.x; p[4] = x.v.y; p[5] = x.v.z;
}
template <class R> __device__ __forceinline__ sv<R> get_sv(const R* p) {
  return {{p[0], p[1], p[2]}, {p[3], p[4], p[5]}};
}
template <class R> __device__ __forceinline__ void put_ai6(R* p, const ai6<R>& I) {
  p[0] = I.A.xx; p[1] = I.A.yy; p[2] = I.A.zz; p[3] = I.A.xy; p[4] = I.A.xz; p[5] = I.A.yz;
#pragma unroll
  for (int k = 0; k < 9; ++k) p[6 + k] = I.B.a[k];
  p[15] = I.C.xx; p[16] = I.C.yy; p[17] = I.C.zz; p[18] = I.C.xy; p[19] = I.C.xz; p[20] = I.C.yz;
}
template <class R> __device__ __forceinline__ ai6<R> get_ai6(const R* p) {
  ai6<R> o;
  o.A = s3<R>{p[0], p[1], p[2], p[3], p[4], p[5]};
#pragma unroll
  for (int k = 0; k < 9; ++k) o.B.a[k] = p[6 + k];
  o.C = s3<R>{p[15], p[16], p[17], p[18], p[19], p[20]};
  return o;
}
// a compiler-only barrier between levels: slot reads are not moved above the
// writes of the level before (the hardware keeps one wave's LDS order)
__device__ __forceinline__ void level_fence() { asm volatile("" ::: "memory"); }

// doubles of a floating joint's coordinates in LDS: q, v, torques, accelerations
constexpr int kTreeFloat = 7 + 6 + 6 + 6;
// most LDS a lane can account for (a floating body alone)
constexpr int kTreeLaneBytes = (kTreeSlot + kTreeFloat) * 8;
// LDS doubles of an instance: its bodies' slots, then its floating joints
inline __host__ __device__ int tree_seg_doubles(int nb, int floating) { return kTreeSlot * nb + kTreeFloat * floating; }
// LDS bytes of one wave
inline int tree_wave_bytes(int nb, int floating) { return 64 / nb * tree_seg_doubles(nb, floating) * 8; }

// Whether a topology runs on this kernel: at most 64 bodies, none with more
// than kTreeMaxChildren children.
inline bool tree_topology_ok(int nb, const int* parent) {
  if (nb < 1 || nb > 64) return false;
  for (int i = 0; i < nb; ++i) {
    int c = 0;
    for (int k = i + 1; k < nb; ++k) c += parent[k] == i ? 1 : 0;
    if (c > kTreeMaxChildren) return false;
  }
  return true;
}

// L D L^T of a floating joint's 6x6 inertia, packed by rows: unit lower factor
// below the diagonal, reciprocal pivots on it; false if a pivot is not positive.
__device__ __forceinline__ bool ldl6(const ai6<double>& I, double (&L)[21]) {
  L[0] = I.A.xx;
  L[1] = I.A.xy; L[2] = I.A.yy;
  L[3] = I.A.xz; L[4] = I.A.yz; L[5] = I.A.zz;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) L[(3 + r) * (4 + r) / 2 + c] = I.B.a[3 * c + r];
  L[9] = I.C.xx;
  L[13] = I.C.xy; L[14] = I.C.yy;
  L[18] = I.C.xz; L[19] = I.C.yz; L[20] = I.C.zz;
  bool ok = true;
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    // column j below the pivot still holds L_ij d_j of the columns before
    const int jj = j * (j + 1) / 2;
    ok = ok && (L[jj + j] > 0.0);
    const double inv = recip(L[jj + j]);
#pragma unroll
    for (int i = j + 1; i < 6; ++i) {
      const int ii = i * (i + 1) / 2;
      const double lij = L[ii + j] * inv;
#pragma unroll
      for (int k = j + 1; k <= i; ++k) L[ii + k] -= lij * L[k * (k + 1) / 2 + j];
    }
#pragma unroll
    for (int i = j + 1; i < 6; ++i) L[i * (i + 1) / 2 + j] *= inv;
    L[jj + j] = inv;
  }
  return ok;
}
__device__ __forceinline__ void ldl6_solve(const double (&L)[21], double (&x)[6]) {
#pragma unroll
  for (int i = 1; i < 6; ++i)
#pragma unroll
    for (int k = 0; k < i; ++k) x[i] -= L[i * (i + 1) / 2 + k] * x[k];
#pragma unroll
  for (int i = 0; i < 6; ++i) x[i] *= L[i * (i + 1) / 2 + i];
#pragma unroll
  for (int i = 4; i >= 0; --i)
#pragma unroll
    for (int k = i + 1; k < 6; ++k) x[i] -= L[k * (k + 1) / 2 + i] * x[k];
}

// Contact wrench on a body (contact.rs:97-129) in its frame: points [c0, c1)
// of the bucket against every half-space, the body's world pose (Rw, tw).
template <class R>
__device__ __forceinline__ sv<R> tree_contacts(const BucketArgs& a, int inst, int c0, int c1, const m3<double>& Rw,
                                               const v3<double>& tw, const sv<R>& vel) {
  const Soa<double> cpS(a.cp, NCF * a.nc, a.Bp), hpS(a.hp, NHF * a.nh, a.Bp);
  const m3<R> RwR = cvt<R>(Rw);
  sv<R> fe{{R(0), R(0), R(0)}, {R(0), R(0), R(0)}};
  for (int h = 0; h < a.nh; ++h) {
    auto hpar = [&](int fld) { return hpS.ld(fld * a.nh + h, inst); };
    const v3<double> n{hpar(HF_NORMAL), hpar(HF_NORMAL + 1), hpar(HF_NORMAL + 2)};
    const v3<double> nb_ = mulT(Rw, n);
    const double off = dot(tw - v3<double>{hpar(HF_POINT), hpar(HF_POINT + 1), hpar(HF_POINT + 2)}, n);
    const R alpha = R(hpar(HF_ALPHA)), mu = R(hpar(HF_MU));
    for (int cc = c0; cc < c1; ++cc) {
      auto cpar = [&](int fld) { return cpS.ldx(fld * a.nc, inst, cc); };
      const v3<double> pb{cpar(CF_P), cpar(CF_P + 1), cpar(CF_P + 2)};
      const double dist = dot(nb_, pb) + off;
      if (dist <= kInsideMargin) {
        const v3<R> pbR = cvt<R>(pb);
        const v3<R> vw = mul(RwR, vel.v + cross(vel.w, pbR));
        const v3<R> F = contact_force(R(-dist), cvt<R>(n), vw, R(cpar(CF_K)), R(kHalfspaceK), alpha, mu);
        const v3<R> Fb = mulT(RwR, F);
        fe.w = fe.w + cross(pbR, Fb);
        fe.v = fe.v + Fb;
      }
    }
  }
  return fe;
}

// The children's lanes of body j, a byte each
__device__ __forceinline__ unsigned long long tree_children(const BucketArgs& a, int ch0, int nch) {
  unsigned long long c = 0;
  for (int k = 0; k < nch; ++k) c |= (unsigned long long)a.child[ch0 + k] << (8 * k);
  return c;
}

// DYN: one evaluation at the batch's state instead of steps, leaving only vdot.
template <class R, bool DYN = false>
__device__ __forceinline__ void wave_tree_body(const BucketArgs& a, int tid, double dt, int n_steps) {
  const int nb = a.nb, Bp = a.Bp;
  const int ipw = 64 / nb;  // instances per wave
  const int w = tid & 63, seg = w / nb, j = w - seg * nb;
  const int inst = (tid >> 6) * ipw + seg;
  if (seg >= ipw || inst >= a.B) return;  // an instance's lanes leave together
  int my_steps = n_steps;
  if (!DYN && a.active) {  // serving: the instance's remaining horizon
    const int left = a.active[inst];
    if (left <= 0) return;
    my_steps = min(my_steps, left);
    if (j == 0) a.active[inst] = left - my_steps;
  }
  // ---- topology of this lane's body (tables built by the host)
  const int maxd = a.max_depth;
  const int par = a.parent[j], depth = a.depth[j];
  const int ch0 = a.child_start[j], nch = a.child_start[j + 1] - ch0;
  const unsigned long long child = tree_children(a, ch0, nch);
  const int qo = a.qoff[j], vo = a.voff[j];
  const Soa<int> kindS(a.kind, nb, Bp);
  const int kind = kindS.ldx(0, inst, j);
  const bool one = kind == K_REV || kind == K_PRI;
  // exchange slots: the instance's and this lane's; then its floating joints'
  // coordinates (one more q than v each, so qo - vo numbers them)
  double* const lds = (double*)GP_DYN_LDS + ((size_t)(threadIdx.x >> 6) * ipw + seg) * tree_seg_doubles(nb, a.nq - a.nv);
  double* const mine = lds + j * kTreeSlot;
  R* const mineR = (R*)mine;
  double* const fl = lds + nb * kTreeSlot + (qo - vo) * kTreeFloat;
  // ---- parameters and state of this lane's body and joint, for the launch
  const Soa<double> bpS(a.bp, NBF * nb, Bp);
  const Soa<R> bpR(pick<R>(a.bp, a.bpf), NBF * nb, Bp);
  auto pd = [&](int f) { return bpS.ldx(f * nb, inst, j); };
  auto pr = [&](int f) { return bpR.ldx(f * nb, inst, j); };
  m3<double> Rt;
#pragma unroll
  for (int k = 0; k < 9; ++k) Rt.a[k] = pd(BF_RT + k);
  const v3<double> pt{pd(BF_PT), pd(BF_PT + 1), pd(BF_PT + 2)};
  const s3<R> J{pr(BF_J), pr(BF_J + 1), pr(BF_J + 2), pr(BF_J + 3), pr(BF_J + 4), pr(BF_J + 5)};
  const v3<R> mc{pr(BF_C), pr(BF_C + 1), pr(BF_C + 2)};
  const R mass = pr(BF_M);
  const double sk = kind == K_PRI ? pd(BF_SK) : 0.0;
  const double sl = kind == K_PRI ? pd(BF_SL) : 0.0;
  const Soa<double> qS(a.q, a.nq, Bp), vS(a.v, a.nv, Bp), tauS(a.tau, a.nv, Bp), vdotS(a.vdot, a.nv, Bp);
  double q = 0.0, v = 0.0, tau = 0.0, vd = 0.0;  // of a one-DOF joint
  if (one) {
    q = qS.ldx(0, inst, qo);
    v = vS.ldx(0, inst, vo);
    tau = tauS.ldx(0, inst, vo);
  } else if (kind == K_FLOAT) {
#pragma unroll
    for (int k = 0; k < 7; ++k) fl[k] = qS.ldx(k, inst, qo);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      fl[7 + k] = vS.ldx(k, inst, vo);
      fl[13 + k] = tauS.ldx(k, inst, vo);
    }
  }
  const bool contacts = a.nc > 0;
  const int c0 = a.cstart[j], c1 = a.cstart[j + 1];
  bool ok = true;
  for (int s = 0; s < my_steps; ++s) {
    // ---- this joint's transform (E, r: parent -> body) and velocity S qd
    m3<R> E;
    v3<R> r;
    sv<R> vj{{R(0), R(0), R(0)}, {R(0), R(0), R(0)}};
    m3<double> Rw;  // body -> parent, then world: rotation and translation, FP64 (contacts, floating pose)
    v3<double> tw;
    if (kind == K_FLOAT) {
      Rw = mul(Rt, quat_mat(fl[0], fl[1], fl[2], fl[3]));
      tw = pt + mul(Rt, v3<double>{fl[4], fl[5], fl[6]});
      const m3<R> Rm = cvt<R>(Rw);
      E = m3<R>{{Rm.a[0], Rm.a[3], Rm.a[6], Rm.a[1], Rm.a[4], Rm.a[7], Rm.a[2], Rm.a[5], Rm.a[8]}};
      r = cvt<R>(tw);
      vj = sv<R>{{R(fl[7]), R(fl[8]), R(fl[9])}, {R(fl[10]), R(fl[11]), R(fl[12])}};
    } else {
      R cs = R(1), sn = R(0), dd = R(0);
      if (kind == K_REV) sincos_q(q, &sn, &cs);
      if (kind == K_PRI) dd = R(q);
      joint_frame(cvt<R>(Rt), cvt<R>(pt), cs, sn, dd, E, r);
      if (kind == K_REV) vj.w.z = R(v);
      if (kind == K_PRI) vj.v.z = R(v);
      if (contacts) {
        const m3<double> Ed = cvt<double>(E);
        Rw = m3<double>{{Ed.a[0], Ed.a[3], Ed.a[6], Ed.a[1], Ed.a[4], Ed.a[7], Ed.a[2], Ed.a[5], Ed.a[8]}};
        tw = cvt<double>(r);
      }
    }
    // ---- pass 1, root to leaves by depth: velocities (and world poses);
    // slot: velocity (R) from the start, world rotation doubles [6, 15),
    // world translation doubles [15, 18)
    sv<R> vel = vj;
    auto put_pose = [&]() {
      put_sv(mineR, vel);
      if (contacts) {
#pragma unroll
        for (int k = 0; k < 9; ++k) mine[6 + k] = Rw.a[k];
        mine[15] = tw.x; mine[16] = tw.y; mine[17] = tw.z;
      }
    };
    level_fence();  // the previous step's pass-3 reads come first
    if (depth == 0) put_pose();
    for (int d = 1; d <= maxd; ++d) {
      level_fence();
      if (depth == d) {
        const double* ps = lds + par * kTreeSlot;
        vel = xmotion(E, r, get_sv<R>((const R*)ps)) + vj;
        if (contacts) {
          m3<double> pR;
#pragma unroll
          for (int k = 0; k < 9; ++k) pR.a[k] = ps[6 + k];
          tw = v3<double>{ps[15], ps[16], ps[17]} + mul(pR, tw);
          Rw = mul(pR, Rw);
        }
        if (d < maxd) put_pose();
      }
    }
    // velocity-product acceleration, rigid-body bias force, contact forces
    const sv<R> cb = crm(vel, vj);
    const ai6<R> I = rigid(J, mc, mass);
    sv<R> pA;
    {
      // v x* (I v): w x (J w) + c x g and m g + w x (w x c) with g = w x v
      const v3<R> g = cross(vel.w, vel.v), hw = mul(J, vel.w), wc = cross(vel.w, mc);
      pA = sv<R>{cross(vel.w, hw) + cross(mc, g), mass * g + cross(vel.w, wc)};
    }
    if (contacts && c0 < c1) pA = pA - tree_contacts<R>(a, inst, c0, c1, Rw, tw, vel);
    // ---- pass 2, leaves to root by depth: articulated inertias and bias forces
    ai6<R> IA = I;
    sv<R> U{{R(0), R(0), R(0)}, {R(0), R(0), R(0)}};
    double Dinv = 0.0, u = 0.0;
    // a one-DOF joint's U, D and u (tq: torque and prismatic spring, dynamics.rs:298-315)
    auto solve_one = [&]() {
      const bool rev = kind == K_REV;
      U = rev ? col(IA, 2) : col(IA, 5);
      Dinv = recip(double(rev ? IA.A.zz : IA.C.zz));
      ok = ok && (Dinv > 0.0);
      const double tq = tau - sk * (q - sl);
      u = tq - double(rev ? pA.w.z : pA.v.z);
    };
    for (int d = maxd; d >= 1; --d) {
      if (depth == d) {
        // in place: IA becomes the joint's Ia
        sv<R> pa;
        if (one) {
          solve_one();
          const R inv = R(Dinv);
          const sv<R> uD{inv * U.w, inv * U.v};
          IA = rank1_down(IA, U, uD);
          const R uR = R(u);
          pa = pA + mul(IA, cb) + sv<R>{uR * uD.w, uR * uD.v};
        } else if (kind == K_FLOAT) {
          // Ia = I^A - I^A (I^A)^-1 I^A = 0 (IA stays for pass 3); pA + u is the whole torque
#pragma unroll
          for (int k = 0; k < 21; ++k) mineR[k] = R(0);
          pa = sv<R>{{R(fl[13]), R(fl[14]), R(fl[15])}, {R(fl[16]), R(fl[17]), R(fl[18])}};
        } else {
          pa = pA + mul(IA, cb);
        }
        // slot (R): articulated inertia [0, 21), bias force [21, 27)
        if (kind != K_FLOAT) put_ai6(mineR, xtix(E, r, IA));
        put_sv(mineR + 21, xtforce(E, r, pa));
      }
      // parents (depth d - 1) take their children's parts, in child order
      level_fence();
      if (depth == d - 1) {
        for (int k = 0; k < nch; ++k) {
          const R* cs = (const R*)(lds + (int)((child >> (8 * k)) & 63) * kTreeSlot);
          add_to(IA, get_ai6<R>(cs));
          pA = pA + get_sv<R>(cs + 21);
        }
      }
      level_fence();  // the slots read here are written again only in pass 3
    }
    if (depth == 0 && one) solve_one();
    // ---- pass 3, root to leaves by depth: accelerations, then the joint's step
    for (int d = 0; d <= maxd; ++d) {
      level_fence();
      if (depth == d) {
        sv<R> pacc{{R(0), R(0), R(0)}, {R(0), R(0), R(a.g)}};  // gravity as the base's acceleration
        if (d > 0) pacc = get_sv<R>((const R*)(lds + par * kTreeSlot));
        sv<R> ap = xmotion(E, r, pacc) + cb;
        if (one) {
          const double qdd = (u - double(dot6(U, ap))) * Dinv;
          vd = qdd;
          if (kind == K_REV) ap.w.z += R(qdd);
          else ap.v.z += R(qdd);
        } else if (kind == K_FLOAT) {
          const ai6<double> Id = cvt<double>(IA);
          const sv<double> apd{cvt<double>(ap.w), cvt<double>(ap.v)}, pAd{cvt<double>(pA.w), cvt<double>(pA.v)};
          const sv<double> Ia = mul(Id, apd);
          double L[21];
          double x[6] = {fl[13] - pAd.w.x - Ia.w.x, fl[14] - pAd.w.y - Ia.w.y, fl[15] - pAd.w.z - Ia.w.z,
                         fl[16] - pAd.v.x - Ia.v.x, fl[17] - pAd.v.y - Ia.v.y, fl[18] - pAd.v.z - Ia.v.z};
          ok = ldl6(Id, L) && ok;
          ldl6_solve(L, x);
#pragma unroll
          for (int t = 0; t < 6; ++t) fl[19 + t] = x[t];
          ap = ap + sv<R>{{R(x[0]), R(x[1]), R(x[2])}, {R(x[3]), R(x[4]), R(x[5])}};
        }
        if (d < maxd) put_sv(mineR, ap);  // slot (R): acceleration from the start
      }
    }
    if constexpr (DYN) break;
    // ---- semi-implicit Euler of this lane's joint (integrators.rs:276-319); a
    // non-finite acceleration leaves v non-finite for good
    if (kind == K_FLOAT) {
      double qf[7], vf[6];
#pragma unroll
      for (int k = 0; k < 7; ++k) qf[k] = fl[k];
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        vf[k] = fl[7 + k] + fl[19 + k] * dt;
        fl[7 + k] = vf[k];
      }
      advance_floating(qf, vf, dt, qf);
#pragma unroll
      for (int k = 0; k < 7; ++k) fl[k] = qf[k];
    } else if (one) {
      v = v + vd * dt;
      q += v * dt;
    }
  }
  if (one) {
    if constexpr (!DYN) {
      qS.stx(0, inst, qo, q);
      vS.stx(0, inst, vo, v);
    }
    vdotS.stx(0, inst, vo, vd);
    ok = ok && isfinite(q) && isfinite(v) && isfinite(vd);
  } else if (kind == K_FLOAT) {
#pragma unroll
    for (int k = 0; k < 7; ++k) {
      const double x = fl[k];
      if constexpr (!DYN) qS.stx(k, inst, qo, x);
      ok = ok && isfinite(x);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const double x = fl[7 + k], y = fl[19 + k];
      if constexpr (!DYN) vS.stx(k, inst, vo, x);
      vdotS.stx(k, inst, vo, y);
      ok = ok && isfinite(x) && isfinite(y);
    }
  }
  if (!ok) a.fault[inst] = 1;  // any lane's fault is the instance's
}

// Two waves per SIMD (at most 256 registers a lane)
template <class R>
__global__ void __launch_bounds__(256, 2) wave_tree_kernel(BucketArgs a, double dt, int n_steps) {
  wave_tree_body<R>(a, blockIdx.x * blockDim.x + threadIdx.x, dt, n_steps);
}
// Every bucket of a batch of trees in one launch, at the occupancy of the
// kernel above (the grouped launch over all compiled topologies runs at one
// wave per SIMD).
template <class R>
__global__ void __launch_bounds__(256, 2) grouped_tree_kernel(const GroupTable* __restrict__ t, double dt, int n_steps) {
  int b = 0;
  while (b + 1 < t->n && (int)blockIdx.x >= t->block_start[b + 1]) ++b;  // uniform per workgroup
  const BucketArgs a = t->args[b];
  const int tid = ((int)blockIdx.x - t->block_start[b]) * (int)blockDim.x + (int)threadIdx.x;
  wave_tree_body<R>(a, tid, dt, n_steps);
}

// The table entry that owns workgroup b (uniform), for a query over every bucket.
__device__ __forceinline__ int query_entry(const QueryEntry* t, int n, unsigned b) {
  int e = 0;
  for (int hi = n; hi - e > 1;) {
    const int mid = (e + hi) / 2;
    if (t[mid].first <= b) e = mid;
    else hi = mid;
  }
  return e;
}
template <class R>
static int launch_wave_tree(const BucketArgs& a, double dt, int n_steps, int block, hipStream_t s) {
  dim3 blk(block), grid((unsigned)((fast_threads(TOPO_TREE, a.B, a.nb) + block - 1) / block));
  const unsigned lds = (unsigned)(block / 64 * tree_wave_bytes(a.nb, a.nq - a.nv));
  hipLaunchKernelGGL((wave_tree_kernel<R>), grid, blk, lds, s, a, dt, n_steps);
  return (int)hipGetLastError();
}

}  // namespace gp
