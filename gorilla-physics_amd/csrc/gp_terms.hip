// gp_terms.hip — the joint-space terms of M(q) vdot + c(q, v) = tau + tau_c
// at a batch's state: the mass matrix M by the composite-rigid-body algorithm
// (the quantity of mechanism.rs:637-696, RBDA Table 6.2) and the bias
// c(q, v) - tau_c by recursive Newton-Euler with zero joint accelerations
// (the quantity of dynamics.rs:233-251, RBDA Table 5.1). FP64, runtime
// topology, one instance per lane, in the aligned body frames of the plain
// kernel: a 1-DOF joint's motion subspace is e_z (angular for revolute,
// linear for prismatic) and a floating joint's is the identity in the body
// frame, so every entry S_i^T (...) S_j is the reference's, whose floating
// velocity is the body twist in the body frame.
//
// Two kernels. terms_kernel: one instance per lane, per-body intermediates in
// device scratch; any topology, spring contacts. tree_terms_kernel: one body
// per lane (as gp_tree_impl.h: instances packed in waves, levels exchanging
// through LDS), every bucket of a batch in one launch, and only the term that
// is asked for; any tree without spring contacts and with at most
// kTreeMaxChildren children a body. The first is bound by its chains of
// dependent scratch loads, bucket after bucket (13 buckets of 1,500 chains and
// quadrupeds: 13 launches of 113 us for either term); the second, 18 us for M
// and 11 us for c of the same batch, by its levels' latency. vdot, M and c of
// that batch through the host calls: 6.7 ms before, 0.8 ms now.
#include "gp_fast_impl.h"
#include "gp_plain_impl.h"

namespace gp {

namespace {

// component k of the motion-subspace column c of body i's joint applied to a
// force-like 6-vector f: S_c^T f
__device__ inline double s_dot(int kind, int c, const sv<double>& f) {
  if (kind == K_REV) return f.w.z;
  if (kind == K_PRI) return f.v.z;
  return c < 3 ? (&f.w.x)[c] : (&f.v.x)[c - 3];
}
__device__ inline int n_dof(int kind) { return kind == K_FLOAT ? 6 : (kind == K_FIXED ? 0 : 1); }

// out: [nv * nv + nv][Bp]: M row-major, then c - tau_c
__global__ void __launch_bounds__(64) terms_kernel(BucketArgs a, double* out) {
  const int lane = blockIdx.x * blockDim.x + threadIdx.x;
  if (lane >= a.B) return;
  const int nb = a.nb, nv = a.nv, Bp = a.Bp;
  const Strided q{a.q + lane, Bp}, v{a.v + lane, Bp};
  const Strided M{out + lane, Bp}, c{out + (size_t)nv * nv * Bp + lane, Bp};
  PlainCtx X{a, lane};
  // transforms, velocities, velocity-product accelerations, rigid inertias,
  // bias forces v x* (I v) - f_contact; the spring contacts' state is left alone
  plain_kinematics(a, lane, q, v, true, false);
  // ---- recursive Newton-Euler with vdot = 0: a_i = X_i a_parent + c_i
  // (gravity as the base's acceleration), f_i = I_i a_i + v x* (I v) - f_ext
  for (int i = 0; i < nb; ++i) {
    const int pr = a.parent[i];
    const sv<double> ap = pr < 0 ? sv<double>{{0, 0, 0}, {0, 0, a.g}} : X.ldv(PF_ACC, pr);
    const sv<double> ai = xmotion(X.ldm(PF_E, i), X.ld3(PF_R, i), ap) + X.ldv(PF_CB, i);
    X.stv(PF_ACC, i, ai);
    X.stv(PF_PA, i, X.ldv(PF_PA, i) + mul(X.ldi(i), ai));
  }
  for (int i = nb - 1; i >= 0; --i) {  // leaves to root: tau_i = S_i^T f_i, f_parent += X^T f_i
    const int k = a.kind[i * Bp + lane];
    const sv<double> f = X.ldv(PF_PA, i);
    for (int col = 0; col < n_dof(k); ++col) c[a.voff[i] + col] = s_dot(k, col, f);
    const int pr = a.parent[i];
    if (pr >= 0) X.stv(PF_PA, pr, X.ldv(PF_PA, pr) + xtforce(X.ldm(PF_E, i), X.ld3(PF_R, i), f));
  }
  // ---- composite inertias, leaves to root (the rigid inertias are in PF_IA)
  for (int i = nb - 1; i >= 0; --i) {
    const int pr = a.parent[i];
    if (pr < 0) continue;
    ai6<double> P = X.ldi(pr);
    add_to(P, xtix(X.ldm(PF_E, i), X.ld3(PF_R, i), X.ldi(i)));
    X.sti(pr, P);
  }
  // ---- M: F = Ic_i S_i carried towards the root, M_ij = S_j^T F
  for (int i = 0; i < nb; ++i) {
    const int ki = a.kind[i * Bp + lane];
    const ai6<double> Ic = X.ldi(i);
    for (int ca = 0; ca < n_dof(ki); ++ca) {
      const int row = a.voff[i] + ca;
      const int sidx = ki == K_REV ? 2 : ki == K_PRI ? 5 : ca;
      sv<double> F = col(Ic, sidx);
      for (int cb = 0; cb < n_dof(ki); ++cb) M[row * nv + a.voff[i] + cb] = s_dot(ki, cb, F);
      for (int j = i; a.parent[j] >= 0;) {
        F = xtforce(X.ldm(PF_E, j), X.ld3(PF_R, j), F);
        j = a.parent[j];
        const int kj = a.kind[j * Bp + lane];
        for (int cb = 0; cb < n_dof(kj); ++cb) {
          const int colj = a.voff[j] + cb;
          const double m = s_dot(kj, cb, F);
          M[row * nv + colj] = m;
          M[colj * nv + row] = m;
        }
      }
    }
  }
  // entries of joints that support neither body stay zero
  for (int i = 0; i < nb; ++i)
    for (int j = 0; j < nb; ++j) {
      bool related = false;
      for (int k = i; k >= 0 && !related; k = a.parent[k]) related = k == j;
      for (int k = j; k >= 0 && !related; k = a.parent[k]) related = k == i;
      if (related) continue;
      const int ni = n_dof(a.kind[i * Bp + lane]), nj = n_dof(a.kind[j * Bp + lane]);
      for (int r = 0; r < ni; ++r)
        for (int cc = 0; cc < nj; ++cc) M[(a.voff[i] + r) * nv + a.voff[j] + cc] = 0.0;
    }
}

// A lane's slot in the queries: the exchange part (kTreeSlot), the joint's E
// and r, and two words (parent, kind and first row; the bodies up to the root).
// Odd, so a wave's 64-bit accesses spread over the banks.
constexpr int kTermsSlot = kTreeSlot + 12 + 2;
__device__ __forceinline__ unsigned long long pack_body(int par, int kind, int vo) {
  return (unsigned long long)(unsigned char)(par + 1) | (unsigned long long)kind << 8 | (unsigned long long)vo << 16;
}

// s_dot by selects, not by address
__device__ __forceinline__ double s_row(int kind, int c, const sv<double>& f) {
  return kind == K_REV ? f.w.z : kind == K_PRI ? f.v.z : comp(f, c);
}

// MASS: M's entries; else c - tau_c.
template <bool MASS>
__global__ void __launch_bounds__(64, 2) tree_terms_kernel(const QueryEntry* __restrict__ t, int n, double* out) {
  const int e = query_entry(t, n, blockIdx.x);
  const BucketArgs a = t[e].a;
  const int nb = a.nb, nv = a.nv, Bp = a.Bp, ipw = 64 / nb;
  const int w = (int)threadIdx.x, seg = w / nb, j = w - seg * nb;
  const int inst = (int)(blockIdx.x - t[e].first) * ipw + seg;
  if (seg >= ipw || inst >= a.B) return;  // an instance's lanes leave together
  const int maxd = a.max_depth, depth = a.depth[j], par = a.parent[j];
  const int ch0 = a.child_start[j], nch = a.child_start[j + 1] - ch0;
  const unsigned long long child = tree_children(a, ch0, nch);
  const int qo = a.qoff[j], vo = a.voff[j];
  const Soa<int> kindS(a.kind, nb, Bp);
  const int kind = kindS.ldx(0, inst, j);
  double* const lds = (double*)GP_DYN_LDS + (size_t)seg * nb * kTermsSlot;
  double* const mine = lds + j * kTermsSlot;
  const Soa<double> bpS(a.bp, NBF * nb, Bp), qS(a.q, a.nq, Bp), vS(a.v, nv, Bp);
  auto pd = [&](int f) { return bpS.ldx(f * nb, inst, j); };
  m3<double> Rw;
#pragma unroll
  for (int k = 0; k < 9; ++k) Rw.a[k] = pd(BF_RT + k);
  v3<double> tw{pd(BF_PT), pd(BF_PT + 1), pd(BF_PT + 2)};
  const s3<double> J{pd(BF_J), pd(BF_J + 1), pd(BF_J + 2), pd(BF_J + 3), pd(BF_J + 4), pd(BF_J + 5)};
  const v3<double> mc{pd(BF_C), pd(BF_C + 1), pd(BF_C + 2)};
  const double mass = pd(BF_M);
  // this joint's transform (E, r: parent -> body) and velocity S qd
  sv<double> vj{{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
  if (kind == K_FLOAT) {
    auto q = [&](int k) { return qS.ldx(k, inst, qo); };
    tw = tw + mul(Rw, v3<double>{q(4), q(5), q(6)});
    Rw = mul(Rw, quat_mat(q(0), q(1), q(2), q(3)));
    if constexpr (!MASS) {
      auto v = [&](int k) { return vS.ldx(k, inst, vo); };
      vj = sv<double>{{v(0), v(1), v(2)}, {v(3), v(4), v(5)}};
    }
  } else if (kind == K_REV || kind == K_PRI) {
    const double q = qS.ldx(0, inst, qo), v = MASS ? 0.0 : vS.ldx(0, inst, vo);
    if (kind == K_REV) {
      double s, c;
      sincos_q(q, &s, &c);
      Rw = mul(Rw, m3<double>{{c, -s, 0.0, s, c, 0.0, 0.0, 0.0, 1.0}});
      vj.w.z = v;
    } else {
      tw = tw + q * v3<double>{Rw.a[2], Rw.a[5], Rw.a[8]};
      vj.v.z = v;
    }
  }
  const m3<double> E{{Rw.a[0], Rw.a[3], Rw.a[6], Rw.a[1], Rw.a[4], Rw.a[7], Rw.a[2], Rw.a[5], Rw.a[8]}};
  const v3<double> r = tw;
  if constexpr (MASS) {
    double* const er = mine + kTreeSlot;
#pragma unroll
    for (int k = 0; k < 9; ++k) er[k] = E.a[k];
    er[9] = r.x; er[10] = r.y; er[11] = r.z;
    auto words = [&](int b) { return (unsigned long long*)(lds + b * kTermsSlot + kTreeSlot + 12); };
    words(j)[0] = pack_body(par, kind, vo);
    // ---- composite inertias, leaves to root
    ai6<double> Ic = rigid(J, mc, mass);
    for (int d = maxd; d >= 1; --d) {
      level_fence();
      if (depth == d) put_ai6(mine, xtix(E, r, Ic));
      level_fence();
      if (depth == d - 1)
        for (int k = 0; k < nch; ++k) add_to(Ic, get_ai6<double>(lds + (int)((child >> (8 * k)) & 63) * kTermsSlot));
    }
    level_fence();
    // ---- M: F = Ic_i S_i carried towards the root, M_ij = S_j^T F; every
    // entry is written once, by the lane of the body further out
    double* const M = out + t[e].moff[inst];
    unsigned long long above = 1ull << j;  // this body and those up to the root
    for (int b = par; b >= 0; b = (int)(words(b)[0] & 0xff) - 1) above |= 1ull << b;
    words(j)[1] = above;
    const int nj = n_dof(kind);
    const sv<double> one = kind == K_REV ? col(Ic, 2) : col(Ic, 5);
#pragma unroll
    for (int c = 0; c < 6; ++c) {  // unrolled: a column picked by a constant stays in registers
      if (c >= nj) break;
      const int row = vo + c;
      sv<double> F = kind == K_FLOAT ? col(Ic, c) : one;
      for (int k = 0; k < nj; ++k) M[row * nv + vo + k] = s_row(kind, k, F);
      int b = j, up = par;
      while (up >= 0) {
        const double* eb = lds + b * kTermsSlot + kTreeSlot;
        m3<double> Eb;
#pragma unroll
        for (int k = 0; k < 9; ++k) Eb.a[k] = eb[k];
        F = xtforce(Eb, v3<double>{eb[9], eb[10], eb[11]}, F);
        b = up;
        const unsigned long long x = words(b)[0];
        up = (int)(x & 0xff) - 1;
        const int kb = (int)(x >> 8) & 0xff, cb = (int)(x >> 16);
        for (int k = 0; k < n_dof(kb); ++k) {
          const double m = s_row(kb, k, F);
          M[row * nv + cb + k] = m;
          M[(cb + k) * nv + row] = m;
        }
      }
    }
    level_fence();
    // entries of joints that support neither body are zero
    for (int b = 0; b < nb; ++b) {
      if (((above >> b) & 1) || ((words(b)[1] >> j) & 1)) continue;
      const unsigned long long x = words(b)[0];
      const int kb = n_dof((int)(x >> 8) & 0xff), cb = (int)(x >> 16);
      for (int c = 0; c < nj; ++c)
        for (int k = 0; k < kb; ++k) M[(vo + c) * nv + cb + k] = 0.0;
    }
  } else {
    // ---- recursive Newton-Euler with vdot = 0: a_i = X_i a_parent + c_i
    // (gravity as the base's acceleration), f_i = I_i a_i + v x* (I v) - f_ext;
    // slot: velocity [0, 6), acceleration [6, 12), world pose [12, 24)
    const bool contacts = a.nc > 0;
    sv<double> vel = vj, acc = xmotion(E, r, sv<double>{{0.0, 0.0, 0.0}, {0.0, 0.0, a.g}}) + crm(vel, vj);
    auto put = [&]() {
      put_sv(mine, vel);
      put_sv(mine + 6, acc);
      if (contacts) {
#pragma unroll
        for (int k = 0; k < 9; ++k) mine[12 + k] = Rw.a[k];
        mine[21] = tw.x; mine[22] = tw.y; mine[23] = tw.z;
      }
    };
    if (depth == 0) put();
    for (int d = 1; d <= maxd; ++d) {
      level_fence();
      if (depth == d) {
        const double* p = lds + par * kTermsSlot;
        vel = xmotion(E, r, get_sv<double>(p)) + vj;
        acc = xmotion(E, r, get_sv<double>(p + 6)) + crm(vel, vj);
        if (contacts) {
          m3<double> R;
#pragma unroll
          for (int k = 0; k < 9; ++k) R.a[k] = p[12 + k];
          tw = v3<double>{p[21], p[22], p[23]} + mul(R, tw);
          Rw = mul(R, Rw);
        }
        if (d < maxd) put();
      }
    }
    const ai6<double> I = rigid(J, mc, mass);
    sv<double> f = mul(I, acc) + crf(vel, mul(I, vel));
    const int c0 = a.cstart[j], c1 = a.cstart[j + 1];
    if (contacts && c0 < c1) f = f - tree_contacts<double>(a, inst, c0, c1, Rw, tw, vel);
    for (int d = maxd; d >= 1; --d) {  // leaves to root: f_parent += X^T f
      level_fence();
      if (depth == d) put_sv(mine, xtforce(E, r, f));
      level_fence();
      if (depth == d - 1)
        for (int k = 0; k < nch; ++k) f = f + get_sv<double>(lds + (int)((child >> (8 * k)) & 63) * kTermsSlot);
    }
    double* const c = out + t[e].voff[inst] + vo;
    for (int k = 0; k < n_dof(kind); ++k) c[k] = s_row(kind, k, f);
  }
}

}  // namespace

int launch_terms(const BucketArgs& a, double* out, void* stream) {
  const int block = 64;
  hipLaunchKernelGGL(terms_kernel, dim3((a.B + block - 1) / block), dim3(block), 0, (hipStream_t)stream, a, out);
  return (int)hipGetLastError();
}

int launch_tree_terms(const QueryEntry* d_table, int n, unsigned blocks, int lds, double* M, double* c, void* stream) {
  if (n == 0 || blocks == 0) return 0;
  if (M)
    hipLaunchKernelGGL(tree_terms_kernel<true>, dim3(blocks), dim3(64), (unsigned)lds, (hipStream_t)stream, d_table, n,
                       M);
  else
    hipLaunchKernelGGL(tree_terms_kernel<false>, dim3(blocks), dim3(64), (unsigned)lds, (hipStream_t)stream, d_table, n,
                       c);
  return (int)hipGetLastError();
}

// the larger of a terms wave and a dynamics wave
int query_lds_per_wave(int nb, int floating) {
  const int terms = 64 / nb * nb * kTermsSlot * 8, dyn = tree_wave_bytes(nb, floating);
  return terms > dyn ? terms : dyn;
}

}  // namespace gp
